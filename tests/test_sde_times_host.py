"""constant_grid and the times of the saved rows, computed for all steps at once, against the
step-by-step definitions (constant.py:30-104 with the end clipping of _integrate.py:278-284,
319-322; the kernels' row order): the same float64 values."""
import math

import numpy as np
import pytest

from diffrax_amd._sde import _row_times, constant_grid


def _grid_by_steps(t0, t1, dt0):
    num = int(math.ceil((t1 - t0) / float(np.nextafter(dt0, math.inf))))
    floor = t1
    for _ in range(100):
        floor = float(np.nextafter(floor, -math.inf))
    ts, tnext, n, tprev = [t0], min(t0 + dt0, t1), 1, t0
    while tprev < t1:
        ts.append(tnext)
        n += 1
        tn = t1 if n == num else t0 + (t1 - t0) * (n / num)
        tprev = min(tnext, t1)
        tnext = t1 if tn > floor else tn
    return np.array(ts)


@pytest.mark.parametrize("t0", [0.0, -3.7, 1e6])
@pytest.mark.parametrize("span", [1.0, 0.3, 1e-3])
def test_constant_grid(t0, span):
    rng = np.random.default_rng(3)
    t1 = t0 + span
    s = t1 - t0
    dts = [s, 2 * s, s * (1 - 1e-15), s / 3]
    for n in rng.integers(1, 700, 40):
        dts += [s / n, np.nextafter(s / n, 0), np.nextafter(s / n, 9), rng.uniform(s / 800, 2 * s)]
    for dt in dts:
        assert np.array_equal(constant_grid(t0, t1, float(dt)), _grid_by_steps(t0, t1, float(dt)))


@pytest.mark.parametrize("k", [0, 1, 3, 7, 100])
@pytest.mark.parametrize("flags", [(0, 0), (1, 0), (0, 1), (1, 1)])
def test_row_times(k, flags):
    rng = np.random.default_rng(k)
    for N in (1, 2, 7, 30):
        grid = constant_grid(0.25, 2.0, 1.75 / N)
        for ts in (None, np.empty(0), np.sort(rng.uniform(0.25, 2.0, 9)),
                   np.sort(np.concatenate((grid, grid[:1], [0.25, 2.0])))):
            want, i = [0.25] if flags[0] else [], 0
            for n in range(N):
                while ts is not None and i < ts.size and ts[i] <= grid[n + 1]:
                    want.append(ts[i])
                    i += 1
                if k and (n + 1) % k == 0:
                    want.append(grid[n + 1])
            if flags[1] and not (k and N % k == 0):
                want.append(2.0)
            got = _row_times(grid, ts, bool(flags[0]), bool(flags[1]), k, 0.25, 2.0)
            assert np.array_equal(got, np.array(want))
