"""Times of an SDE solve's saved rows with NaN among the save times (CPU only): the rows end
there, as a walk over the steps finds them."""
import numpy as np
import pytest

from diffrax_amd import _sde


def _walk(grid, ts, save_t0, save_t1, k, t0, t1):
    out, i, N = [t0] if save_t0 else [], 0, len(grid) - 1
    for n in range(N):
        while i < len(ts) and ts[i] <= grid[n + 1]:
            out.append(ts[i])
            i += 1
        if k and (n + 1) % k == 0:
            out.append(grid[n + 1])
    return np.array(out + ([t1] if save_t1 and not (k and N % k == 0) else []))


@pytest.mark.parametrize("k", [0, 1, 3])
@pytest.mark.parametrize("at", [0, 1, 3, 4])
def test_rows_end_at_a_nan(at, k):
    grid = _sde.constant_grid(0.0, 1.0, 0.1)
    ts = np.array([0.0, 0.25, 0.5, 0.5, 1.0])
    ts[at] = np.nan
    for save_t0 in (False, True):
        for save_t1 in (False, True):
            args = (grid, ts, save_t0, save_t1, k, 0.0, 1.0)
            assert np.array_equal(_sde._row_times(*args), _walk(*args))
