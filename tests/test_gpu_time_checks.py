"""dfx_check_times: the checks of device-resident t1 / SaveAt(ts) (_integrate.py:1107-1112,
1222-1235), word for word against the host form on the same times."""
import numpy as np
import pytest
import torch

from diffrax_amd import _integrate

pytestmark = pytest.mark.gpu


def _host_bits(t0, t1, dt0, ts):
    t1 = np.atleast_1d(t1)
    bits = 1 if dt0 is not None and ((t1 - t0) * dt0 < 0).any() else 0
    if ts is not None:
        dirs = np.where(t0 < t1, 1.0, -1.0)[:, None]
        tn, t1n = np.atleast_2d(ts) * dirs, t1[:, None] * dirs
        bits |= 2 if (tn[:, 1:] < tn[:, :-1]).any() else 0
        bits |= 4 if ((tn > t1n) | (tn < t0 * dirs)).any() else 0
    return bits


@pytest.mark.parametrize("rows,n", [(1, 1), (1, 2), (3, 0), (255, 5), (257, 64), (4099, 33)])
@pytest.mark.parametrize("t1_rows", [True, False])
@pytest.mark.parametrize("ts_rows", [True, False])
def test_bits_match_the_host(cuda, rows, n, t1_rows, ts_rows):
    rng = np.random.default_rng(rows + n)
    dev = lambda a: torch.tensor(np.ascontiguousarray(a), device=cuda)
    for sign in (1.0, -1.0):
        t1 = sign * (rng.uniform(2.0, 3.0, rows) if t1_rows else np.full(1, 2.0))
        base = np.sort(rng.uniform(0.5, 1.5, (rows, n) if ts_rows else n), axis=-1) * sign
        cases = [(t1, sign, base), (t1, -sign, base), (t1, None, base)]
        for where in ([0, -1] if n else []):
            for v in (np.nan, np.inf, -np.inf, sign * 4.0, -sign * 0.25):
                bad = base.copy()
                bad.reshape(-1)[where] = v
                cases.append((t1, sign, bad))
            bad = t1.copy()
            bad[where] = np.nan
            cases.append((bad, sign, base))
        for t1v, dt0, ts in cases:
            with np.errstate(invalid="ignore"):
                want = _host_bits(0.0, t1v, dt0, ts if n else None)
            got = _integrate._TimeChecks(0.0, dev(t1v), dt0, dev(ts) if n else None, cuda).bits()
            assert got == want, (sign, dt0, got, want)
        if not t1_rows and n:   # t1 as a number (the neural-ODE kernel's)
            got = _integrate._TimeChecks(0.0, float(t1[0]), None, dev(base), cuda).bits()
            assert got == _host_bits(0.0, t1, None, base)
