"""The neural-ODE discrete adjoint over tiles that take different numbers of steps: segments
in which some tiles have no step left, a partial last tile, and trajectories that end before
the longest of their tile, against float64 replay of the recorded steps."""
import numpy as np
import pytest

from tests.test_gpu_mlp_grad import _device_grads, _replay_grads, _setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("matmul", ["f32", "bf16"])
@pytest.mark.parametrize("B,C,n_ts", [(1, 1, 2), (33, 2, 40), (70, 3, 9), (70, 32, 1)])
def test_uneven_tiles_against_fp64_replay(cuda, matmul, B, C, n_ts):
    Wn, y0, _, _ = _setup(matmul, B=B, n_ts=n_ts)
    rng = np.random.default_rng(B + C)
    # the first tile near a slow region with a flat field, the others spread wider
    y0 = (rng.normal(size=(B, 64)) * np.where(np.arange(B) < 32, 0.01, 3.0)[:, None]).astype(np.float32)
    ts = np.sort(rng.uniform(0.0, 1.0, n_ts))
    ts[-1] = 1.0
    w = rng.normal(size=(B, n_ts, 64)).astype(np.float32)
    grads, grid, nacc = _device_grads(Wn, y0, ts, w, matmul, C, max_steps=32)
    if B > 32:
        assert nacc[:32].max() != nacc[32:].max()   # tiles of different lengths
    ref, _ = _replay_grads(Wn, y0, ts, w, grid, nacc)
    for name, g, r in zip(("y0", "W1", "b1", "W2", "b2", "W3", "b3"), grads, ref):
        rel = float((g - r).abs().max() / r.abs().max())
        assert rel < 1e-4, (name, rel)   # the adjoint's bar, both forms
