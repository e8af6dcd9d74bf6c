"""The neural-ODE gradient against the float64 replay at the accuracy that its products are held
to.  Bound, normwise: the activations' and deltas' float32 rounding (2^-24, three layers and
their transposes, errors independent over hundreds of rows) and three-piece products (2^-23)
leave a few 2^-23; 2e-6 is seventeen of them.  A product without its third piece or without one
of the 2^-16 corrections is off by 2^-17 = 8e-6 of an operand and does not pass."""
import numpy as np
import pytest

from tests.test_gpu_mlp_grad import _device_grads, _replay_grads, _setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("matmul", ["f32", "bf16"])
@pytest.mark.parametrize("B,C", [(40, 2), (70, 32)])
def test_against_fp64_replay(cuda, matmul, B, C):
    Wn, y0, ts, w = _setup(matmul, B=B, C=C, seed=B)
    grads, grid, nacc = _device_grads(Wn, y0, ts, w, matmul, C, max_steps=32)
    ref, _ = _replay_grads(Wn, y0, ts, w, grid, nacc)
    for name, g, r in zip(("y0", "W1", "b1", "W2", "b2", "W3", "b3"), grads, ref):
        rel = float((g - r).abs().max() / r.abs().max())
        print(f"{matmul} {name}: {rel:.2e}")
        assert rel < 2e-6, (name, rel)
