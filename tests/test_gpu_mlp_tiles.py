"""The neural-ODE kernel's choice of wavefronts per tile over the batch size: one tile and its
remainders, and both sides of one tile per CU (256 tiles of 32).  Every row equals the row
of a solve in another batch, bit for bit, and the vector field a float64 evaluation."""
import numpy as np
import pytest
import torch

import diffrax_amd as dfx
from diffrax_amd import _mlp

pytestmark = pytest.mark.gpu


def _field(cuda, matmul, seed=3):
    rng = np.random.default_rng(seed)
    shapes = [(256, 64), (256,), (256, 256), (256,), (64, 256), (64,)]
    P = [rng.normal(0.0, np.sqrt(2.0 / sum(s)) if len(s) == 2 else 0.1, size=s) for s in shapes]
    return dfx.MLPField(*[torch.tensor(p, dtype=torch.float32, device=cuda) for p in P],
                        matmul=matmul)


@pytest.mark.parametrize("matmul", ["f32", "bf16"])
@pytest.mark.parametrize("B", [1, 31, 32, 33, 8192, 8193])
def test_rows_do_not_depend_on_the_batch_or_the_waves(cuda, matmul, B):
    term = dfx.ODETerm(_field(cuda, matmul))
    y = torch.tensor(np.random.default_rng(1).normal(size=(8200, 64)), dtype=torch.float32,
                     device=cuda)
    ts = torch.linspace(0.0, 1.0, 4, dtype=torch.float64)

    def solve(y0, launch=None):
        return dfx.diffeqsolve(term, dfx.Tsit5(), 0.0, 1.0, 0.1, y0, saveat=dfx.SaveAt(ts=ts),
                               stepsize_controller=dfx.PIDController(rtol=1e-5, atol=1e-7),
                               launch=launch)
    ref = solve(y[-B - 3:].clone(), launch=4 if B < 8000 else 8)
    for launch in (None, 4, 8):   # the batch of ref without its first row: other tiles
        got = solve(y[-B - 2:-2].clone(), launch)
        assert torch.equal(got.ys, ref.ys[1:1 + B])
        assert torch.equal(got.stats["num_steps"], ref.stats["num_steps"][1:1 + B])


@pytest.mark.parametrize("matmul", ["f32", "bf16"])
@pytest.mark.parametrize("R", [1, 32, 45])
def test_vector_field_against_float64(cuda, matmul, R):
    vf = _field(cuda, matmul, seed=8)
    y = torch.tensor(np.random.default_rng(R).normal(size=(R, 64)), dtype=torch.float32,
                     device=cuda)
    want = vf(0.0, y.double())
    # 2^-24 relative per product and sum of up to 256 terms of size about 1, and the hardware
    # exp2 / log2 / rcp of the activations at 1 ulp: 2e-6, the vector field's bar
    assert (_mlp.mlp_eval(vf, y).double() - want).abs().max() < 2e-6
