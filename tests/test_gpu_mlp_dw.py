"""The weight-gradient GEMM by itself: dW of one segment against the float64 products of the
very rows (deltas and layer inputs) that the segment left in its row buffers."""
import ctypes
import math

import numpy as np
import pytest
import torch

import diffrax_amd as dfx
from diffrax_amd import _lib, _mlp
from tests.test_gpu_mlp_grad import _weights

pytestmark = pytest.mark.gpu

WIDTHS = (256, 64, 256, 256, 64, 256)   # delta1, z, delta2, h1, delta3, h2


def _segment(cuda, matmul, B, steps):
    """One segment of `steps` equal steps; returns the six row matrices and dW."""
    rng = np.random.default_rng(3)
    W = [torch.tensor(a, dtype=torch.float32, device=cuda) for a in _weights()]
    y0 = torch.tensor(rng.normal(size=(B, 64)).astype(np.float32), device=cuda)
    plan = _mlp.prepare_mlp(dfx.ODETerm(dfx.MLPField(*W, matmul=matmul)), dfx.Tsit5(), 0.0, 1.0,
                            1.0 / steps, y0, dfx.SaveAt(t1=True),
                            dfx.PIDController(rtol=1.0, atol=1.0, dtmax=1.0 / steps), steps, cuda,
                            ckpt_every=steps)
    plan.launch()
    assert plan.max_accepted() == steps and int(plan.stats[:, 1].min()) == steps
    lib, sizes = _lib.load(), [ctypes.c_size_t(0) for _ in range(3)]
    _lib.check(lib.dfx_mlp_adj_workspace(ctypes.byref(plan.prob), steps, *map(ctypes.byref, sizes)))
    zs, rows, part = (torch.empty(s.value // 4, device=cuda) for s in sizes)
    ybar = torch.tensor(rng.normal(size=(B, 64)).astype(np.float32), device=cuda)
    ys_bar, dw = ybar[:, None].clone(), torch.zeros(98880, device=cuda)
    io = _mlp.MlpAdjIO(grid=plan.grid.data_ptr(), ckpt=plan.ckpt.data_ptr(),
                       stats=plan.stats.data_ptr(), ys_bar=ys_bar.data_ptr(),
                       ybar=ybar.data_ptr(), zs=zs.data_ptr(), rows=rows.data_ptr(),
                       partial=part.data_ptr(), dw=dw.data_ptr())
    _lib.check(lib.dfx_mlp_adj_segment(
        ctypes.byref(plan.prob), ctypes.c_void_p(plan.packed.data_ptr()),
        *(ctypes.c_void_p(b.data_ptr()) for b in plan.b), ctypes.byref(io), 0, steps,
        _mlp._stream()))
    blocks, off, out = -(-B // 32) * (1 + 6 * steps), 0, []
    alloc = rows.numel() // sum(WIDTHS)
    for w in WIDTHS:   # blocks of 32 rows: [column / 32][row / 8][row / 4 % 2][column % 32][row % 4]
        buf = rows[off:off + blocks * 32 * w].view(blocks, w // 32, 4, 2, 32, 4)
        out.append(buf.permute(0, 2, 3, 5, 1, 4).reshape(blocks * 32, w))
        off += alloc * w
    return out, dw, blocks


@pytest.mark.parametrize("matmul,B,steps", [("f32", 1, 1), ("f32", 70, 1), ("bf16", 70, 4),
                                            ("f32", 2048, 4), ("f32", 8192, 64)])
def test_weight_gradient_of_the_rows(cuda, matmul, B, steps):
    """Bound, of the largest element: float32 rounding (2^-24 of the running sum, which stays
    below the result's largest) of every accumulation of one accumulator, six products of 16
    rows each, independent of one another, so their root; no accumulator sums more than 4,096
    rows; and 8 units for the chunks' sum and the products of pieces left out.  Without the
    third pieces the sums would be off by 6e-6."""
    rows, dw, blocks = _segment(cuda, matmul, B, steps)
    per_chunk = max(min(4, blocks), min(128, math.ceil(blocks / 80)))
    tol = (8.0 + math.sqrt(per_chunk * 32 / 16 * 6)) * 2.0 ** -24
    off = 0
    for a, b in ((0, 1), (2, 3), (4, 5)):
        ref = torch.zeros(rows[a].shape[1], rows[b].shape[1], dtype=torch.float64, device=cuda)
        for i in range(0, rows[a].shape[0], 1 << 16):
            ref += rows[a][i:i + (1 << 16)].double().T @ rows[b][i:i + (1 << 16)].double()
        got = dw[off:off + ref.numel()].view_as(ref).double()
        off += ref.numel()
        err = float((got - ref).abs().max() / ref.abs().max())
        print(f"dW{a // 2 + 1}: {err:.2e} (bound {tol:.2e})")
        assert err < tol, (a, err, tol)
    for a in (0, 2, 4):   # the bias gradients: column sums of the deltas
        ref = rows[a].double().sum(0)
        got = dw[off:off + ref.numel()].double()
        off += ref.numel()
        assert float((got - ref).abs().max() / rows[a].double().abs().sum(0).max()) < 2.0 ** -20
