"""What an SDE solve records for its gradient (CPU only: no kernel is launched)."""
import pytest
import torch

from diffrax_amd import _sde


def _record(N, checkpoints, dtype, P=300, d=8):
    z = torch.zeros(d, dtype=dtype)
    s = _sde._Sde(torch.zeros((P, d), dtype=dtype), z, z, z, torch.zeros((N, P, d)),
                  torch.linspace(0.0, 1.0, N + 1, dtype=torch.float64), False, True, True,
                  checkpoints)
    assert (s.ckpt is None) != (s.sens is None)
    assert bool(s.io.ckpt) != bool(s.io.sens)
    return s


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("N", [1, 8, 9, 40, 100])
def test_a_given_number_of_checkpoints_bounds_the_record(N, dtype):
    """The derivatives' 2 P d + 2 d float64 take the checkpoints' place only within the
    checkpoints' bytes; by default always."""
    assert _record(N, None, dtype).sens is not None
    for checkpoints in (1, 2, 5, 100):
        s = _record(N, checkpoints, dtype)
        states = max(-(-N // _sde._ck_for(N, checkpoints)) - 1, 1)
        rec = s.sens if s.sens is not None else s.ckpt
        assert rec.numel() * rec.element_size() <= states * 300 * 8 * dtype.itemsize
    assert _record(100, 100, dtype).sens is not None
