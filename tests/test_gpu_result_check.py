"""throw=True reads the result codes through dfx_check_results: the first code in batch order
that is neither successful nor an event raises, wherever it lies in its block's run."""
import numpy as np
import pytest
import torch

from diffrax_amd._integrate import raise_unless_okay
from diffrax_amd._solution import RESULTS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 255, 4096, 8191, 8192, 12289, 300_000])
def test_first_failure(cuda, n):
    codes = torch.zeros(n, dtype=torch.int32, device=cuda)
    raise_unless_okay(codes)
    codes.fill_(int(RESULTS.event_occurred))
    raise_unless_okay(codes)
    rng = np.random.default_rng(n)
    for at in sorted({0, n - 1, n // 2, int(rng.integers(n))}):
        codes[n // 3:].zero_()
        codes[at] = 2
        codes[at + 1:] = 1                              # later failures do not count
        with pytest.raises(RuntimeError) as e:
            raise_unless_okay(codes)
        assert e.value.args[0] == RESULTS[2]
        codes.fill_(int(RESULTS.event_occurred))
    with pytest.raises(RuntimeError):
        raise_unless_okay(codes, okay=0)


def test_empty(cuda):
    raise_unless_okay(torch.zeros(0, dtype=torch.int32, device=cuda))
