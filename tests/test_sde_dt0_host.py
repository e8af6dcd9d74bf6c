"""A dt0 against which the span of a constant-step solve vanishes is refused (CPU only)."""
import math

import numpy as np
import pytest

from diffrax_amd import _sde


@pytest.mark.parametrize("t1,dt0", [(1.0, math.inf), (5e-324, 1e300)])
def test_no_steps_is_an_error(t1, dt0):
    with pytest.raises(ValueError):
        _sde.constant_grid(0.0, t1, dt0)


def test_one_step():
    assert np.array_equal(_sde.constant_grid(0.0, 1.0, 1e308), [0.0, 1.0])
