"""Charges (div M) of every kernel that forms them, against the oracle's
reference stencil bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F = np.float32
D = (F(5e-9), F(4e-9), F(3e-9))


def _hfield(mg, M, dims, use_fmm):
    n = int(np.prod(dims))
    H, ch, pot = np.zeros(3 * n, F), np.zeros(n, F), np.zeros(n, F)
    assert mg.Hfield(M, H, ch, pot, F(0), *dims, *D, 3, F(1.2566e-6), F(8.6e5), F(1.3e-11), 1, 1, 0, use_fmm) == 0
    return ch, pot


# the potential's own kernels: 1/r table and transforms; the FMM's upward pass
@pytest.mark.parametrize("dims,use_fmm", [((30, 21, 3), 0), ((70, 45, 3), 0), ((30, 21, 3), 1)])
def test_quotients_beyond_the_float_range(mg, orc, dims, use_fmm):
    """Differences whose quotient by the cell size overflows give infinities
    of their sign, and NaN only where the stencil's sum has both."""
    n = int(np.prod(dims))
    M = (np.random.default_rng(n).normal(size=3 * n) * 5e5).astype(F)
    big = np.random.default_rng(1).integers(0, 3 * n, 40)
    M[big] = np.where(np.arange(40) % 2, F(1), F(-1)) * F(2.0) ** (98 + np.arange(40) % 29)
    ch, _ = _hfield(mg, M, dims, use_fmm)
    with np.errstate(all="ignore"):
        want = orc.divergence_3d(M, dims, D)
    assert np.isinf(want).sum() >= 20
    assert np.array_equal(ch, want, equal_nan=True)
