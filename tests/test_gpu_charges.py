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


# the charge kernel's forms, reached by the FMM above 524,288 cells: four cells a thread at 2, 3 and 4 layers, the column
# walk at a width that is no multiple of four (3, 4 and other layers), one cell per thread and layer below 1,048,576 cells
@pytest.mark.parametrize("dims", [(1024, 512, 2), (1000, 350, 3), (640, 410, 4), (701, 500, 3), (701, 380, 4),
                                  (1049, 1000, 1), (900, 600, 1), (449, 400, 3)])
def test_charge_kernels(mg, orc, dims, monkeypatch):
    n = int(np.prod(dims))
    M = (np.random.default_rng(n).standard_normal(3 * n) * 5e5).astype(F)
    M[np.random.default_rng(1).random(3 * n) < 0.2] = 0.0
    want = orc.divergence_3d(M, dims, D)
    for walk in ("0", "1"):
        monkeypatch.setenv("MMS_GPU_STAGE_ONE_CELL", walk)
        ch, _ = _hfield(mg, M, dims, 1)
        assert np.array_equal(ch, want), walk
