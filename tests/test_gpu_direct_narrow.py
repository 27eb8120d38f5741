"""The LDS-table form of the exact pair sum: films that fill their groups of
four targets poorly, on both sides of the chip's 256 workgroups, and cell
sizes on both sides of the range in which the charges' divisions are by a
corrected reciprocal."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F = np.float32


# 2046, 2048 and 2050 groups; a single group; x remainders 1 to 3
@pytest.mark.parametrize("dims", [(1, 682, 3), (2, 1024, 2), (5, 205, 5), (3, 1, 1), (37, 40, 3)])
@pytest.mark.parametrize("d", [(5e-9, 4e-9, 3e-9), (7.3e-9, 7.3e-9, 7.3e-9), (1e-20, 1e-20, 1e-20), (1.0, 2.0, 0.7)])
def test_charge_and_potential(mg, orc, dims, d):
    d = tuple(F(v) for v in d)
    n = int(np.prod(dims))
    M = (np.random.default_rng(n).normal(size=3 * n) * 5e5).astype(F)
    H, ch, pot = np.zeros(3 * n, F), np.zeros(n, F), np.zeros(n, F)
    assert mg.Hfield(M, H, ch, pot, F(0), *dims, *d, 0, F(1.2566e-6), F(8.6e5), F(1.3e-11), 1, 1, 0, 0) == 0
    assert np.array_equal(ch, orc.divergence_3d(M, dims, d))
    probes = np.unique(np.r_[0, n - 1, np.random.default_rng(1).integers(0, n, 200)])
    ex = orc.potential_probes_f64(ch, dims, d, probes)
    a = orc.potential_probes_f64(np.abs(ch), dims, d, probes)
    # at most 128 FP32 products a piece, as for the form's other shapes
    assert np.all(np.abs(pot[probes].astype(float) - ex) <= 131 * 2.0 ** -24 * a + 2.0 ** -23 * np.abs(ex))
