"""FP32 M2L with one, two and four column tiles a workgroup, against the FP64 FMM oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F = np.float32
D5 = (F(5e-9),) * 3


# one tile (small; leaf width 8; 64-slot blocks keep four), two (one round of four-tile workgroups), four
@pytest.mark.parametrize("dims,P,leaf", [((20, 17, 2), 4, 4), ((96, 70, 3), 6, 4), ((130, 70, 2), 6, 8),
                                         ((60, 60, 1), 7, 4), ((256, 250, 3), 3, 4), ((400, 300, 3), 5, 4)])
def test_fp32_m2l_column_tiles(mg, dims, P, leaf):
    from oracle import fmm_oracle as fo
    xd, yd, zd = dims
    q = (np.random.default_rng(yd).normal(size=(zd, yd, xd)) * 1e14).astype(F)
    with mg.Film(*dims, *D5, solver=mg.SOLVER_FMM, P=P, m2l_precision=mg.M2L_FP32, leaf_width=leaf) as f:
        pot = f.potential(q.ravel())
    ref = fo.FmmOracle(xd, yd, zd, P, w=leaf).potential_units(q.astype(float)).ravel() * float(D5[0]) ** 2
    assert np.linalg.norm(pot - ref) / np.linalg.norm(ref) < 2e-6  # FP32 rounding, as for whole films


# the 16-bit forms' shapes: one round of one tile, of two tiles, beyond
@pytest.mark.parametrize("dims,P,leaf", [((20, 17, 2), 4, 4), ((64, 60, 3), 6, 4), ((128, 120, 4), 6, 4),
                                         ((256, 250, 3), 3, 4), ((400, 300, 3), 5, 8)])
@pytest.mark.parametrize("form,tol", [("BF16X3", 2e-5), ("BF16", 3e-3), ("FP16", 8e-4), ("FP16X2", 8e-4)])
def test_sixteen_bit_m2l_column_tiles(mg, dims, P, leaf, form, tol):
    from oracle import fmm_oracle as fo
    xd, yd, zd = dims
    q = (np.random.default_rng(yd).normal(size=(zd, yd, xd)) * 1e14).astype(F)
    with mg.Film(*dims, *D5, solver=mg.SOLVER_FMM, P=P, m2l_precision=getattr(mg, "M2L_" + form), leaf_width=leaf) as f:
        pot = f.potential(q.ravel())
    ref = fo.FmmOracle(xd, yd, zd, P, w=leaf).potential_units(q.astype(float)).ravel() * float(D5[0]) ** 2
    assert np.linalg.norm(pot - ref) / np.linalg.norm(ref) < tol  # the forms' tolerances on whole films
