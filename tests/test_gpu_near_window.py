"""The 16-bit near field's charge window: rows that start on 16 bytes and rows
that do not, one layer to more than the registers hold, against the FP64 FMM oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F = np.float32
D5 = (F(5e-9),) * 3


# widths of every remainder by 4; edges one past a block of 64 x 32 cells; 1 to 6 layers (a group of four and its rest)
@pytest.mark.parametrize("dims", [(68, 36, 1), (65, 33, 3), (70, 70, 4), (67, 40, 5), (132, 64, 6)])
# tolerances: those of the same forms on whole films (FP16 and BF16 roundings of operator and charges)
@pytest.mark.parametrize("form,tol", [("BF16X3", 2e-5), ("FP16", 8e-4), ("FP16X2_FP16X2NEAR", 8e-4)])
def test_sixteen_bit_near_field_windows(mg, dims, form, tol):
    from oracle import fmm_oracle as fo
    xd, yd, zd = dims
    q = (np.random.default_rng(xd + zd).normal(size=(zd, yd, xd)) * 1e14).astype(F)
    with mg.Film(*dims, *D5, solver=mg.SOLVER_FMM, P=4, m2l_precision=getattr(mg, "M2L_" + form), leaf_width=8) as f:
        pot = f.potential(q.ravel())
    ref = fo.FmmOracle(xd, yd, zd, 4, w=8).potential_units(q.astype(float)).ravel() * float(D5[0]) ** 2
    assert np.linalg.norm(pot - ref) / np.linalg.norm(ref) < tol
