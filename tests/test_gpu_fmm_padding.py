"""Films much smaller than their padded square: the FMM passes run on the
boxes that hold cells only, against the FP64 FMM oracle on the whole square."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F = np.float32
D5 = (F(5e-9),) * 3


# a strip of tiles in x, in y; one box column past a tile; leaf width 2 (leaf locals through memory)
@pytest.mark.parametrize("dims,leaf", [((260, 60, 2), 4), ((36, 257, 1), 4), ((140, 30, 3), 2), ((520, 100, 1), 8)])
@pytest.mark.parametrize("form,tol", [("fp32", 2e-6), ("bf16x3", 2e-5)])
def test_fmm_on_the_boxes_that_hold_cells(mg, dims, leaf, form, tol):
    from oracle import fmm_oracle as fo
    xd, yd, zd = dims
    q = (np.random.default_rng(xd).normal(size=(zd, yd, xd)) * 1e14).astype(F)
    prec = {"fp32": mg.M2L_FP32, "bf16x3": mg.M2L_BF16X3}[form]
    with mg.Film(*dims, *D5, solver=mg.SOLVER_FMM, P=4, m2l_precision=prec, leaf_width=leaf) as f:
        # a state that is not finite must not reach the next one through the skipped boxes' sums
        f.potential(np.full(q.size, np.inf, F))
        pot = f.potential(q.ravel())
    ref = fo.FmmOracle(xd, yd, zd, 4, w=leaf).potential_units(q.astype(float)).ravel() * float(D5[0]) ** 2
    assert np.linalg.norm(pot - ref) / np.linalg.norm(ref) < tol


# both sides of the line between the narrow and the wide M2L workgroups, one and two target layers in the last group
@pytest.mark.parametrize("dims,P", [((96, 96, 3), 4), ((96, 96, 1), 6), ((250, 190, 4), 6), ((300, 280, 3), 6),
                                    ((300, 280, 3), 3)])
@pytest.mark.parametrize("form,tol", [("fp32", 2e-6), ("bf16x3", 2e-5)])
def test_m2l_workgroup_shapes(mg, dims, P, form, tol):
    from oracle import fmm_oracle as fo
    xd, yd, zd = dims
    q = (np.random.default_rng(yd).normal(size=(zd, yd, xd)) * 1e14).astype(F)
    prec = {"fp32": mg.M2L_FP32, "bf16x3": mg.M2L_BF16X3}[form]
    with mg.Film(*dims, *D5, solver=mg.SOLVER_FMM, P=P, m2l_precision=prec, leaf_width=4) as f:
        pot = f.potential(q.ravel())
    ref = fo.FmmOracle(xd, yd, zd, P, w=4).potential_units(q.astype(float)).ravel() * float(D5[0]) ** 2
    assert np.linalg.norm(pot - ref) / np.linalg.norm(ref) < tol
