"""The pair loop over source chunks, which serves grids that neither the 1/r
table nor the transforms take (sides above 2,048, more than 16 layers, deep
films with long y sides), against FP64 direct sums of the oracle.

Tolerance, with A = sum_j |rho_j| dV / r at a cell and u = 2^-24: FP32 sums of
256 products (256 u A), 1/r by the hardware's reciprocal square root (one ulp,
2 u) of r^2 (two additions and three squares, 2 u after the root); with cell
sizes that are no powers of two apart the coordinates' products are rounded
too, 2 (side) u of a neighbour's distance.  FP64 over the chunks."""
import numpy as np
import pytest

from test_gpu_direct_forms import _charge
from test_zz_no_alloc import _Hip

pytestmark = pytest.mark.gpu
F = np.float32
U = 2.0 ** -24
EXACT, ODD = (F(4e-9), F(4e-9), F(2e-9)), (F(5e-9), F(4e-9), F(3e-9))


def _check(orc, pot, q, dims, d):
    n = q.size
    probes = np.unique(np.r_[0, n - 1, np.random.default_rng(1).integers(0, n, 400)])
    ex = orc.potential_probes_f64(q, dims, d, probes)
    a = orc.potential_probes_f64(np.abs(q), dims, d, probes)
    tol = (260 + (2 * max(dims[1:]) if d is ODD else 0)) * U * a + 2 * U * np.abs(ex)
    err = np.abs(pot[probes].astype(float) - ex)
    assert np.all(err <= tol), float((err / tol).max())


# a long row, a long column, many layers, a deep film with a long y side; sizes that fill their last block and chunk by one
@pytest.mark.parametrize("dims,d", [((2050, 9, 1), EXACT), ((9, 2050, 1), EXACT), ((31, 31, 18), ODD),
                                    ((64, 32, 17), ODD), ((3, 600, 10), EXACT), ((16641, 1, 1), EXACT)])
def test_chunks_against_fp64(mg, orc, dims, d):
    q = _charge(int(np.prod(dims)), dims[0])
    pot = np.full(q.size, np.nan, F)
    assert mg.calc_potential_exact(q, *dims, *d, pot, 1, 0) == 0, mg.last_error()
    _check(orc, pot, q, dims, d)
    hip = _Hip(mg)
    try:
        dq, dp = hip.put(q), hip.alloc(q.nbytes)
        assert mg.lib().mms_potential_exact_noalloc(dq, dp, *dims, *d, None) == 0, mg.last_error()
        assert np.array_equal(hip.get(dp, q.size), pot)
    finally:
        hip.free()


@pytest.mark.parametrize("split", [2, 4])
def test_source_chunk_multipliers(mg, orc, split):
    dims = (31, 31, 18)
    q = _charge(int(np.prod(dims)), 4)
    with mg.Film(*dims, *ODD, solver=mg.SOLVER_DIRECT, direct_split=split) as f:
        assert f.shape()["direct_split"] == split
        _check(orc, f.potential(q), q, dims, ODD)


def test_tuned_chunks(mg, orc):
    """The tuner's choice among the multipliers keeps the potential."""
    dims = (31, 31, 18)
    q = _charge(int(np.prod(dims)), 5)
    with mg.Film(*dims, *ODD, solver=mg.SOLVER_DIRECT) as f:
        rep = f.autotune(reps=2)
        assert rep.count("ms/solve") == 3 and f.shape()["direct_split"] in (1, 2, 4)
        _check(orc, f.potential(q), q, dims, ODD)


def test_charge_and_pair_loop_of_a_field_call(mg, orc):
    dims = (31, 31, 18)
    n = int(np.prod(dims))
    M = (np.random.default_rng(n).normal(size=3 * n) * 5e5).astype(F)
    H, ch, pot = np.zeros(3 * n, F), np.zeros(n, F), np.zeros(n, F)
    assert mg.Hfield(M, H, ch, pot, F(0), *dims, *ODD, 0, F(1.2566e-6), F(8.6e5), F(1.3e-11), 1, 1, 0, 0) == 0
    assert np.array_equal(ch, orc.divergence_3d(M, dims, ODD))
    _check(orc, pot, ch, dims, ODD)
