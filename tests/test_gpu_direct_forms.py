"""The exact pair sum's forms: the 1/r table in LDS (small grids) and the FP64
transforms (larger ones), against FP64 direct sums of the oracle.

Tolerances: with A = sum_j |rho_j| dV / r at a cell, the table form adds at
most 128 FP32 products a piece (the table entry's, the product's and the
sums' roundings: (128 + 3) 2^-24 A); the transforms are FP64 (their error is
under 1e-13 of the largest A) and round once to FP32."""
import numpy as np
import pytest

from test_zz_no_alloc import _Hip

pytestmark = pytest.mark.gpu
F = np.float32
U = 2.0 ** -24


def _charge(n, seed):
    return (np.random.default_rng(seed).normal(size=n) * 1e14).astype(F)


def _check(orc, pot, q, dims, d, table):
    n = q.size
    probes = np.arange(n) if n <= 20000 else np.unique(np.r_[0, n - 1, np.random.default_rng(1).integers(0, n, 300)])
    ex = orc.potential_probes_f64(q, dims, d, probes)
    a = orc.potential_probes_f64(np.abs(q), dims, d, probes)
    tol = (131 * U * a if table else 1e-13 * a.max()) + 2 * U * np.abs(ex)
    err = np.abs(pot[probes].astype(float) - ex)
    assert np.all(err <= tol), float((err / tol).max())


# table: one cell, single rows and columns, a row of several pieces, group and row remainders, the largest
# transforms: every padded length of either axis, one to five and sixteen layers, odd sides
@pytest.mark.parametrize("dims,table", [((1, 1, 1), True), ((5, 1, 1), True), ((1, 37, 2), True), ((1025, 1, 3), True),
                                        ((31, 29, 5), True), ((40, 50, 3), True),
                                        ((33, 32, 6), False), ((32, 33, 7), False), ((65, 31, 5), False),
                                        ((64, 129, 1), False), ((257, 90, 2), False), ((128, 61, 16), False),
                                        ((513, 40, 4), False), ((40, 513, 3), False), ((1025, 9, 2), False),
                                        ((9, 1030, 2), False), ((2048, 4, 1), False)])
def test_direct_forms_against_fp64(mg, orc, dims, table):
    d = (F(5e-9), F(4e-9), F(3e-9))
    q = _charge(int(np.prod(dims)), dims[0])
    pot = np.full(q.size, np.nan, F)
    assert mg.calc_potential_exact(q, *dims, *d, pot, 1, 0) == 0, mg.last_error()
    _check(orc, pot, q, dims, d, table)
    # the entry point that allocates nothing takes the same form
    hip = _Hip(mg)
    try:
        dq, dp = hip.put(q), hip.alloc(q.nbytes)
        assert mg.lib().mms_potential_exact_noalloc(dq, dp, *dims, *d, None) == 0, mg.last_error()
        assert np.array_equal(hip.get(dp, q.size), pot)
    finally:
        hip.free()


@pytest.mark.parametrize("dims", [(30, 21, 3), (1, 9, 4), (70, 45, 3), (66, 64, 2)])
def test_charge_formed_in_the_potential_kernels(mg, orc, dims):
    """Hfield's charge (formed by the potential's own kernels) is the
    reference stencil's bit for bit, its potential that of this charge."""
    d = (F(5e-9), F(4e-9), F(3e-9))
    n = int(np.prod(dims))
    M = (np.random.default_rng(n).normal(size=3 * n) * 5e5).astype(F)
    H, ch, pot = np.zeros(3 * n, F), np.zeros(n, F), np.zeros(n, F)
    assert mg.Hfield(M, H, ch, pot, F(0), *dims, *d, 0, F(1.2566e-6), F(8.6e5), F(1.3e-11), 1, 1, 0, 0) == 0
    assert np.array_equal(ch, orc.divergence_3d(M, dims, d))
    ref = np.zeros(n, F)
    assert mg.calc_potential_exact(ch, *dims, *d, ref, 1, 0) == 0
    assert np.array_equal(pot, ref)


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_transforms_leave_nonfinite_charges_to_the_pair_sum(mg, bad):
    """One charge that is not finite: every other cell's potential is that
    value, the cell's own is NaN (0 times it), as the pair loop gives; the
    next call on the same film is unaffected."""
    dims = (64, 50, 3)
    d = (F(5e-9),) * 3
    q = _charge(int(np.prod(dims)), 3)
    good, again, pot = (np.zeros_like(q) for _ in range(3))
    assert mg.calc_potential_exact(q, *dims, *d, good, 1, 0) == 0
    b = q.copy()
    b[4321] = bad
    assert mg.calc_potential_exact(b, *dims, *d, pot, 1, 0) == 0
    other = np.delete(pot, 4321)
    assert np.isnan(pot[4321]) and (np.all(np.isnan(other)) if np.isnan(bad) else np.all(other == bad))
    assert mg.calc_potential_exact(q, *dims, *d, again, 1, 0) == 0
    assert np.array_equal(again, good) and np.all(np.isfinite(good))


# the reference's order from the 1/r table: first size that takes it and the last that does not, rows shorter and
# longer than a chunk, sources in one row or one column, a last chunk that is cut and chunks without sources
@pytest.mark.parametrize("dims", [(64, 64, 1), (65, 63, 1), (4100, 1, 1), (1, 4100, 1), (1, 1, 4099), (37, 12, 11),
                                  (5, 900, 1), (1025, 4, 1)])
def test_reference_order_table_against_the_restated_kernel(mg, orc, dims):
    n = int(np.prod(dims))
    q = _charge(n, n)
    q[::7] = 0.0
    d = (F(5e-9), F(4e-9), F(3e-9))
    pot = np.full(n, np.nan, F)
    assert mg.calc_potential_exact_gpu(q, *dims, *d, pot) == 0, mg.last_error()
    assert np.array_equal(pot, orc.calc_potential_exact_refgpu(q, dims, d))


@pytest.mark.parametrize("dims", [(70, 61, 1), (512, 513, 1)])
def test_reference_order_table_and_division_agree(mg, dims):
    """A charge so small that its quotients are denormal sends the call to the
    dividing kernel; it changes no sum, so both give the same bits."""
    n = int(np.prod(dims))
    q = _charge(n, 5)
    q[n // 3] = 0.0
    d = (F(5e-9),) * 3
    a, b = np.zeros(n, F), np.zeros(n, F)
    assert mg.calc_potential_exact_gpu(q, *dims, *d, a) == 0
    q[n // 3] = F(1e-21)  # q dV about 1e-46, 0 in float or denormal
    q[n // 3 + 1] = F(1e-19)
    assert mg.calc_potential_exact_gpu(q, *dims, *d, b) == 0
    q[n // 3 + 1] = 0.0
    q[n // 3] = 0.0
    assert mg.calc_potential_exact_gpu(q, *dims, *d, a) == 0
    assert np.array_equal(a, b)


def test_reference_order_leaves_nonfinite_charges_to_the_division(mg, orc):
    dims, d = (80, 60, 1), (F(5e-9),) * 3
    q = _charge(4800, 6)
    for bad in (np.inf, np.nan):
        q[1234] = bad
        pot = np.zeros(4800, F)
        assert mg.calc_potential_exact_gpu(q, *dims, *d, pot) == 0
        assert np.array_equal(pot, orc.calc_potential_exact_refgpu(q, dims, d), equal_nan=True)
