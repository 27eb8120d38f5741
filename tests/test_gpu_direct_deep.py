"""Films of 5 to 16 layers by the transforms: every length of the column
kernel's products over 8 and 16 layers, against FP64 direct sums (tolerance
as in test_gpu_direct_forms: FP64 transforms, one rounding to FP32), and the
call that forms the tables itself bit for bit."""
import numpy as np
import pytest

from test_gpu_direct_forms import _charge, _check
from test_zz_no_alloc import _Hip

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.mark.parametrize("dims", [(20, 25, 16), (50, 11, 11), (70, 40, 9), (40, 100, 8), (30, 200, 16), (300, 150, 5),
                                  (20, 500, 8), (24, 260, 5), (5, 1000, 4), (3, 2048, 2), (600, 600, 1)])
def test_deep_films_against_fp64(mg, orc, dims):
    d = (F(5e-9), F(4e-9), F(3e-9))
    q = _charge(int(np.prod(dims)), dims[0])
    pot = np.full(q.size, np.nan, F)
    assert mg.calc_potential_exact(q, *dims, *d, pot, 1, 0) == 0, mg.last_error()
    _check(orc, pot, q, dims, d, False)
    hip = _Hip(mg)
    try:
        dq, dp = hip.put(q), hip.alloc(q.nbytes)
        for _ in range(2):
            assert mg.lib().mms_potential_exact_noalloc(dq, dp, *dims, *d, None) == 0, mg.last_error()
            assert np.array_equal(hip.get(dp, q.size), pot)
    finally:
        hip.free()
