"""The call that allocates nothing, captured into a graph: every replay forms
its tables and potential anew from the charges then in the device array."""
import ctypes as C

import numpy as np
import pytest

from test_zz_no_alloc import _Hip

pytestmark = pytest.mark.gpu
F = np.float32
D = (F(5e-9), F(4e-9), F(3e-9))


# the 1/r table, the transforms with their tables (few and many layers), the pair loop
@pytest.mark.parametrize("dims", [(32, 32, 3), (70, 65, 2), (33, 32, 6), (31, 31, 18)])
def test_captured_call(mg, dims):
    hip = _Hip(mg)
    h = hip.h
    n = int(np.prod(dims))
    rng = np.random.default_rng(n)
    stream, graph, run = C.c_void_p(), C.c_void_p(), C.c_void_p()
    try:
        dq, dp = hip.alloc(4 * n), hip.alloc(4 * n)
        assert h.hipStreamCreateWithFlags(C.byref(stream), 1) == 0
        assert h.hipStreamBeginCapture(stream, 1) == 0
        rc = mg.lib().mms_potential_exact_noalloc(dq, dp, *dims, *D, stream)
        assert h.hipStreamEndCapture(stream, C.byref(graph)) == 0 and rc == 0, mg.last_error()
        assert h.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)) == 0
        for k in range(4):
            q = (rng.normal(size=n) * 1e14).astype(F)
            assert h.hipMemcpy(dq, q.ctypes.data_as(C.c_void_p), q.nbytes, 1) == 0
            assert h.hipGraphLaunch(run, stream) == 0 and h.hipStreamSynchronize(stream) == 0
            want = np.zeros(n, F)
            assert mg.calc_potential_exact(q, *dims, *D, want, 1, 0) == 0
            assert np.array_equal(hip.get(dp, n), want), k
            # the scratch in another call's hands between two replays
            a, b = hip.alloc(4 * 12000), hip.alloc(4 * 12000)
            assert h.hipMemset(a, 0, 4 * 12000) == 0
            assert mg.lib().mms_potential_exact_noalloc(a, b, 100, 60, 2, *D, None) == 0
            assert h.hipDeviceSynchronize() == 0
    finally:
        if run:
            h.hipGraphExecDestroy(run)
        if graph:
            h.hipGraphDestroy(graph)
        if stream:
            h.hipStreamDestroy(stream)
        hip.free()
