"""Small films at leaf width 4: the charges formed in the FMM's upward pass
against the charge kernel's, which a profiling window runs by itself.  Both
evaluate the same expression, so trajectories are equal bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F = np.float32
D5 = (F(5e-9),) * 3


# one layer, odd widths, cells past the last whole subtree, a strip, more than four layers
@pytest.mark.parametrize("dims,P", [((17, 16, 1), 3), ((33, 18, 2), 4), ((64, 64, 3), 3), ((161, 117, 4), 6),
                                    ((20, 260, 6), 2)])
@pytest.mark.parametrize("use_graph", [False, True])
def test_charges_in_the_upward_pass(mg, dims, P, use_graph):
    n = int(np.prod(dims))
    M = np.random.default_rng(n).normal(size=(n, 3))
    M = (M / np.linalg.norm(M, axis=1, keepdims=True) * 8.6e5).astype(F)
    out = []
    for profiled in (False, True):
        with mg.Film(*dims, *D5, solver=mg.SOLVER_FMM, P=P, leaf_width=4) as f:
            f.set_m(M)
            if profiled:
                f.profile_begin()
            f.steps(3, 1e-13, use_graph=use_graph and not profiled)
            f.sync()
            if profiled:
                f.profile_end()
            out.append(f.get_m())
    assert np.array_equal(out[0], out[1])
