"""Calls that are served although memory of a faster form cannot be had, on
the stand-in runtime."""
import pytest

from hip_stub import run


def test_time_marching_without_pinned_memory(tmp_path):
    run(tmp_path, f"import os; os.chdir({str(tmp_path)!r})" + r"""
dims, n = (16, 16, 2), 512
M = np.random.default_rng(1).standard_normal(3 * n).astype(F)
stub.stub_fail_pinned(1)
assert mg.time_marching(np.ones(n, np.uint8), M, F(0), F(1e-16), *dims, F(5e-9), F(5e-9), F(5e-9), 3, F(1.2566371e-6),
                        F(8.6e5), F(1.3e-11), F(0.5), F(2.211e5), 1, 1, 1, 0, sim_name="s") == 0, mg.last_error()
assert os.path.exists("s/Mdynamics.dat")
""")


@pytest.mark.parametrize("solver,dims", [(2, (100, 80, 1)), (0, (100, 80, 1)), (0, (600, 500, 2))])
def test_plans_without_the_memory_of_their_faster_form(tmp_path, solver, dims):
    """The reference-order sum keeps its dividing kernel, the direct sum its
    pair loop, whichever of the plan's allocations fails."""
    run(tmp_path, f"solver, dims = {solver}, {dims}" + r"""
film = lambda: mg.Film(*dims, F(5e-9), F(5e-9), F(5e-9), solver=solver)
stub.stub_fail_malloc(0)
q = np.ones(int(np.prod(dims)), F)
def launches(f):
    stub.stub_clear()
    f.potential(q)
    return stub.stub_launches()
with film() as f:
    total = stub.stub_mallocs()
    faster = launches(f)
for k in (total - 1, total):  # the plan's two allocations are the last
    stub.stub_fail_malloc(k)
    with film() as f:
        assert launches(f) == (1 if solver == 2 else 2), (k, faster)
""")
