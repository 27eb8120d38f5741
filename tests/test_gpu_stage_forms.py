"""The forms of the stencil kernels -- one cell per thread and layer below
1,048,576 cells, four cells per thread or a column walk from there on -- give
the column walk's results bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F = np.float32
D = (F(5e-9), F(4e-9), F(3e-9))


def _film(dims, seed):
    rng = np.random.default_rng(seed)
    n = int(np.prod(dims))
    mat = (rng.random(n) < 0.8).astype(np.uint8)
    M = rng.standard_normal((n, 3))
    M = (M / np.linalg.norm(M, axis=1, keepdims=True) * 8.6e5 * mat[:, None]).astype(F).ravel()
    return mat, M


# one cell, one layer, ragged small films; both sides of the line; four-cell and one-cell widths above it
@pytest.mark.parametrize("dims", [(1, 1, 1), (65, 3, 1), (70, 9, 2), (37, 11, 5), (1024, 511, 2), (1024, 512, 2),
                                  (701, 500, 3)])
def test_stage_forms_match_the_column_walk(mg, orc, dims, monkeypatch):
    mat, M = _film(dims, dims[0])
    out = []
    for one in ("0", "1"):
        monkeypatch.setenv("MMS_GPU_STAGE_ONE_CELL", one)
        with mg.Film(*dims, *D, external=mg.EXT_RAMP, material=mat) as f:
            f.set_m(M)
            f.steps(2, 1e-14, use_graph=False)
            out.append(f.get_m())
    assert np.array_equal(out[0], out[1])


# the run-time form with every extra input and output, and the field and charge kernels
@pytest.mark.parametrize("dims", [(33, 18, 4), (20, 21, 1)])
def test_rk4_step_forms_match_the_column_walk(mg, orc, dims, monkeypatch):
    mat, M = _film(dims, 3)
    n = mat.size
    out = []
    for one in ("0", "1"):
        monkeypatch.setenv("MMS_GPU_STAGE_ONE_CELL", one)
        a = [np.full(3 * n, F(7)) for _ in range(4)]
        ch, pot = np.zeros(n, F), np.zeros(n, F)
        args = (*dims, *D, 3, F(1.2566371e-6), F(8.6e5), F(1.3e-11))
        assert mg.Hfield(M, a[1], ch, pot, F(0), *args, 1, 1, 1, 1) == 0
        assert np.array_equal(ch, orc.divergence_3d(M, dims, D))
        st, _ = mg.rk4_step(F(0), F(1e-14), mat, M, a[0], a[1], a[2], a[3], ch, pot, *args, F(0.5), F(2.211e5),
                            1, 1, 1, 1)
        assert st == 0, mg.last_error()
        out.append([v.copy() for v in a + [ch, pot]])
    for u, v in zip(*out):
        assert np.array_equal(u, v)
