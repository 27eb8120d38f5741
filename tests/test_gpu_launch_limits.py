"""Grids of many layers and batches of many films: more than 65,535 layers, and
films x layers^2 beyond that number, take the forms whose launches fit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F = np.float32


def test_more_layers_than_a_grid_dimension(mg, orc, monkeypatch):
    dims, d = (1, 1, 65600), (F(5e-9),) * 3
    M = np.random.default_rng(1).standard_normal((dims[2], 3))
    M = (M / np.linalg.norm(M, axis=1, keepdims=True) * 8.6e5).astype(F).ravel()
    out = []
    for one in ("0", "1"):
        monkeypatch.setenv("MMS_GPU_STAGE_ONE_CELL", one)
        with mg.Film(*dims, *d, solver=mg.SOLVER_DIRECT, demag=0) as f:
            f.set_m(M)
            f.steps(2, 1e-14, use_graph=False)
            out.append(f.get_m())
    assert np.array_equal(out[0], out[1]) and np.all(np.isfinite(out[0]))


def test_many_deep_films_in_a_batch(mg):
    nf, dims, d = 660, (21, 20, 10), (F(5e-9),) * 3  # 660 * 10^2 > 65535
    n = int(np.prod(dims))
    q = (np.random.default_rng(2).normal(size=(nf, n)) * 1e14).astype(F)
    with mg.FilmBatch([(dims[0], dims[1], (0.0, 0.0, 0.0))] * nf, dims[2], *d, solver=mg.SOLVER_FMM, P=2) as b:
        pot = b.potential(q).reshape(nf, n)
    with mg.Film(*dims, *d, solver=mg.SOLVER_FMM, P=2) as f:
        for k in (0, 331, nf - 1):
            ref = f.potential(q[k])
            assert np.linalg.norm(pot[k] - ref) <= 2e-6 * np.linalg.norm(ref)  # FP32 sums in another order
