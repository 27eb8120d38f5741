"""One cell per thread and layer against the column walk over hundreds of
steps: the same states bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.mark.parametrize("dims,kw", [((70, 45, 1), dict(demag=0)), ((100, 90, 2), dict(solver=1, P=4)),
                                     ((256, 256, 3), dict(solver=1, P=4)), ((37, 41, 5), dict(solver=0)),
                                     ((1023, 700, 2), dict(demag=0))])
def test_states_after_many_steps(mg, dims, kw, monkeypatch):
    n = int(np.prod(dims))
    M = np.random.default_rng(n).standard_normal((n, 3))
    M = (M / np.linalg.norm(M, axis=1, keepdims=True) * 8.6e5).astype(F).ravel()
    out = []
    for walk in ("0", "1"):
        monkeypatch.setenv("MMS_GPU_STAGE_ONE_CELL", walk)
        with mg.Film(*dims, F(5e-9), F(4e-9), F(3e-9), **kw) as f:
            f.set_m(M)
            f.steps(300, 1e-13)
            out.append((f.get_m(), f.hfield()))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
    assert not np.array_equal(out[0][0], M)
