"""The host side of the copies between the caller's arrays and the device, on
the stand-in runtime (no kernel runs: what set_m uploads, get_m downloads)."""
from hip_stub import run

FILM = r"""
n = int(sys.argv[3]) if len(sys.argv) > 3 else 200000
M = np.random.default_rng(n).standard_normal(3 * n).astype(F)
f = mg.Film(n, 1, 1, F(5e-9), F(5e-9), F(5e-9), demag=0)
stub.stub_clear()
"""


def test_uploads_below_the_threads_line_are_the_runtimes_copy(tmp_path):
    """One copy straight from the caller's array (2.4 MB; the pinned chunks are
    slower there), and through the chunks from 16 MiB on."""
    run(tmp_path, FILM + r"""
f.set_m(M)
assert [(s, b) for _, s, b in copies()] == [(M.ctypes.data, M.nbytes)], copies()
assert np.array_equal(f.get_m(), M)
n = (16 << 20) // 12 + 1
M = np.random.default_rng(n).standard_normal(3 * n).astype(F)
with mg.Film(n, 1, 1, F(5e-9), F(5e-9), F(5e-9), demag=0) as g:
    stub.stub_clear()
    g.set_m(M)
    assert len(copies()) > 1 and all(s != M.ctypes.data for _, s, _ in copies())
    assert np.array_equal(g.get_m(), M)
""")


def test_a_call_without_pinned_memory_is_the_runtimes_copy(tmp_path):
    """Where the chunks' memory cannot be had, both directions still serve
    every array, and the next call tries the chunks again."""
    run(tmp_path, FILM.replace("200000", "2000000") + r"""
stub.stub_fail_pinned(1)
f.set_m(M)
out = f.get_m()
assert np.array_equal(out, M) and len(copies()) == 2, copies()
stub.stub_fail_pinned(0)
stub.stub_clear()
f.set_m(-M)
assert np.array_equal(f.get_m(), -M) and len(copies()) > 2
""")
