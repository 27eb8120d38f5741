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


def test_memory_the_runtime_knows_is_copied_directly(tmp_path):
    """Pinned and device arrays of the caller, also inside a larger
    allocation, go to the runtime as they are; a call's pageable arrays beside
    them take the chunks if they are large enough by themselves."""
    run(tmp_path, FILM.replace("200000", "2000000") + r"""
check = lambda rc: (_ for _ in ()).throw(AssertionError(mg.last_error())) if rc else None
for alloc in (stub.stub_pin, stub.stub_device):
    p = alloc(M.nbytes + 64) + 64
    C.memmove(p, M.ctypes.data, M.nbytes)
    a = np.ctypeslib.as_array((C.c_float * M.size).from_address(p))
    stub.stub_clear()
    f.set_m(a)
    assert [(s, b) for _, s, b in copies()] == [(p, M.nbytes)], copies()
    a[:] = 0
    stub.stub_clear()
    check(lib.mms_get_m(f._ctx, a))
    assert [(d, b) for d, _, b in copies()] == [(p, M.nbytes)] and np.array_equal(a, M)
# Hfield's three results, the field pinned: the others (16 MB) by chunks
n, dims, d = 2000000, (2000, 1000, 1), (F(5e-9),) * 3
H = np.ctypeslib.as_array((C.c_float * (3 * n)).from_address(stub.stub_pin(12 * n)))
ch, pot = np.full(n, F(7)), np.full(n, F(7))
stub.stub_clear()
assert mg.Hfield(M, H, ch, pot, F(0), *dims, *d, 3, F(1.2566e-6), F(8.6e5), F(1.3e-11), 1, 1, 0, 1) == 0
to = [t for t, _, b in copies()]
assert to.count(H.ctypes.data) == 1 and ch.ctypes.data not in to and pot.ctypes.data not in to
assert not ch.any() and not pot.any()  # the stand-in's device memory
""")


def test_downloads_wait_once(tmp_path):
    """Chunks are waited for one by one, and the stream is not waited for
    again after them; the runtime's copies need that wait."""
    run(tmp_path, FILM + r"""
f.set_m(M)
stub.stub_clear()
assert np.array_equal(f.get_m(), M)  # 2.4 MB: chunks
assert len(copies()) > 1 and stub.stub_syncs() == 0
with mg.Film(1000, 1, 1, F(5e-9), F(5e-9), F(5e-9), demag=0) as g:
    g.set_m(M[:3000])
    stub.stub_clear()
    assert np.array_equal(g.get_m(), M[:3000])
    assert len(copies()) == 1 and stub.stub_syncs() == 1
""")
