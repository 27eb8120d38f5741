"""Attributes that the library sets on its kernels, on the stand-in runtime."""
from hip_stub import run


def test_lds_limits_do_not_depend_on_the_call(tmp_path):
    """A kernel's LDS limit belongs to the kernel, and callers of several
    threads share it: films of any depth and size set the same one, or a
    launch could meet another call's smaller limit."""
    run(tmp_path, r"""
p = stub.stub_device(1 << 26)
seen = {}
for dims in ((64, 64, 5), (64, 64, 9), (64, 64, 16), (200, 200, 5), (200, 200, 16), (300, 500, 8), (300, 257, 5),
             (90, 70, 1), (70, 90, 2), (128, 120, 3), (128, 120, 4), (8, 8, 2), (50, 40, 3), (5, 1000, 1)):
    stub.stub_clear()
    assert lib.mms_potential_exact_noalloc(p, p, *dims, F(5e-9), F(5e-9), F(5e-9), None) == 0, mg.last_error()
    assert stub.stub_launches() and limits()
    for kernel, value in limits():
        assert seen.setdefault(kernel, value) == value, dims
""")
