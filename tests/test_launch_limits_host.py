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


def test_a_call_without_kept_tables_is_three_launches(tmp_path):
    """Where the transforms serve the call that allocates nothing, their tables
    are formed in the launches that transform the charges."""
    run(tmp_path, r"""
p = stub.stub_device(1 << 26)
for dims in ((33, 32, 6), (1300, 5, 1), (9, 1030, 2), (64, 129, 1), (20, 20, 16), (300, 300, 3)):
    stub.stub_clear()
    assert lib.mms_potential_exact_noalloc(p, p, *dims, F(5e-9), F(5e-9), F(5e-9), None) == 0, mg.last_error()
    assert stub.stub_launches() == 3, (dims, stub.stub_launches())
""")


def test_the_scratch_serves_every_grid_up_to_its_cells(tmp_path):
    """The largest tables and work arrays: 1025 x 136 x 15 has the most."""
    run(tmp_path, r"""
p = stub.stub_device(1 << 26)
for dims in ((1025, 136, 15), (1025, 146, 14), (1025, 292, 7), (2048, 1024, 1), (2048, 64, 16), (65, 2016, 16),
             (128, 1024, 16), (1, 131072, 16), (2097152, 1, 1)):
    assert lib.mms_potential_exact_noalloc(p, p, *dims, F(5e-9), F(5e-9), F(5e-9), None) == 0, (dims, mg.last_error())
assert lib.mms_potential_exact_noalloc(p, p, 2097153, 1, 1, F(5e-9), F(5e-9), F(5e-9), None) != 0
""")


def test_reference_order_form_by_width(tmp_path):
    """One launch (the dividing kernel) for films one cell wide, five (flag,
    charges, pairs, join and the dividing kernel's check) for wider ones."""
    run(tmp_path, r"""
for dims, want in (((1, 5000, 1), 1), ((1, 100, 150), 1), ((2, 2500, 1), 5), ((5000, 1, 1), 5), ((2, 2000, 1), 1)):
    with mg.Film(*dims, F(5e-9), F(5e-9), F(5e-9), solver=mg.SOLVER_DIRECT_REFGPU) as f:
        stub.stub_clear()
        f.potential(np.ones(int(np.prod(dims)), F))
        assert stub.stub_launches() == want, (dims, stub.stub_launches())
""")
