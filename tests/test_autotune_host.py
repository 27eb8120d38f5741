"""What the autotuner tries for the direct sum's forms, on the stand-in runtime."""
import pytest

from hip_stub import run


@pytest.mark.parametrize("dims,form", [((24, 24, 4), "table"), ((64, 64, 3), "transforms"), ((40, 40, 17), "chunks")])
def test_source_chunks_are_tuned_where_there_are_any(tmp_path, dims, form):
    """The table and transform forms have nothing to choose: the shape stays as
    it was asked for and no solve is timed.  The pair loop's three candidates
    are timed (the stand-in's clock makes the first the fastest)."""
    run(tmp_path, f"dims, form = {dims}, '{form}'" + r"""
with mg.Film(*dims, F(5e-9), F(5e-9), F(5e-9), solver=mg.SOLVER_DIRECT, direct_split=2) as f:
    stub.stub_clear()
    rep = f.autotune(reps=2)
    assert "chosen" in rep, rep
    if form == "chunks":
        assert [l[:14] for l in rep.splitlines()[:3]] == [f"direct split={k}" for k in (1, 2, 4)], rep
        assert f.shape()["direct_split"] == 1
    else:
        assert "split" not in rep and form in rep and f.shape()["direct_split"] == 2, rep
        assert stub.stub_launches() <= 1  # the charge
""")
