"""The time loop's text dump: the device's %g against the C library's."""
import os
import subprocess

import numpy as np
import pytest

F = np.float32
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

MAIN = r"""
#include <stdio.h>
#include "text_format.hpp"
static const mms::Pow10 T[] = {MMS_POW10_ROWS};
int main() {
    uint32_t u;
    while (fread(&u, 4, 1, stdin) == 1) {
        float f;
        memcpy(&f, &u, 4);
        char a[64], b[64] = {0};
        snprintf(a, sizeof a, "%g", f);
        const mms::GNum g = mms::g_split(f, T);
        mms::g_write(g, b);
        if (strcmp(a, b) || (int)strlen(a) != mms::g_length(g)) { printf("%08x %s %s\n", u, a, b); return 1; }
    }
    return 0;
}
"""


def _values():
    """Random bit patterns, every exponent's ends, the neighbours of powers of
    ten and of ties of six digits, zeros, infinities, NaNs."""
    rng = np.random.default_rng(5)
    u = [rng.integers(0, 2**32, 400000, dtype=np.uint64).astype(np.uint32)]
    e = np.arange(256, dtype=np.uint32) << np.uint32(23)
    u += [e, e + np.uint32(1), e + np.uint32(0x7fffff)]
    with np.errstate(over="ignore"):
        p = np.concatenate([np.array([10.0 ** k for k in range(-45, 39)]),
                            (np.arange(100000, 1000000, 997)[:, None] + 0.5).ravel() / 4,
                            (np.arange(100000, 999999, 1013) + 0.5) * 1e3, np.arange(999990, 1000010) + 0.5]).astype(F)
    v = p.view(np.uint32)
    u += [v, v - np.uint32(1), v + np.uint32(1)]
    u = np.concatenate(u)
    return np.concatenate([u, u | np.uint32(1 << 31)])


def test_format_agrees_with_the_c_library(tmp_path):
    src = tmp_path / "t.cpp"
    src.write_text(MAIN)
    exe = str(tmp_path / "t")
    subprocess.run(["g++", "-O2", "-I", os.path.join(ROOT, "mms-gpu_amd", "csrc"), "-o", exe, str(src)], check=True)
    r = subprocess.run([exe], input=_values().tobytes(), capture_output=True)
    assert r.returncode == 0, r.stdout.decode()


# one line, a block and its remainder, more blocks than the buffer holds (one dump in several pieces)
@pytest.mark.gpu
@pytest.mark.parametrize("dims", [(1, 1, 1), (16, 16, 1), (19, 7, 5), (400, 70, 3)])
def test_dump_of_a_marched_film(mg, tmp_path, dims):
    """One accepted step: Mdynamics.dat holds the final state, z, x, y order,
    in the C library's %g."""
    xd, yd, zd = dims
    n = xd * yd * zd
    rng = np.random.default_rng(n)
    mat = (rng.random(n) < 0.7).astype(np.uint8)
    mat[0] = 1
    M = rng.standard_normal((n, 3)) * np.array([1, 1e-3, 1e-12])
    M = (M / np.linalg.norm(M, axis=1, keepdims=True) * 8.6e5 * mat[:, None]).astype(F).ravel()
    d = (F(5e-9),) * 3
    assert mg.time_marching(mat, M, F(0), F(1e-16), *dims, *d, 3, F(1.2566371e-6), F(8.6e5), F(1.3e-11), F(0.5),
                            F(2.211e5), 1, 1, 1, 0, sim_name=str(tmp_path / "s")) == 0, mg.last_error()
    m = M.reshape(zd, yd, xd, 3).transpose(0, 2, 1, 3).reshape(-1, 3)
    want = "".join("%g %g %g \n" % tuple(float(c) for c in v) for v in m)
    assert (tmp_path / "s" / "Mdynamics.dat").read_text() == want
