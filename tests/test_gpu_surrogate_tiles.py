"""The surrogate's convolutions walk the 16 x 16 tiles of all layers: fewer
tiles than workgroups, one tile more, workgroups whose tiles lie in several layers."""
import os
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F = np.float32
sys.path.insert(0, os.path.dirname(__file__))


# tiles: 5, 257 (one strip), 300 in 5 layers, 816 in 3
@pytest.mark.parametrize("dims", [(16, 16, 5), (16, 4100, 1), (160, 90, 5), (272, 250, 3)])
def test_conv_tiles_of_all_layers(mg, dims):
    import surrogate_ref
    from mms_gpu import workloads as wl
    n = int(np.prod(dims))
    rng = np.random.default_rng(n)
    rho = (rng.standard_normal(n) * 1e14).astype(F)
    w = (rng.standard_normal(int(mg.lib().mms_surrogate_weight_count())) * 0.08).astype(F)
    mat = np.ones(n, np.uint8)
    with mg.Film(*dims, *(F(5e-9),) * 3, Ms=wl.MS) as f:
        f.surrogate_init(w, charge_scale=1e14, potential_scale=2.0)
        got = f.surrogate_potential(rho)
    ref = surrogate_ref.forward(w, rho, mat, dims, 1e-14, 2.0)
    # BF16 activations: the tolerance of the forward pass
    assert np.linalg.norm(got - ref) / np.linalg.norm(ref) < 2e-2
    per = np.abs(got - ref).reshape(dims[2], -1).max(axis=1) / np.abs(ref).max()
    assert per.max() < 0.2  # no tile of any layer is another's or missing
