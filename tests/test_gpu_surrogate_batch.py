"""The trainer's batch: more pairs than one gather launch takes, pairs out of
order and repeated, and the mode mixing's groups of layers with a remainder."""
import os
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F = np.float32
sys.path.insert(0, os.path.dirname(__file__))


# 5 layers (a group of four and one); 66 pairs (64 and two), a cell count that is no multiple of a block
@pytest.mark.parametrize("dims,batch", [((17, 16, 5), 1), ((18, 13, 1), 66)])
def test_batch_order_and_loss(mg, dims, batch):
    import surrogate_ref
    from mms_gpu import workloads as wl
    rng = np.random.default_rng(batch)
    w = (rng.standard_normal(int(mg.lib().mms_surrogate_weight_count())) * 0.08).astype(F)
    idx = rng.integers(0, 3, batch)
    dx, Ms = F(5e-9), F(wl.MS)
    with mg.SurrogateTrainer(*dims, dx, Ms, batch, weights=w) as t:
        t.generate(3, 2010, P=0)
        g, loss = t.gradient(idx)
        one = np.asarray(t.eval(idx))
        pairs = [t.pair(int(i)) for i in idx]
    rho, phi = (np.concatenate([p[k] for p in pairs]) for k in (0, 1))
    lref, gref = surrogate_ref.loss_and_grad(w, rho, phi, dims, batch, float(dx / Ms), float(Ms * dx))
    # BF16 activations and gradients: the tolerances of the gradient against autograd
    assert abs(loss - lref) <= 1e-3 * abs(lref)
    assert np.linalg.norm(g - gref) / np.linalg.norm(gref) < 1e-2
    for k in set(idx.tolist()):  # a pair's residual is the same wherever it stands in the batch
        assert np.ptp(one[idx == k]) == 0
