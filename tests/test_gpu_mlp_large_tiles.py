"""The MLP's 64 x 64 tiles (products of at least a tile a CU) at ragged sizes,
and beside 16 x 32 tiles in one network: forward, gradient and a training step
against FP64 backpropagation."""
import numpy as np
import pytest

import phylommand_amd as P

from oracle import learn_oracle as LO

pytestmark = pytest.mark.gpu

# a sum of K random terms at FP32 is off by about 0.4 sqrt(K) 2^-24 of its own
# spread, 1.1e-6 at K = 2100, in each of three layers and back
TOL = 2e-5


@pytest.mark.parametrize("n_in,n_hid,n_out,B", [(70, 1030, 5, 1025),      # every product in large tiles
                                                (33, 2100, 3, 513),
                                                (5, 700, 2, 3000)])       # the layers large, the gradients small
def test_large_products(n_in, n_hid, n_out, B):
    print(f"mlp {n_in}-{n_hid}-{n_hid}-{n_out} batch {B}", flush=True)
    rng = np.random.default_rng(n_hid)
    x = rng.normal(0, 1, (B, n_in)).astype(np.float32)
    t = rng.normal(0, 1, (B, n_out)).astype(np.float32)
    net = P.MLP(n_in, n_hid, n_out, max_batch=B, seed=3)
    w = net.params()
    ref, _ = LO.mlp_forward(w, x, n_in, n_hid, n_out)
    assert np.linalg.norm(net.forward(x) - ref) <= TOL * np.linalg.norm(ref)
    loss, g = net.grad(x, t)
    ref_loss, ref_g = LO.mlp_grad(w, x, t, n_in, n_hid, n_out)
    assert loss == pytest.approx(ref_loss, rel=TOL)
    assert np.linalg.norm(g - ref_g) <= TOL * np.linalg.norm(ref_g)
    # one step: Adam moves each weight by lr against its gradient's sign
    assert net.train(x, t, epochs=1, batch=B, lr=1e-2)[0] == pytest.approx(ref_loss, rel=TOL)
    want, _, _ = LO.adam_step(w.astype(np.float64), ref_g, np.zeros_like(ref_g), np.zeros_like(ref_g), step=1, lr=1e-2)
    big = np.abs(ref_g) > 1e-5
    np.testing.assert_allclose(net.params()[big], want[big], atol=1e-4)
    net.close()
