"""The MLP's tile kernels at the edges of their tiles (16 rows, 32 columns,
64-long pieces of a sum): forward, gradient and Adam against FP64
backpropagation, and batches in shuffled order through train()."""
import numpy as np
import pytest

import phylommand_amd as P

from oracle import learn_oracle as LO

pytestmark = pytest.mark.gpu

# the sums run over at most 130 terms of one sign pattern at FP32: a relative
# error of n 2^-24 < 8e-6 of the sum of magnitudes
TOL = 1e-5


@pytest.mark.parametrize("n_in,n_hid,n_out,B", [(1, 1, 1, 1), (5, 17, 3, 2), (64, 32, 12, 16), (65, 33, 13, 17),
                                                (63, 64, 32, 64), (128, 130, 33, 65), (130, 31, 40, 130)])
def test_mlp_sizes_around_the_tiles(n_in, n_hid, n_out, B):
    print(f"mlp {n_in}-{n_hid}-{n_hid}-{n_out} batch {B}", flush=True)
    rng = np.random.default_rng(n_in + n_hid + B)
    x = rng.normal(0, 1, (B, n_in)).astype(np.float32)
    t = rng.normal(0, 1, (B, n_out)).astype(np.float32)
    net = P.MLP(n_in, n_hid, n_out, max_batch=B, seed=3)
    w = net.params()
    y = net.forward(x)
    ref, _ = LO.mlp_forward(w, x, n_in, n_hid, n_out)
    assert np.linalg.norm(y - ref) <= TOL * max(np.linalg.norm(ref), 1e-3)
    loss, g = net.grad(x, t)
    ref_loss, ref_g = LO.mlp_grad(w, x, t, n_in, n_hid, n_out)
    assert loss == pytest.approx(ref_loss, rel=TOL)
    assert np.linalg.norm(g - ref_g) <= TOL * max(np.linalg.norm(ref_g), 1e-6)
    net.close()


def test_training_steps_follow_the_gradients():
    """Two full-batch epochs: the second step sees the first one's weights (and
    the transposed copy that goes back through them)."""
    rng = np.random.default_rng(5)
    x = rng.normal(0, 1, (48, 20)).astype(np.float32)
    t = rng.normal(0, 1, (48, 7)).astype(np.float32)
    net = P.MLP(20, 40, 7, max_batch=48, seed=9)
    w = net.params().astype(np.float64)
    losses = net.train(x, t, epochs=2, batch=48, lr=1e-2)
    m, v = np.zeros_like(w), np.zeros_like(w)
    want = []
    for step in (1, 2):
        loss, g = LO.mlp_grad(w, x, t, 20, 40, 7)
        want.append(loss)
        w, m, v = LO.adam_step(w, g, m, v, step=step, lr=1e-2)
    np.testing.assert_allclose(losses, want, rtol=1e-4)
    big = np.abs(g) > 1e-5
    np.testing.assert_allclose(net.params()[big], w[big], atol=1e-4)
    net.close()
