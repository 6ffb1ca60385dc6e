"""Training sets past 2^31 elements: a minibatch's rows may lie further apart
than 32 bits of elements reach."""
import numpy as np
import pytest

import phylommand_amd as P

pytestmark = pytest.mark.gpu


def test_rows_two_to_the_31_elements_apart():
    """10,240 samples of 2^18 features (10.7 GB), all zero but one column: the
    training is that of one feature, to the bit (adding zero products changes no
    sum, and a zero gradient leaves its weight)."""
    n, n_in, col, B = 10_240, 1 << 18, 200_003, 640
    print(f"mlp {n} x {n_in}", flush=True)
    rng = np.random.default_rng(4)
    x1 = rng.normal(0, 1, (n, 1)).astype(np.float32)
    t = (np.sin(3 * x1) + 0.1 * rng.normal(0, 1, (n, 1))).astype(np.float32)
    small, big = P.MLP(1, 2, 1, max_batch=B, seed=2), P.MLP(n_in, 2, 1, max_batch=B, seed=2)
    w = small.params()
    wide = np.zeros(big.n_params, np.float32)
    at = np.concatenate([2 * col + np.arange(2), 2 * n_in + np.arange(len(w) - 2)])     # [W1 | b1 W2 b2 W3 b3]
    wide[at] = w
    big.set_params(wide)
    want = small.train(x1, t, epochs=2, batch=B, lr=1e-2, seed=5)
    x = np.zeros((n, n_in), np.float32)
    x[:, col] = x1[:, 0]
    got = big.train(x, t, epochs=2, batch=B, lr=1e-2, seed=5)
    wide = big.params()
    small_w = small.params()
    small.close()
    big.close()
    assert np.array_equal(got, want) and not np.array_equal(small_w, w)
    assert np.array_equal(wide[at], small_w) and np.count_nonzero(wide) == np.count_nonzero(small_w)
