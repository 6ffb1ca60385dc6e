"""The one-workgroup walk's rule on either side of its line for 2 and 8
categories, from half a block a CU on: the same values as the walk of whole
trees and the oracle."""
import numpy as np
import pytest

from phylommand_amd import synth
from helpers import gpu_context, oracle_problem

pytestmark = pytest.mark.gpu


# 8 categories: 85 taxa in one workgroup, 120 and 250 in two launches at 8200
# sites; 250 taxa in one workgroup again at 10,000
@pytest.mark.parametrize("n,m,C,prec", [(85, 8200, 8, 0), (120, 8200, 8, 0), (250, 8200, 8, 0), (250, 10_000, 8, 0),
                                        (180, 8200, 8, 1), (250, 8200, 2, 1)])
def test_either_side_of_the_rule(oracle, n, m, C, prec):
    """FP32: a site's stored partials round to 2^-24 (1e-5 a site, as in the
    other walks' tests); FP64 differs in no bit from the whole-tree walk."""
    print(f"pieces n={n} m={m} C={C} prec={prec}", flush=True)
    wl = synth.gtr_gamma_workload(n_tips=n, m=500, C=C, alpha=0.7, gap_frac=0.05, seed=n + C)
    _, ref = oracle_problem(oracle, wl).loglik()
    ref = np.tile(ref, m // 500 + 1)[:m]
    wl.masks = np.ascontiguousarray(np.tile(wl.masks, (1, m // 500 + 1))[:, :m])
    with gpu_context(wl, precision=prec) as ctx:
        total, site = ctx.loglik(per_site=True)
        ctx.set_tail_split(False)
        plain_total, plain = ctx.loglik(per_site=True)
    if prec == 1:
        assert total == plain_total and np.array_equal(site, plain)
    assert np.abs(site / ref - 1).max() <= (1e-9 if prec == 1 else 1e-5)
    assert abs(total - ref.sum()) <= 1e-9 * abs(ref.sum()) + (0 if prec == 1 else 1e-3)
