"""The one-workgroup walk of a whole tree in pieces (few site blocks): the
same bits as the two launches that store through memory, and as the plain walk
in FP64, at the edges of its range: the smallest trees it takes, site counts
around a block and around a block a CU, taxa past what LDS stages, trees whose
results do not fit, one to eight categories, weights."""
import numpy as np
import pytest

import phylommand_amd as P
from phylommand_amd import synth
from helpers import gpu_context, oracle_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m,C,prec", [
    (16, 64, 4, 0), (17, 1, 4, 0), (17, 63, 1, 1), (18, 65, 2, 0), (40, 700, 8, 0), (40, 700, 8, 1),
    (33, 16128, 4, 0), (33, 16385, 4, 0), (64, 9000, 1, 1), (128, 9000, 4, 1), (250, 9000, 4, 0), (256, 300, 1, 0),
    (257, 300, 1, 0), (90, 16384, 2, 1),
])
def test_pieces_match_the_other_walks(oracle, n, m, C, prec):
    print(f"pieces n={n} m={m} C={C} prec={prec}", flush=True)
    wl = synth.gtr_gamma_workload(n_tips=n, m=min(m, 500), C=C, alpha=0.7, gap_frac=0.05, seed=n + C)
    wl.masks = np.ascontiguousarray(np.tile(wl.masks, (1, m // 500 + 1))[:, :m])
    w = np.random.default_rng(n).integers(1, 4, m).astype(float)
    got = {}
    for keep in (False, True):
        with gpu_context(wl, precision=prec) as ctx:
            ctx.set_keep_partials(keep)          # every partial stored: two launches
            first = ctx.loglik(per_site=True)
            again = ctx.loglik()
            ctx.set_site_weights(w)
            got[keep] = (*first, again, ctx.loglik())
    assert got[False][0] == got[False][2] == got[True][0]
    assert got[False][3] == got[True][3]
    assert np.array_equal(got[False][1], got[True][1])
    tot, site, _, weighted = got[False]
    if prec == 1:
        with gpu_context(wl, precision=prec) as ctx:
            ctx.set_tail_split(False)
            plain = ctx.loglik(per_site=True)
        assert tot == plain[0] and np.array_equal(site, plain[1])
    k = min(m, 500)                              # the sites repeat after 500
    wl.masks = np.ascontiguousarray(wl.masks[:, :k])
    _, ref = oracle_problem(oracle, wl).loglik()
    ref = np.tile(ref, m // k + 1)[:m]
    rel = np.abs(site - ref) / np.maximum(np.abs(ref), 1.0)
    assert rel.max() <= (1e-9 if prec == 1 else 1e-5)
    assert abs(weighted - float(np.dot(w, site))) <= 1e-9 * abs(weighted)


def test_precision_and_categories_changed_on_one_topology():
    """Programs follow the category count; FP64 slots may not fit where FP32's did."""
    print("pieces: precision and categories changed", flush=True)
    wls = {C: synth.gtr_gamma_workload(n_tips=128, m=9000, C=C, alpha=0.7, gap_frac=0.05, seed=3) for C in (1, 4, 8)}
    wl = wls[4]
    with gpu_context(wl) as ctx:
        for prec, C in [(0, 4), (1, 4), (1, 8), (0, 1), (0, 4), (1, 1)]:
            ctx.set_precision(prec)
            ctx.set_categories(wls[C].cat_rates, wls[C].cat_weights)
            tot = ctx.loglik()
            with gpu_context(wl, precision=1) as ref:
                ref.set_categories(wls[C].cat_rates, wls[C].cat_weights)
                ref.set_tail_split(False)
                want = ref.loglik()
            assert abs(tot - want) <= (1e-3 if prec == 0 else 1e-9 * abs(want)), (prec, C, tot, want)
