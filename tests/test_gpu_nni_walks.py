"""NNI neighbourhoods by the outer-partial walks where their layouts can go
wrong: state counts around the operand slots and tiles, one category and many,
site counts around a wave, taxa past what a workgroup stages,
unary nodes, FP64, site weights, every mode, and lengths changed in between."""
import numpy as np
import pytest

import phylommand_amd as P
from phylommand_amd import synth
from helpers import gpu_context
from test_gpu_edge import _tree, _workload

pytestmark = pytest.mark.gpu


def _check(oracle, wl, ctx, mode, eff=None, w=None, n_check=6, seed=0):
    """Base and a sample of variants (always the first and the last two)
    against the oracle.  FP32 tips and partials round to 2^-24 relative a
    product; the site value's error stays within 1e-5, and the totals of
    these few thousand sites within 1e-3, as in the plain evaluations."""
    t = wl.tree
    m, S = wl.masks.shape[1], len(wl.pi)
    mb = np.zeros((t.n_nodes, m), np.uint32)
    mb[: t.n_tips] = wl.masks
    eff = t.blen if eff is None else eff
    w = np.ones(m) if w is None else w

    def ref(l, r):
        _, site = oracle.Problem(l, r, t.root, eff, mb, S, wl.Q, wl.pi, pi=wl.pi, cat_rates=wl.cat_rates,
                                 cat_w=wl.cat_weights).loglik()
        return float(np.dot(w, site))

    base, variants = ctx.nni_score(mode)
    assert [(v, s) for v, s, _ in variants] == oracle.nni_list(t.left, t.right, t.root, mode)
    want = ref(t.left, t.right)
    assert abs(base - want) <= 1e-3 + 1e-9 * abs(want)
    pick = np.random.default_rng(seed).permutation(len(variants))[:n_check].tolist() + [0, len(variants) - 2, len(variants) - 1]
    for k in sorted(set(pick)):
        v, side, lnl = variants[k]
        want = ref(*oracle.nni_apply(t.left, t.right, t.root, v, side))
        assert abs(lnl - want) <= 1e-3 + 1e-9 * abs(want), (v, side, lnl, want)


@pytest.mark.parametrize("n,m,S,C,prec,mode", [
    (9, 65, 4, 1, 0, 1), (11, 64, 4, 8, 1, 0), (13, 1, 4, 2, 0, 1), (7, 257, 2, 4, 1, 1), (300, 130, 4, 4, 0, 1),
    (6, 17, 5, 1, 0, 1), (8, 16, 8, 2, 1, 0), (8, 15, 9, 4, 0, 1), (9, 33, 16, 4, 1, 1), (9, 63, 17, 1, 0, 0),
    (9, 1, 19, 8, 1, 1), (10, 48, 21, 2, 0, 1), (8, 49, 24, 4, 1, 1), (8, 31, 25, 1, 0, 1), (8, 80, 32, 4, 0, 1),
    (140, 20, 20, 4, 1, 1), (530, 70, 4, 1, 1, 1),      # (more than 1024 variants)
])
def test_walks_match_the_oracle_at_layout_edges(oracle, n, m, S, C, prec, mode):
    print(f"nni walks n={n} m={m} S={S} C={C} prec={prec} mode={mode}", flush=True)
    kw = dict(rate_dist="gamma", freq_conc=2.0) if S > 4 else {}
    wl = synth.gtr_gamma_workload(n_tips=n, m=m, C=C, S=S, alpha=0.7, gap_frac=0.05, seed=40 + n + S, **kw)
    rng = np.random.default_rng(m + S)
    w = rng.integers(1, 5, m).astype(float)
    eff = wl.tree.blen * rng.uniform(0.5, 2.0, wl.tree.n_nodes)
    with gpu_context(wl, precision=prec) as ctx:
        _check(oracle, wl, ctx, mode)
        ctx.set_edge_lengths(eff)          # rebuilds every form of P
        ctx.set_site_weights(w)
        _check(oracle, wl, ctx, mode, eff=eff, w=w, n_check=2)


@pytest.mark.parametrize("S", [5, 16, 20, 23, 32])
def test_both_builders_give_the_same_scores(S):
    """P built on the host passes through the same layouts: the two builders'
    entries agree to 1e-10 or better, and so do FP64 scores."""
    print(f"nni builders S={S}", flush=True)
    wl = synth.gtr_gamma_workload(n_tips=10, m=70, C=2, S=S, alpha=0.7, gap_frac=0.05, seed=S, rate_dist="gamma",
                                  freq_conc=2.0)
    got = []
    for builder in (1, 2):
        with gpu_context(wl, precision=1, builder=builder) as ctx:
            base, variants = ctx.nni_score(1)
            got.append([base] + [x[2] for x in variants])
    np.testing.assert_allclose(got[0], got[1], rtol=1e-9)


@pytest.mark.parametrize("S,prec", [(4, 0), (4, 1), (20, 0), (20, 1)])
def test_unary_nodes_pass_their_child(oracle, S, prec):
    """A unary internal node on a path, inside the neighbourhood: exchanging
    its missing child keeps the tree, alone and in a batch."""
    print(f"nni unary S={S} prec={prec}", flush=True)
    # tips 0..4; 5 = (0,1); 6 = unary above 5; 7 = (2,3); 8 = (6,7); 9 = root (8,4)
    t = _tree([-1] * 5 + [0, 5, 2, 6, 8], [-1] * 5 + [1, -1, 3, 7, 4], 9,
              [0.1, 0.2, 0.15, 0.25, 0.05, 0.3, 0.12, 0.2, 0.1, 0.0], 5)
    wl = _workload(t, 130, C=2, S=S, seed=6)
    with gpu_context(wl, precision=prec) as ctx:
        _check(oracle, wl, ctx, 1)
        single = ctx.nni_score(1)[1]
    if S == 4:
        with P.Batch(2, prec) as b:
            b.add(wl.masks, t.left, t.right, t.root, t.blen, wl.Q, wl.pi, wl.cat_rates, wl.cat_weights, nni_mode=1)
            b.finalize(autotune=False)
            nni = b.run()[1]
        np.testing.assert_allclose(nni, [x[2] for x in single], rtol=1e-9)
