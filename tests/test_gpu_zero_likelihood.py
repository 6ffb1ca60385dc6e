"""Sites of likelihood zero: a model in which one state exchanges with no other,
and a site with that state at one tip and another state at the next.  Its
log-likelihood is minus infinity under every tree, and so are all totals that
hold it, whichever sum they pass through, and no others."""
import numpy as np
import pytest

import phylommand_amd as P
from phylommand_amd import synth
from helpers import gpu_context

pytestmark = pytest.mark.gpu


def _workload(n, m, S, C, bad, seed):
    kw = dict(rate_dist="gamma", freq_conc=2.0) if S > 4 else {}
    wl = synth.gtr_gamma_workload(n_tips=n, m=m, S=S, C=C, alpha=0.7, gap_frac=0.05, seed=seed, **kw)
    Q = np.array(wl.Q).reshape(S, S)
    Q[S - 1, :] = Q[:, S - 1] = 0.0
    np.fill_diagonal(Q, 0.0)
    np.fill_diagonal(Q, -Q.sum(1))
    masks = np.array(wl.masks)
    masks[masks == 1 << (S - 1)] = 1
    if bad is not None:
        masks[0, bad], masks[1, bad] = 1, 1 << (S - 1)
    wl.Q, wl.masks = Q, masks
    return wl


@pytest.mark.parametrize("n,m,S,C,prec,bad", [
    (8, 1, 4, 1, 0, 0), (8, 130, 4, 4, 1, 64), (24, 3000, 4, 4, 0, 0), (24, 3000, 4, 1, 1, 2999), (24, 40000, 4, 4, 0, 20000),
    (300, 500, 4, 2, 0, 499), (8, 33, 20, 1, 0, 32), (24, 2000, 20, 4, 1, 0),
])
def test_totals_are_minus_infinity(n, m, S, C, prec, bad):
    print(f"zero likelihood n={n} m={m} S={S} C={C} prec={prec} site {bad}", flush=True)
    wl = _workload(n, m, S, C, bad, 60 + n)
    w = np.ones(m)
    with gpu_context(wl, precision=prec) as ctx:
        for weights in (None, w):
            ctx.set_site_weights(weights)
            total, site = ctx.loglik(per_site=True)
            assert site[bad] == -np.inf and np.isfinite(np.delete(site, bad)).all()
            assert total == -np.inf and ctx.loglik() == -np.inf
            base, variants = ctx.nni_score(1)
            assert base == -np.inf and [x for _, _, x in variants] == [-np.inf] * len(variants)


@pytest.mark.parametrize("prec", [P.PREC_FP32, P.PREC_FP64])
@pytest.mark.parametrize("tiling", [(64, 4), (256, 1)])
def test_batch_totals_are_minus_infinity(prec, tiling):
    """One work item and many, the site in the first, a middle and the last of
    them; the alignments beside them keep their values."""
    sizes = [(8, 60, 3), (12, 3000, 0), (12, 3000, 1500), (12, 3000, 2999), (12, 3000, None), (9, 200, None)]
    wls = [_workload(n, m, 4, 4, bad, 70 + m) for n, m, bad in sizes]
    print(f"zero likelihood batch prec={prec} tiling={tiling}", flush=True)
    with P.Batch(4, prec) as b:
        for wl in wls:
            t = wl.tree
            b.add(wl.masks, t.left, t.right, t.root, t.blen, wl.Q, wl.pi, wl.cat_rates, wl.cat_weights, nni_mode=1)
        b.set_tiling(*tiling)
        b.finalize(autotune=False)
        tot, nni = b.run()
        off, _, _ = b.nni_layout()
    for i, (_, _, bad) in enumerate(sizes):
        got = np.append(nni[off[i]:off[i + 1]], tot[i])
        assert len(got) > 1
        if bad is not None:
            assert (got == -np.inf).all()
        else:
            with gpu_context(wls[i], precision=prec) as ctx:
                base, variants = ctx.nni_score(1)
            np.testing.assert_allclose(got, [x for _, _, x in variants] + [base], rtol=1e-8)
