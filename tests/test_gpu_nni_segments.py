"""NNI neighbourhoods on either side of the line between walks of one edge and
of several (nni_segment_edges: 16 waves a CU, 8 of wide states), alone and as a
batch of one, against the oracle."""
import numpy as np
import pytest

import phylommand_amd as P
from phylommand_amd import synth
from helpers import gpu_context
from test_gpu_nni_walks import _check

pytestmark = pytest.mark.gpu


# site blocks x inner edges x categories a CU (256 CUs): 14.8, 18.4; 3.3, 29.5; 8.3, 16.5
@pytest.mark.parametrize("n,m,S,C,prec", [(60, 1000, 4, 4, 0), (60, 1200, 4, 4, 0), (14, 250, 20, 4, 0), (60, 300, 20, 4, 1),
                                          (530, 256, 4, 1, 1), (530, 500, 4, 1, 1)])
def test_either_side_of_the_line(oracle, n, m, S, C, prec):
    print(f"nni segments n={n} m={m} S={S} C={C} prec={prec}", flush=True)
    kw = dict(rate_dist="gamma", freq_conc=2.0) if S > 4 else {}
    wl = synth.gtr_gamma_workload(n_tips=n, m=m, C=C, S=S, alpha=0.7, gap_frac=0.05, seed=n + m, **kw)
    with gpu_context(wl, precision=prec) as ctx:
        _check(oracle, wl, ctx, 1)
        single = ctx.nni_score(1)[1]
    if S == 4:
        t = wl.tree
        with P.Batch(C, prec) as b:
            b.add(wl.masks, t.left, t.right, t.root, t.blen, wl.Q, wl.pi, wl.cat_rates, wl.cat_weights, nni_mode=1)
            b.finalize(autotune=False)
            nni = b.run()[1]
        # (FP32: a context's evaluation may store other partials than a batch's)
        np.testing.assert_allclose(nni, [x[2] for x in single], rtol=1e-8 if prec == 0 else 1e-11)
