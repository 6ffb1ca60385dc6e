"""Inputs read from host memory and kernel arguments: lengths, models and
weights changed between evaluations in any order give the values a fresh
context gives, bit for bit, and programs and site values follow a new topology
or more sites."""
import numpy as np
import pytest

import phylommand_amd as P
from phylommand_amd import synth
from helpers import gpu_context, oracle_problem

pytestmark = pytest.mark.gpu


def _wl(n, m, S, C, seed):
    kw = dict(rate_dist="gamma", freq_conc=2.0) if S > 4 else {}
    return synth.gtr_gamma_workload(n_tips=n, m=m, C=C, S=S, alpha=0.7, gap_frac=0.05, seed=seed, **kw)


def _fresh(wl, prec, builder):
    with gpu_context(wl, precision=prec, builder=builder) as ctx:
        return ctx.loglik(per_site=True)


@pytest.mark.parametrize("S,C,prec,builder", [
    (2, 1, 0, P.P_EIGEN), (3, 2, 1, P.P_EIGEN), (4, 4, 0, P.P_EIGEN), (4, 8, 1, P.P_EIGEN), (4, 4, 1, P.P_PADE),
    (5, 8, 1, P.P_EIGEN), (20, 4, 0, P.P_EIGEN), (32, 1, 1, P.P_EIGEN), (20, 2, 0, P.P_PADE),
])
def test_changed_inputs_match_a_fresh_context(S, C, prec, builder):
    _changed_inputs(9, S, C, prec, builder)


@pytest.mark.parametrize("n", [192, 193])
def test_lengths_at_the_limit_of_the_arguments(n):
    """383 nodes' lengths are kernel arguments, 385 nodes' are in pinned memory."""
    _changed_inputs(n, 4, 2, 1, P.P_EIGEN)


def _changed_inputs(n, S, C, prec, builder):
    print(f"inputs n={n} S={S} C={C} prec={prec} builder={builder}", flush=True)
    a, b = _wl(n, 130, S, C, 50 + S), _wl(n, 130, S, C, 70 + S)
    b.tree, b.masks = a.tree, a.masks
    want = [_fresh(x, prec, builder) for x in (a, b)]
    n = a.tree.n_nodes
    with gpu_context(a, precision=prec, builder=builder) as ctx:
        for k in (0, 1, 0, 1, 1):
            x = (a, b)[k]
            ctx.set_edge_lengths(np.full(n, 0.3))
            if builder == P.P_EIGEN:
                ctx.simulate(40, x.pi, 1)                   # other lengths' P, not waited for by the host below
            ctx.set_edge_lengths(x.tree.blen)
            ctx.set_model(x.Q, x.pi, x.pi, builder)
            ctx.set_categories(x.cat_rates, x.cat_weights)
            tot, site = ctx.loglik(per_site=True)
            assert tot == want[k][0] and np.array_equal(site, want[k][1])
        # weights alone, by tips set again
        ctx.set_tips(a.masks, S)
        tot, site = ctx.loglik(per_site=True)
        assert tot == want[1][0] and np.array_equal(site, want[1][1])


def test_programs_and_site_values_follow_larger_problems(oracle):
    """One context, each problem larger than the one before, then the first again."""
    wls = [_wl(n, m, 4, 2, n) for n, m in [(4, 1), (9, 64), (70, 999), (300, 4097)]]
    first = None
    with P.Context(0, P.PREC_FP64) as ctx:
        for wl in wls + wls[:1]:
            t = wl.tree
            print(f"inputs taxa={t.n_tips} sites={wl.masks.shape[1]}", flush=True)
            ctx.set_tips(wl.masks, 4)
            ctx.set_topology(t.left, t.right, t.root)
            ctx.set_edge_lengths(t.blen)
            ctx.set_model(wl.Q, wl.pi, wl.pi, P.P_EIGEN)
            ctx.set_categories(wl.cat_rates, wl.cat_weights)
            tot, site = ctx.loglik(per_site=True)
            ref_tot, ref_site = oracle_problem(oracle, wl).loglik()
            assert abs(tot - ref_tot) <= 1e-9 * max(1.0, abs(ref_tot))
            assert np.max(np.abs(site - ref_site) / np.maximum(np.abs(ref_site), 1.0)) <= 1e-9
            first = first or tot
    assert tot == first
