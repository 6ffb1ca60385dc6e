"""The work that users of phylommand_amd have it do, as cases that a timing
program runs: likelihood evaluations of DNA and protein alignments (the step
of a model fit, of a branch-length optimiser, of a program that scores tree
after tree), NNI neighbourhoods, batches of alignments, and the learned
proposal's simulator and training.

Every case goes through the package's public entry points with host arrays,
as a user's program calls them.  Alignments are simulated down a Yule tree
under the case's model (discrete gamma rates, a fraction of the cells gaps),
so site patterns repeat as often as they do in such data.

listed() gives the fixed cases, draw() more of the same ranges, prepare() a
state, run() one pass on it, work() the bytes and operations a pass cannot do
without, exact() the same outputs in 64 bits by plain torch.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

DEV = "cuda"


# ---- the cases -------------------------------------------------------------

def listed():
    return [
        # One evaluation of the GTR+G4 model fit: new rates, frequencies, shape
        # and scale on a 32-taxon alignment with FP64 partials (the learned
        # proposal's held-out fits take about 1,000 of these each).
        dict(name="fit_eval_32x2000", kind="fit", taxa=32, sites=2000, cats=4, mean_blen=0.1, alpha=0.8, gap=0.04),
        # treeator's per-site output: one rate category, FP64 partials, an odd
        # number of sites.
        dict(name="persite_f64_50x4099", kind="dna_site", taxa=50, sites=4099, cats=1, mean_blen=0.1, alpha=1.0,
             gap=0.05),
        # Scoring tree after tree on one alignment (a tree file given to
        # treeator): a new topology and its lengths before every evaluation.
        dict(name="new_tree_50x10000", kind="tree", taxa=50, sites=10_000, cats=4, mean_blen=0.08, alpha=0.6,
             gap=0.05),
        # The benchmark's DNA workload as an optimiser runs it: new edge
        # lengths, then the evaluation.
        dict(name="dna_128x100000", kind="dna", taxa=128, sites=100_000, cats=4, mean_blen=0.05, alpha=0.5, gap=0.05),
        # A large alignment: more taxa, sites and longer branches.
        dict(name="dna_250x250000", kind="dna", taxa=250, sites=250_000, cats=4, mean_blen=0.1, alpha=0.8, gap=0.03),
        # Small protein alignment, per-site values with FP64 partials.
        dict(name="protein_site_24x1999", kind="protein_site", taxa=24, sites=1999, cats=4, mean_blen=0.1, alpha=1.0,
             gap=0.05),
        # The 20-state workload of the benchmark, new lengths each time.
        dict(name="protein_64x20000", kind="protein", taxa=64, sites=20_000, cats=4, mean_blen=0.05, alpha=1.0,
             gap=0.03),
        # Every NNI neighbour of the DNA benchmark tree after its lengths
        # changed (one step of a hill-climbing tree search).
        dict(name="nni_dna_128x100000", kind="nni_dna", taxa=128, sites=100_000, cats=4, mean_blen=0.05, alpha=0.5,
             gap=0.05),
        # The same for a protein tree of ordinary size.
        dict(name="nni_protein_40x5000", kind="nni_protein", taxa=40, sites=5000, cats=4, mean_blen=0.08, alpha=1.0,
             gap=0.03),
        # Many alignments of uneven size with their neighbourhoods (the
        # 512-alignment workload's distribution, fewer of them).
        dict(name="batch_24", kind="batch", align=24, max_taxa=256, max_sites=20_000, cats=4, mean_blen=0.05,
             gap=0.05),
        # Training data of the learned proposal: simulate and featurise.
        dict(name="features_512x32x2000", kind="features", align=512, taxa=32, sites=2000, cats=4, gap=0.04),
        # One epoch of the proposal's training.
        dict(name="mlp_epoch_4096", kind="mlp", samples=4096, hidden=512, batch=256),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["fit", "dna_site", "tree", "dna", "dna", "protein_site", "protein", "nni_dna", "nni_protein",
                       "batch", "features", "mlp"])
    common = dict(mean_blen=round(math.exp(rng.uniform(math.log(0.02), math.log(0.25))), 4),
                  gap=round(rng.uniform(0.0, 0.08), 4))
    shape = dict(alpha=round(math.exp(rng.uniform(math.log(0.3), math.log(2.0))), 3), **common)
    if kind == "fit":
        return dict(kind=kind, taxa=rng.randint(8, 64), sites=_log_int(rng, 500, 5000), cats=4, **shape)
    if kind == "dna_site":
        return dict(kind=kind, taxa=rng.randint(9, 120), sites=_log_int(rng, 500, 20_000), cats=rng.choice([1, 2, 4]),
                    **shape)
    if kind == "tree":
        return dict(kind=kind, taxa=rng.randint(16, 128), sites=_log_int(rng, 1000, 50_000), cats=rng.choice([1, 4]),
                    **shape)
    if kind == "dna":
        return dict(kind=kind, taxa=rng.randint(16, 250), sites=_log_int(rng, 2000, 200_000),
                    cats=rng.choice([1, 4, 4, 8]), **shape)
    if kind == "protein_site":
        return dict(kind=kind, taxa=rng.randint(8, 48), sites=_log_int(rng, 300, 4000), cats=rng.choice([1, 4]),
                    **shape)
    if kind == "protein":
        return dict(kind=kind, taxa=rng.randint(16, 100), sites=_log_int(rng, 1000, 30_000), cats=rng.choice([1, 4]),
                    **shape)
    if kind == "nni_dna":
        return dict(kind=kind, taxa=rng.randint(12, 128), sites=_log_int(rng, 1000, 100_000), cats=rng.choice([1, 4]),
                    **shape)
    if kind == "nni_protein":
        return dict(kind=kind, taxa=rng.randint(10, 48), sites=_log_int(rng, 500, 8000), cats=rng.choice([1, 4]),
                    **shape)
    if kind == "batch":
        return dict(kind=kind, align=rng.randint(6, 24), max_taxa=rng.randint(32, 256),
                    max_sites=_log_int(rng, 2000, 20_000), cats=4, **common)
    if kind == "features":
        return dict(kind=kind, align=_log_int(rng, 64, 1024), taxa=rng.randint(8, 32), sites=_log_int(rng, 300, 2500),
                    cats=4, gap=common["gap"])
    return dict(kind="mlp", samples=_log_int(rng, 1024, 8192), hidden=rng.choice([128, 256, 512]),
                batch=rng.choice([128, 200, 256]))


# ---- inputs ----------------------------------------------------------------

def _states(case):
    return 20 if "protein" in case["kind"] else 4


def _yule(n, rng, mean_blen):
    """A random rooted binary tree: tips 0..n-1, internal nodes n..2n-2."""
    kids, leaves, nxt = {}, [0], 1
    while len(leaves) < n:
        v = leaves.pop(int(rng.integers(len(leaves))))
        kids[v] = (nxt, nxt + 1)
        leaves += [nxt, nxt + 1]
        nxt += 2
    ren, tip, inner = {}, 0, n
    for v in range(nxt):
        if v in kids:
            ren[v], inner = inner, inner + 1
        else:
            ren[v], tip = tip, tip + 1
    left = np.full(nxt, -1, np.int32)
    right = np.full(nxt, -1, np.int32)
    for v, (a, b) in kids.items():
        left[ren[v]], right[ren[v]] = ren[a], ren[b]
    blen = rng.exponential(mean_blen, nxt)
    blen[ren[0]] = 0.0
    return dict(left=left, right=right, root=int(ren[0]), blen=blen)


def _preorder(t):
    out, stack = [], [t["root"]]
    while stack:
        v = stack.pop()
        out.append(v)
        if t["left"][v] >= 0:
            stack += [int(t["right"][v]), int(t["left"][v])]
    return out


def _parents(t):
    par = np.full(len(t["left"]), -1, np.int64)
    for v in range(len(par)):
        for c in (t["left"][v], t["right"][v]):
            if c >= 0:
                par[c] = v
    return par


def _rate_matrix(rates, pi):
    S = len(pi)
    Q = np.zeros((S, S))
    Q[np.triu_indices(S, 1)] = rates
    Q = (Q + Q.T) * pi[None, :]
    np.fill_diagonal(Q, -Q.sum(axis=1))
    return Q / -np.dot(pi, np.diag(Q))


def _gamma_rates(alpha, C):
    """Mean rates of C equal-probability categories of a gamma(alpha, alpha)."""
    if C == 1:
        return np.ones(1)
    a = torch.tensor(float(alpha), dtype=torch.float64)
    q = torch.arange(1, C, dtype=torch.float64) / C
    lo, hi = torch.zeros(C - 1, dtype=torch.float64), torch.full((C - 1,), 1e4, dtype=torch.float64)
    for _ in range(200):                  # P(alpha, x) = q by bisection
        mid = 0.5 * (lo + hi)
        below = torch.special.gammainc(a.expand_as(mid), mid) < q
        lo, hi = torch.where(below, mid, lo), torch.where(below, hi, mid)
    cum = torch.special.gammainc((a + 1).expand_as(lo), 0.5 * (lo + hi)).numpy()
    return np.diff(np.concatenate([[0.0], cum, [1.0]])) * C


def _eigen(Q, pi):
    d = np.sqrt(pi)
    lam, U = np.linalg.eigh(0.5 * (d[:, None] * Q / d[None, :] + (d[:, None] * Q / d[None, :]).T))
    return U / d[:, None], lam, U.T * d[None, :]


def _transition(Q, pi, lengths, rates):
    """P[edge, category] = expm(Q length rate), FP64 on the GPU."""
    V, lam, W = _eigen(Q, pi)
    e = np.exp(np.multiply.outer(np.multiply.outer(np.asarray(lengths), np.asarray(rates)), lam))
    V, W, e = (torch.from_numpy(np.ascontiguousarray(x)).to(DEV) for x in (V, W, e))
    return torch.matmul(V * e[..., None, :], W.expand(*e.shape[:2], *W.shape).contiguous())


def _simulate(t, Q, pi, rates, m, gap, gen):
    """Tip state sets [taxa, m] (uint32 masks) of m sites simulated down t."""
    n, S = (len(t["left"]) + 1) // 2, len(pi)
    cum = _transition(Q, pi, t["blen"], rates).clamp_min(0).cumsum(-1)
    cum = cum / cum[..., -1:]
    rnd = lambda *s: torch.rand(*s, device=DEV, generator=gen, dtype=torch.float64)  # noqa: E731
    cat = torch.randint(len(rates), (m,), device=DEV, generator=gen)
    edges = torch.from_numpy(np.cumsum(pi)[:-1].copy()).to(DEV)
    st = {t["root"]: torch.bucketize(rnd(m), edges)}
    masks = torch.empty((n, m), dtype=torch.int32, device=DEV)
    par = _parents(t)
    for v in _preorder(t):
        if v != t["root"]:
            rows = cum[v].reshape(-1, S)[cat * S + st[int(par[v])]]
            st[v] = (rnd(m)[:, None] > rows[:, :-1]).sum(1)
        if v < n:
            masks[v] = torch.where(rnd(m) < gap, (1 << S) - 1, torch.bitwise_left_shift(torch.ones_like(st[v]), st[v]))
    return masks.cpu().numpy().astype(np.uint32)


def _problem(case, seed, taxa=None, sites=None, alpha=None):
    """Tree, model and alignment of one likelihood problem."""
    S, C = _states(case), case["cats"]
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device=DEV).manual_seed(int(seed))
    n, m = taxa or case["taxa"], sites or case["sites"]
    t = _yule(n, rng, case["mean_blen"])
    nr = S * (S - 1) // 2
    ex = rng.gamma(1.0, 1.0, nr) + 0.01
    pi = rng.dirichlet(np.full(S, 5.0 if S == 4 else 2.0)) * (1 - 0.001 * S) + 0.001
    Q = _rate_matrix(ex, pi)
    rates = _gamma_rates(alpha or case["alpha"], C)
    masks = _simulate(t, Q, pi, rates, m, case["gap"], gen)
    lengths = t["blen"] * rng.uniform(0.8, 1.25, len(t["blen"]))     # what the caller evaluates
    return dict(t=t, S=S, C=C, Q=Q, pi=pi, rates=rates, masks=masks, lengths=lengths, ex=ex,
                weights=np.full(C, 1.0 / C))


def _fit_point(case, seed):
    """Relative lengths (mean 1) and the fit's parameter vector: log
    exchangeabilities against the last, frequency logits against the last,
    log shape, log scale."""
    p = _problem(case, seed)
    b = p["lengths"]
    mean = b.sum() / (len(b) - 1)
    x = np.concatenate([np.log(p["ex"][:5] / p["ex"][5]), np.log(p["pi"][:3] / p["pi"][3]),
                        [math.log(case["alpha"]), math.log(mean)]])
    return p, b / mean, x


def _batch_sizes(case):
    """(taxa, sites, shape) of every alignment: part of the case, not of the
    seed; taxa uniform from 8, sites log-uniform from 500."""
    rng = random.Random(case["align"] * 1_000_003 + case["max_taxa"] * 1009 + case["max_sites"])
    return [(rng.randint(8, case["max_taxa"]), _log_int(rng, 500, case["max_sites"]), rng.uniform(0.3, 2.0))
            for _ in range(case["align"])]


def _feature_inputs(case, seed):
    rng = np.random.default_rng(seed)
    k, n = case["align"], case["taxa"]
    trees = [_yule(n, rng, 1.0) for _ in range(k)]
    scale = np.exp(rng.uniform(math.log(0.01), math.log(0.25), k))
    eig, pis, cats = [], [], []
    for _ in range(k):
        pi = rng.dirichlet(np.full(4, 6.0))
        V, lam, W = _eigen(_rate_matrix(np.exp(rng.normal(0.0, 0.5, 6)), pi), pi)
        eig.append(np.concatenate([V.ravel(), W.ravel(), lam]))
        pis.append(pi)
    shapes = np.exp(rng.uniform(math.log(0.15), math.log(4.0), 8))
    table = [_gamma_rates(a, case["cats"]) for a in shapes]
    cats = [table[i % 8] for i in range(k)]
    return dict(n_taxa=n, n_sites=case["sites"], left=np.stack([t["left"] for t in trees]),
                right=np.stack([t["right"] for t in trees]), roots=np.array([t["root"] for t in trees], np.int32),
                blen=np.stack([t["blen"] * s for t, s in zip(trees, scale)]), eig=np.stack(eig), pi=np.stack(pis),
                cat_rates=np.stack(cats), gap_frac=case["gap"], seed=int(seed))


def _mlp_data(case, seed):
    """Standardised features and targets that depend on them."""
    rng = np.random.default_rng(seed)
    x = rng.normal(0.0, 1.0, (case["samples"], 256)).astype(np.float32)
    w = rng.normal(0.0, 1.0, (256, 12)) / 16.0
    t = (x @ w + 0.3 * rng.normal(0.0, 1.0, (case["samples"], 12))).astype(np.float32)
    return x, t


# ---- one pass --------------------------------------------------------------

def prepare(case, seed):
    import phylommand_amd as P
    kind = case["kind"]
    if kind == "features":
        return dict(kind=kind, args=_feature_inputs(case, seed))
    if kind == "mlp":
        x, t = _mlp_data(case, seed)
        return dict(kind=kind, net=P.MLP(256, case["hidden"], 12, max_batch=case["batch"], seed=seed % 1000 + 1), x=x,
                    t=t, batch=case["batch"])
    if kind == "batch":
        b = P.Batch(case["cats"], P.PREC_FP32)
        for i, (n, m, alpha) in enumerate(_batch_sizes(case)):
            p = _problem(case, seed * 1000 + i, n, m, alpha)
            t = p["t"]
            b.add(p["masks"], t["left"], t["right"], t["root"], p["lengths"], p["Q"], p["pi"], p["rates"],
                  p["weights"], nni_mode=1)
        b.finalize(autotune=True)
        return dict(kind=kind, batch=b)
    if kind == "fit":
        p, rel, x = _fit_point(case, seed)
    else:
        p = _problem(case, seed)
    f64 = kind in ("fit", "dna_site", "protein_site")
    ctx = P.Context(0, P.PREC_FP64 if f64 else P.PREC_FP32)
    t = p["t"]
    ctx.set_tips(p["masks"], p["S"])
    ctx.set_topology(t["left"], t["right"], t["root"])
    if kind == "fit":
        return dict(kind=kind, ctx=ctx, rel=rel, cats=case["cats"], x=x)
    ctx.set_edge_lengths(p["lengths"])
    ctx.set_model(p["Q"], p["pi"], p["pi"], P.P_EIGEN)
    ctx.set_categories(p["rates"], p["weights"])
    return dict(kind=kind, ctx=ctx, lengths=p["lengths"], t=t)


def run(state):
    kind = state["kind"]
    if kind == "features":
        from phylommand_amd import sim_features
        return dict(features=sim_features(**state["args"]))
    if kind == "mlp":
        losses = state["net"].train(state["x"], state["t"], epochs=1, batch=state["batch"], lr=1e-3, seed=3)
        return dict(losses=losses, params=state["net"].params())
    if kind == "batch":
        totals, variants = state["batch"].run()
        return dict(totals=totals, variants=variants)
    ctx = state["ctx"]
    if kind == "fit":
        return dict(lnl=np.array([ctx.gtr_gamma_lnl(state["rel"], state["cats"], state["x"])]))
    if kind == "tree":
        t = state["t"]
        ctx.set_topology(t["left"], t["right"], t["root"])
    ctx.set_edge_lengths(state["lengths"])
    if kind in ("nni_dna", "nni_protein"):
        base, variants = ctx.nni_score(1)
        return dict(base=np.array([base]), node=np.array([v for v, _, _ in variants], np.int32),
                    side=np.array([s for _, s, _ in variants], np.int32),
                    lnl=np.array([x for _, _, x in variants]))
    if kind in ("dna_site", "protein_site"):
        total, site = ctx.loglik(per_site=True)
        return dict(total=np.array([total]), site=site)
    return dict(total=np.array([ctx.loglik()]))


# ---- what a pass cannot do without -----------------------------------------

def _prune_work(n, m, S, C):
    """One likelihood evaluation: the tips read once (a byte each), the
    transition matrices and the site values; two S x S products and a
    product of the children per inner node, site and category."""
    return (n * m + (2 * n - 1) * C * S * S * 8.0 + 8.0 * m, (n - 1.0) * m * C * (4 * S * S + S))


def work(case):
    kind = case["kind"]
    if kind == "features":
        k, n, m = case["align"], case["taxa"], case["sites"]
        # a draw per node and site, 16 joint counts per pair of taxa and site
        return dict(bytes=k * (2 * n * 16.0 + 36 * 8 + 256 * 4), flops=k * m * (2.0 * n * 10 + n * (n - 1) / 2))
    if kind == "mlp":
        h, steps = case["hidden"], case["samples"] // case["batch"]
        params = 256.0 * h + h + h * h + h + 12 * h + 12
        return dict(bytes=steps * (params * 4 * 6 + case["batch"] * 268 * 4.0),
                    flops=steps * case["batch"] * 2.0 * (2 * 256 * h + 3 * h * h + 3 * 12 * h))
    if kind == "batch":
        by = fl = 0.0
        for n, m, _ in _batch_sizes(case):
            b, f = _prune_work(n, m, 4, case["cats"])
            by, fl = by + b, fl + 4 * f      # the tree, the outer partials, two variants an inner edge
        return dict(bytes=by, flops=fl)
    b, f = _prune_work(case["taxa"], case["sites"], _states(case), case["cats"])
    return dict(bytes=b, flops=4 * f if kind.startswith("nni") else f)


# ---- the same in 64 bits ---------------------------------------------------

def _tip(masks_row, S):
    bits = torch.from_numpy(masks_row.astype(np.int64)).to(DEV)
    return ((bits[:, None] >> torch.arange(S, device=DEV)) & 1).double()


def _scaled(x, lg):
    """x [C, m, S] with its per-site maximum brought to 1, the log of it added
    to lg [m]."""
    mx = x.amax(dim=(0, 2)).clamp_min(1e-300)
    return x / mx[None, :, None], lg + mx.log()


class _Pruned:
    """Every node's partials of a problem, FP64."""

    def __init__(self, p, lengths=None):
        self.p, self.t = p, p["t"]
        self.P = _transition(p["Q"], p["pi"], p["lengths"] if lengths is None else lengths, p["rates"])
        self.n = p["masks"].shape[0]
        self.m = p["masks"].shape[1]
        self.keep = {}

    def part(self, v):
        """(P_v L_v [C, m, S], log scale [m]): what v's edge passes up."""
        if v < self.n:
            x, lg = _tip(self.p["masks"][v], self.p["S"])[None].expand(self.p["C"], -1, -1), 0.0
        else:
            x, lg = self.keep[v]
        return torch.matmul(x.contiguous(), self.P[v].transpose(1, 2).contiguous()), lg

    def join(self, parts):
        x, lg = parts[0][0], torch.zeros(self.m, dtype=torch.float64, device=DEV) + parts[0][1]
        for y, l2 in parts[1:]:
            x, lg = x * y, lg + l2
        return _scaled(x, lg)

    def sites(self, x, lg):
        pi = torch.from_numpy(self.p["pi"]).to(DEV)
        w = torch.from_numpy(self.p["weights"]).to(DEV)
        return ((x * pi).sum(2) * w[:, None]).sum(0).log() + lg

    def evaluate(self, keep_all=False):
        for v in reversed(_preorder(self.t)):
            if v < self.n:
                continue
            l, r = int(self.t["left"][v]), int(self.t["right"][v])
            self.keep[v] = self.join([self.part(l), self.part(r)])
            if not keep_all:
                self.keep.pop(l, None), self.keep.pop(r, None)
        return self.sites(*self.keep[self.t["root"]])

    def product(self, v, node):
        return torch.matmul(node[0].contiguous(), self.P[v].transpose(1, 2).contiguous()), node[1]

    def variant(self, v, side, par):
        """lnL after exchanging v's left (side 0) or right child with v's
        sibling, or, at the root, with the sibling's left child."""
        t, r = self.t, self.t["root"]
        l, q, u = int(t["left"][v]), int(t["right"][v]), int(par[v])
        out, stay = (l, q) if side == 0 else (q, l)
        sib = int(t["right"][u] if t["left"][u] == v else t["left"][u])
        if u == r:
            a, b = int(t["left"][sib]), int(t["right"][sib])
            nv = self.join([self.part(a), self.part(stay)])
            ns = self.join([self.part(out), self.part(b)])
            return self.sites(*self.join([self.product(v, nv), self.product(sib, ns)])).sum()
        cur = self.join([self.part(sib), self.part(stay)])
        cur = self.join([self.product(v, cur), self.part(out)])
        while u != r:
            up = int(par[u])
            other = int(t["right"][up] if t["left"][up] == u else t["left"][up])
            cur = self.join([self.product(u, cur), self.part(other)])
            u = up
        return self.sites(*cur).sum()


def _neighbours(t, n):
    """(node, side) of every interchange: both sides of every inner edge, the
    root's two edges counted once (the left child's)."""
    r, par = t["root"], _parents(t)
    both = t["left"][r] >= n and t["right"][r] >= n
    return [(v, s) for v in range(n, len(par)) if v != r and not (par[v] == r and (not both or v == t["right"][r]))
            for s in (0, 1)], par


def _nni_exact(p):
    e = _Pruned(p)
    base = e.evaluate(keep_all=True).sum()
    which, par = _neighbours(p["t"], e.n)
    return base, which, [e.variant(v, s, par) for v, s in which]


def _host(x):
    return np.array([float(v) for v in x])


def exact(case, seed):
    kind = case["kind"]
    if kind in ("features", "mlp"):      # random draws, the order of a shuffled epoch
        return None
    if kind == "batch":
        tot, var = [], []
        for i, (n, m, alpha) in enumerate(_batch_sizes(case)):
            base, _, lnl = _nni_exact(_problem(case, seed * 1000 + i, n, m, alpha))
            tot.append(base)
            var += lnl
        return dict(totals=_host(tot), variants=_host(var))
    if kind == "fit":
        p, rel, x = _fit_point(case, seed)
        pi = np.exp(np.append(x[5:8], 0.0))
        pi /= pi.sum()
        p = dict(p, pi=pi, Q=_rate_matrix(np.exp(np.append(x[:5], 0.0)), pi),
                 rates=_gamma_rates(math.exp(x[8]), p["C"]))
        return dict(lnl=_host([_Pruned(p, rel * math.exp(x[9])).evaluate().sum()]))
    p = _problem(case, seed)
    if kind.startswith("nni"):
        base, which, lnl = _nni_exact(p)
        return dict(base=_host([base]), node=None, side=None, lnl=_host(lnl))
    site = _Pruned(p).evaluate()
    if kind in ("dna_site", "protein_site"):
        return dict(total=_host([site.sum()]), site=site.cpu().numpy())
    return dict(total=_host([site.sum()]))
