// CPU check of the NNI walk programs (csrc/nni_program.h): random, caterpillar
// and balanced trees, some with single-child nodes, cut into segments of
// several sizes; every walk is interpreted in doubles over random factors and
// each variant's root value compared with the interchanged tree evaluated from
// its tips.  Operand indexes, save slots and output indexes are checked
// against their ranges.  Prints "ok" or the first mismatch.
#include <cmath>
#include <cstdio>
#include <functional>
#include <random>
#include <vector>

#include "../phylommand_amd/csrc/nni_program.h"

struct Tree {
    int n_taxa = 0, n_nodes = 0, root = -1;
    std::vector<int> left, right;
};
typedef std::vector<double> V4;

static std::mt19937 rng(7);
static double uni() { return std::uniform_real_distribution<double>(0.05, 1.0)(rng); }
static int below(int n) { return std::uniform_int_distribution<int>(0, n - 1)(rng); }

// joins random (shape 0), first-and-next (1: caterpillar) or paired (2:
// balanced) roots of a forest; unary: some joins get a single-child parent
static Tree make(int n, int shape, bool unary) {
    std::vector<std::pair<int, int>> kids;
    std::vector<int> forest;
    for (int i = 0; i < n; ++i) forest.push_back(i);
    const auto add = [&](int a, int b) {
        kids.push_back({a, b});
        return n + (int)kids.size() - 1;
    };
    while (forest.size() > 1) {
        int i = shape == 0 ? below((int)forest.size()) : 0;
        const int a = forest[i];
        forest.erase(forest.begin() + i);
        int j = shape == 0 ? below((int)forest.size()) : 0;
        const int b = forest[j];
        forest.erase(forest.begin() + j);
        int v = below(2) ? add(a, b) : add(b, a);
        if (unary && below(4) == 0) v = add(v, -1);
        if (shape == 1) forest.insert(forest.begin(), v);
        else forest.push_back(v);
    }
    Tree t;
    t.n_taxa = n;
    t.n_nodes = n + (int)kids.size();
    t.root = forest[0];
    t.left.assign(t.n_nodes, -1);
    t.right.assign(t.n_nodes, -1);
    for (size_t k = 0; k < kids.size(); ++k) {
        t.left[n + k] = kids[k].first;
        t.right[n + k] = kids[k].second;
    }
    return t;
}

int main() {
    long checked = 0;
    for (int trial = 0; trial < 240; ++trial) {
        const int shape = trial % 3, n = trial < 30 ? 2 + trial % 6 : 3 + below(60);
        const Tree t = make(n, shape, trial % 4 == 3);
        std::vector<V4> P(t.n_nodes, V4(16)), tip(t.n_taxa, V4(4));
        for (auto& p : P) for (double& x : p) x = uni();
        for (auto& p : tip) for (double& x : p) x = below(2);
        V4 rw(4);
        for (double& x : rw) x = uni();
        const auto mul = [](V4 a, const V4& b) { for (int i = 0; i < 4; ++i) a[i] *= b[i]; return a; };
        const auto mv = [&](int v, const V4& x) {
            V4 y(4, 0.0);
            for (int i = 0; i < 4; ++i) for (int j = 0; j < 4; ++j) y[i] += P[v][i * 4 + j] * x[j];
            return y;
        };
        std::vector<int> L = t.left, R = t.right, par(t.n_nodes, -1);
        std::function<V4(int)> part = [&](int v) -> V4 {
            if (v < t.n_taxa) return tip[v];
            V4 x(4, 1.0);
            for (int k : {L[v], R[v]}) if (k >= 0) x = mul(x, mv(k, part(k)));
            return x;
        };
        for (int v = 0; v < t.n_nodes; ++v) for (int k : {t.left[v], t.right[v]}) if (k >= 0) par[k] = v;
        std::vector<V4> clv(t.n_nodes);
        for (int v = 0; v < t.n_nodes; ++v) clv[v] = part(v);
        // pairs: every inner edge with a partner, some left out in some trials
        std::vector<int> pair_of(t.n_nodes, -1);
        int n_out = 0;
        for (int v = t.n_taxa; v < t.n_nodes; ++v) {
            if (v == t.root) continue;
            const int u = par[v], sib = t.left[u] == v ? t.right[u] : t.left[u];
            const int partner = u != t.root ? sib : sib >= 0 ? t.left[sib] : -1;
            if (partner < 0 || (trial % 5 == 4 && below(3) == 0)) continue;
            pair_of[v] = n_out;
            n_out += 2;
        }
        std::vector<double> want(n_out);
        for (int v = t.n_taxa; v < t.n_nodes; ++v) {
            if (pair_of[v] < 0) continue;
            const int u = par[v], sib = t.left[u] == v ? t.right[u] : t.left[u];
            for (int side = 0; side < 2; ++side) {
                L = t.left;
                R = t.right;
                const int out = side ? t.right[v] : t.left[v], in = u != t.root ? sib : t.left[sib];
                const int w = u != t.root ? u : sib;
                (side ? R[v] : L[v]) = in;
                (L[w] == in ? L[w] : R[w]) = out;
                const V4 r = part(t.root);
                for (int i = 0; i < 4; ++i) want[pair_of[v] + side] += rw[i] * r[i];
            }
        }
        L = t.left;
        R = t.right;
        for (int seg : {1, 3, 8, 1000}) {
            std::vector<NniOp> ops;
            std::vector<int> begin{0};
            build_nni_walks(&t, pair_of, seg, ops, begin);
            std::vector<double> got(n_out, -1.0);
            for (size_t p = 0; p + 1 < begin.size(); ++p) {
                V4 O, B, save[kNniSaves];
                const auto factor = [&](int node) {
                    if (node == -1) return V4(4, 1.0);
                    if (node < 0 || node >= t.n_nodes) { printf("operand out of range\n"); exit(1); }
                    return mv(node, clv[node]);
                };
                for (int k = begin[p]; k < begin[p + 1]; ++k) {
                    const NniOp& o = ops[k];
                    const V4 X = factor(o.x), Y = factor(o.y);
                    if (o.flags & NNI_INIT) { O = rw; B = Y; continue; }
                    if (o.flags & NNI_POP) {
                        if (nni_pop_slot(o.flags) >= kNniSaves) { printf("slot out of range\n"); return 1; }
                        O = save[nni_pop_slot(o.flags)];
                    }
                    const V4 S = o.flags & (NNI_FETCH_S | NNI_ROOT) ? factor(o.s) : B;
                    if (O.empty() || S.empty()) { printf("state not loaded\n"); return 1; }
                    double l[2] = {0, 0};
                    if (o.flags & NNI_PAIR) {
                        const V4 a = mul(mul(O, X), mv(o.v, mul(S, Y))), b = mul(mul(O, Y), mv(o.v, mul(S, X)));
                        for (int i = 0; i < 4; ++i) { l[0] += a[i]; l[1] += b[i]; }
                    } else if (o.flags & NNI_ROOT) {
                        const V4 a = mul(O, mul(mv(o.v, mul(factor(o.c), Y)), mv(o.s, mul(X, factor(o.d)))));
                        double l0 = 0.0;
                        for (double z : a) l0 += z;
                        if (o.var < 0 || o.var >= n_out || got[o.var] >= 0) { printf("output index\n"); return 1; }
                        got[o.var] = l0;
                        B.clear();
                        continue;
                    }
                    if (o.flags & NNI_PAIR) {
                        if (o.var < 0 || o.var + 1 >= n_out || got[o.var] >= 0) { printf("output index\n"); return 1; }
                        const int q = o.flags & NNI_XY ? 1 : 0;
                        got[o.var + q] = l[0];
                        got[o.var + 1 - q] = l[1];
                    }
                    if (o.flags & NNI_SAVE) {
                        if (nni_save_slot(o.flags) >= kNniSaves) { printf("slot out of range\n"); return 1; }
                        save[nni_save_slot(o.flags)] = O;
                    }
                    if (o.flags & NNI_DESC) {
                        const V4 x = mul(O, S);
                        O.assign(4, 0.0);
                        for (int j = 0; j < 4; ++j) for (int i = 0; i < 4; ++i) O[j] += P[o.v][i * 4 + j] * x[i];
                        B = Y;
                    } else {
                        B.clear();
                    }
                }
            }
            for (int k = 0; k < n_out; ++k, ++checked)
                if (!(std::fabs(got[k] - want[k]) <= 1e-11 * want[k])) {
                    printf("trial %d shape %d n %d segment %d variant %d: %.17g, want %.17g\n", trial, shape, n, seg, k,
                           got[k], want[k]);
                    return 1;
                }
        }
    }
    printf("ok %ld\n", checked);
    return checked > 10000 ? 0 : 1;
}
