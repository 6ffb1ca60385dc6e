// CPU check of what an NNI walk fetches ahead (csrc/nni_program.h, nni_ahead):
// the walks of several trees of different sizes lie in one op buffer, as a
// batch lays them out, and a walk's operands, those fetched during its last op
// among them, must be nodes of its own tree: a kernel indexes them with its own
// problem's offsets.  Prints "ok" or the first operand of another tree.
#include <cstdio>
#include <random>
#include <vector>

#include "../phylommand_amd/csrc/nni_program.h"

struct Tree {
    int n_taxa = 0, n_nodes = 0, root = -1;
    std::vector<int> left, right;
};

static std::mt19937 rng(11);

// joins random nodes of a forest, or (caterpillar) each tip to the tree so far
static Tree make(int n, bool caterpillar) {
    Tree t;
    t.n_taxa = n;
    t.n_nodes = 2 * n - 1;
    t.left.assign(t.n_nodes, -1);
    t.right.assign(t.n_nodes, -1);
    std::vector<int> forest;
    for (int i = 0; i < n; ++i) forest.push_back(i);
    for (int v = n; v < t.n_nodes; ++v) {
        int kid[2];
        for (int& k : kid) {
            const size_t i = caterpillar ? (&k == kid ? forest.size() - 1 : 0) : rng() % forest.size();
            k = forest[i];
            forest.erase(forest.begin() + (long)i);
        }
        t.left[v] = kid[0];
        t.right[v] = kid[1];
        forest.push_back(v);
    }
    t.root = forest[0];
    return t;
}

int main() {
    long checked = 0;
    const std::vector<std::vector<int>> batches = {{8, 256}, {256, 8}, {4, 5, 200, 6, 130, 4}, {12, 12}, {4}, {3, 90, 5}};
    for (const auto& taxa : batches)
        for (int per : {1, 6, 64})
            for (int shape = 0; shape < 2; ++shape) {
                std::vector<Tree> trees;
                std::vector<NniOp> ops;
                std::vector<int> begin{0}, owner;
                for (int n : taxa) {
                    trees.push_back(make(n, shape == 1));
                    const Tree& t = trees.back();
                    std::vector<int> pair_of(t.n_nodes, -1);
                    int n_out = 0;
                    for (int v = t.n_taxa; v < t.n_nodes; ++v)
                        if (v != t.root) {
                            pair_of[v] = n_out;
                            n_out += 2;
                        }
                    const size_t first = begin.size();
                    build_nni_walks(&t, pair_of, per, ops, begin);
                    owner.resize(owner.size() + begin.size() - first, (int)trees.size() - 1);
                }
                ops.push_back(NniOp{});     // (readable after the last program)
                for (size_t p = 0; p + 1 < begin.size(); ++p) {
                    const Tree& t = trees[owner[p]];
                    const auto inside = [&](int node) { return node >= -1 && node < t.n_nodes; };
                    NniOp nx = ops[begin[p]];
                    for (int k = begin[p]; k < begin[p + 1]; ++k, ++checked) {
                        const NniOp op = nx;
                        nx = nni_ahead(ops.data(), k, begin[p + 1]);
                        if (op.v != ops[k].v || op.x != ops[k].x || op.y != ops[k].y || op.flags != ops[k].flags) {
                            printf("program %zu op %d is not the one read ahead\n", p, k);
                            return 1;
                        }
                        if (!inside(nx.x) || !inside(nx.y)) {
                            printf("program %zu of a %d-taxon tree fetches nodes %d, %d during op %d of [%d, %d)\n", p,
                                   t.n_taxa, nx.x, nx.y, k, begin[p], begin[p + 1]);
                            return 1;
                        }
                    }
                    // nothing at all past its end: the next program may be another tree's
                    if (nx.x != -1 || nx.y != -1) {
                        printf("program %zu fetches nodes %d, %d past its end\n", p, nx.x, nx.y);
                        return 1;
                    }
                }
            }
    printf("ok %ld\n", checked);
    return checked > 2000 ? 0 : 1;
}
