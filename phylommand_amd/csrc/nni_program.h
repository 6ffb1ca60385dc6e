// nni_program.h -- programs of the NNI neighbourhood scorers (host code, no HIP).
//
// A neighbourhood is scored by outer partials.  For an inner node u let O_u
// be the probability of the data outside u's subtree given u's state (at the
// root: the root weights).  With A = P_a L_a and B = P_b L_b the factors of
// u's children a and b, the outer partial of a is O_a = P_a^T (O_u x B) (x
// elementwise), and for an inner child v of u with children x, y (factors X,
// Y) and sibling factor S the two trees that exchange x or y with the sibling
// have the site likelihoods
//     sum_i (O_u x X)_i (P_v (S x Y))_i   and   sum_i (O_u x Y)_i (P_v (S x X))_i
// (branch lengths move with their subtrees, as in tree::interchange,
// tree.cpp:2480-2518).  One preorder walk over the inner edges therefore
// scores every variant with five matrix-vector products an edge, where a
// program per variant repeats the whole path to the root.  Edges that are
// reached again (below) add descents: the two walks of a 128-taxon tree with 250
// variants hold 190 ops, 60 of them descents alone, and 818 products (625 for
// its edges) against 3,952.
#pragma once

#include <algorithm>
#include <vector>

// One step of the preorder walk: an inner edge.  The walk holds O of its
// current node u and B, the factor of the child of u that is not entered
// first; only what the next step needs stays in registers.
enum NniFlags : int {
    NNI_INIT = 1,       // O = root weights, B = factor of y (x, y: the root's children)
    NNI_POP = 2,        // O from a save slot
    NNI_FETCH_S = 4,    // the sibling's factor S is computed again (else S = B)
    NNI_SAVE = 8,       // O kept in a save slot for the sibling edge
    NNI_DESC = 16,      // v becomes the current node: O = P_v^T (O x S), B = factor of y
    NNI_PAIR = 32,      // score the edge's two variants into var, var + 1
    NNI_ROOT = 64,      // score one variant at a child v of the root into var: v's child
                        // x changes places with the sibling's left child c (d: its
                        // right child); the root sees P_v (C x Y) and P_s (X x D)
    NNI_XY = 128        // x is v's right child (the child entered first is always x)
};

struct alignas(16) NniOp {
    int v;           // the edge's lower end
    int x, y;        // v's children, -1 for none (INIT: the root's)
    int s;           // v's sibling, -1 for none
    int flags;       // NniFlags | save slot to read << 8 | save slot to write << 12
    int var;         // output index of the edge's first variant
    int c, d;        // NNI_ROOT: the sibling's children
};
constexpr int nni_pop_slot(int flags) { return flags >> 8 & 15; }
constexpr int nni_save_slot(int flags) { return flags >> 12 & 15; }

// The op after ops[k] of a program that ends at k1, for a walk that fetches its
// operands x and y ahead.  Past the end it names none: in a batch the op there
// begins another tree's walk, whose nodes this tree's offsets do not reach.
// (ops[k1] is always readable: the next program's first op or a last pad.)
constexpr NniOp nni_ahead(const NniOp* ops, int k, int k1) {
    NniOp o = ops[k + 1];
    if (k + 1 >= k1) o.x = o.y = -1;
    return o;
}

// Save slots a walk may hold (LDS; an edge whose upper node is no longer held
// is reached again from its nearest held ancestor).  One slot leaves a DNA
// workgroup of 128 taxa 27 KB of LDS, five a CU; two left four a CU and ran
// 0.69 against 0.59 ms (128 taxa x 100,000 sites).
constexpr int kNniSaves = 1;

// Builds the walks over inner edges of one tree.
// pair_of[v]: first output index of the two variants of inner node v's edge,
// -1 when they are not scored.  Edges are taken in preorder, childless edges
// first and the largest subtree last at each node, so that a node is held in
// a save slot only while a smaller sibling subtree is walked; where the slots are
// taken, the later sibling is reached by walking down again from its nearest held
// ancestor, or from the root.  The preorder is cut into segments of at most
// max_edges edges, each a program of its own that first walks from the root to
// its start: more workgroups where there are few sites.
template <class TV>
void build_nni_walks(const TV* c, const std::vector<int>& pair_of, int max_edges, std::vector<NniOp>& ops,
                     std::vector<int>& begin) {
    const int n = c->n_nodes, nt = c->n_taxa, root = c->root;
    const auto inner = [&](int v) { return v >= nt; };
    std::vector<int> par(n, -1), order, size(n, 0), stack{root};
    while (!stack.empty()) {
        const int v = stack.back();
        stack.pop_back();
        order.push_back(v);
        for (int k : {c->left[v], c->right[v]})
            if (k >= 0) {
                par[k] = v;
                if (inner(k)) stack.push_back(k);
            }
    }
    std::vector<char> wanted(n, 0);     // v's edge or one below it is scored
    for (size_t i = order.size(); i-- > 0;) {
        const int v = order[i];
        size[v] += 1;
        if (pair_of[v] >= 0) wanted[v] = 1;
        if (v != root) {
            size[par[v]] += size[v];
            wanted[par[v]] |= wanted[v];
        }
    }
    // inner edges in walk order, by their lower node
    struct Edge { int v; bool last; };
    std::vector<Edge> edges;
    const auto kids_of = [&](int u, int (&k)[2]) {
        int m = 0;
        for (int w : {c->left[u], c->right[u]})
            if (w >= 0 && inner(w) && wanted[w]) k[m++] = w;
        if (m == 2 && size[k[1]] < size[k[0]]) std::swap(k[0], k[1]);
        return m;
    };
    {
        std::vector<Edge> st;
        const auto push_kids = [&](int u) {
            int k[2];
            const int m = kids_of(u, k);
            for (int i = m; i-- > 0;) st.push_back({k[i], i == m - 1});
        };
        push_kids(root);
        while (!st.empty()) {
            const Edge e = st.back();
            st.pop_back();
            edges.push_back(e);
            push_kids(e.v);
        }
    }
    const auto sibling = [&](int v) { return c->left[par[v]] == v ? c->right[par[v]] : c->left[par[v]]; };
    const size_t per = (size_t)std::max(1, max_edges);
    const size_t n_seg = (edges.size() + per - 1) / per;
    for (size_t seg = 0, e0 = 0; seg < n_seg; ++seg) {
        const size_t e1 = edges.size() * (seg + 1) / n_seg;
        // later[u]: u's edges still to come in this segment
        std::vector<int> later(n, 0), slot(n, -1);
        for (size_t e = e0; e < e1; ++e) ++later[par[edges[e].v]];
        bool used[kNniSaves] = {};
        int cur = -1;
        const size_t first = ops.size();
        const auto edge_op = [&](int v, bool pop) {
            NniOp o{v, c->left[v], c->right[v], sibling(v), 0, -1, -1, -1};
            if (pop) o.flags = NNI_POP | slot[par[v]] << 8;
            if (pop || ops.size() == first || !(ops.back().flags & (NNI_DESC | NNI_INIT))) {
                o.flags |= NNI_FETCH_S;
            } else if (ops.back().x != v) {      // the op before enters v: its x
                std::swap(ops.back().x, ops.back().y);
                ops.back().flags |= NNI_XY;
            }
            return o;
        };
        const auto init_op = [&]() {
            ops.push_back({root, c->left[root], c->right[root], -1, NNI_INIT, -1, -1, -1});
        };
        for (size_t e = e0; e < e1; ++e) {
            const int v = edges[e].v, u = par[v];
            // bring u's state in: current, saved, or reached from an ancestor that is
            std::vector<int> path;
            int a = u;
            while (a != cur && slot[a] < 0 && a != root) {
                path.push_back(a);
                a = par[a];
            }
            bool pop = a != cur && slot[a] >= 0;
            if (a != cur && !pop) init_op();
            for (size_t i = path.size(); i-- > 0;) {
                NniOp o = edge_op(path[i], pop);
                o.flags |= NNI_DESC;
                ops.push_back(o);
                pop = false;
            }
            if (!path.empty() || !pop) cur = u;
            if (u == root && pair_of[v] >= 0) {
                const int sib = sibling(v), l = c->left[v], r = c->right[v];
                for (int side = 0; side < 2; ++side)
                    ops.push_back({v, side ? r : l, side ? l : r, sib, NNI_ROOT | (pop ? NNI_POP | slot[u] << 8 : 0),
                                   pair_of[v] + side, c->left[sib], c->right[sib]});
            }
            NniOp o = edge_op(v, pop);
            if (pair_of[v] >= 0 && u != root) {
                o.var = pair_of[v];
                o.flags |= NNI_PAIR;
            }
            --later[u];
            if (later[u] == 0 && slot[u] >= 0) {     // u's last edge: its slot is free
                used[slot[u]] = false;
                slot[u] = -1;
            }
            const bool desc = later[v] > 0;
            if (desc) {
                o.flags |= NNI_DESC;
                if (later[u] > 0 && slot[u] < 0)
                    for (int k = 0; k < kNniSaves; ++k)
                        if (!used[k]) {
                            used[k] = true;
                            slot[u] = k;
                            o.flags |= NNI_SAVE;
                            o.flags |= k << 12;
                            break;
                        }
                cur = v;
            } else if (pop) {
                cur = u;
            }
            ops.push_back(o);
        }
        begin.push_back((int)ops.size());
        e0 = e1;
    }
}
