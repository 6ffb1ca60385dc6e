// Every allocation of a few call sequences, and every two, made to fail, under a
// stand-in for the HIP runtime (hip_stand_in.h): the call that meets the failure
// returns an error, and it and the calls after it launch nothing on memory that
// is not there.  Prints "ok" or the sequence, the failure and what was launched.
#include "hip_stand_in.h"

#include <cstdint>
#include <functional>
#include <new>

#include "../include/phylo_hip.h"
#include "../include/phylo_learn.h"

static int bad = 0, runs = 0;

// host allocations above the limit fail
static size_t host_limit = SIZE_MAX;
void* operator new(size_t n, const std::nothrow_t&) noexcept { return n > host_limit ? nullptr : malloc(n); }
void* operator new[](size_t n, const std::nothrow_t&) noexcept { return n > host_limit ? nullptr : malloc(n); }
void* operator new(size_t n) {
    if (void* p = operator new(n, std::nothrow)) return p;
    throw std::bad_alloc();
}
void* operator new[](size_t n) { return operator new(n); }
void operator delete(void* p) noexcept { free(p); }
void operator delete[](void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }
void operator delete[](void* p, size_t) noexcept { free(p); }

// runs body with no failure, then with each of its allocations failing, and each
// two of them
static void sequence(const char* name, const std::function<void()>& body) {
    const auto run = [&](long a, long b) {
        stand_in::allocs = 0;
        stand_in::fail_at[0] = a;
        stand_in::fail_at[1] = b;
        stand_in::faults.clear();
        body();
        ++runs;
        if (!stand_in::live.empty()) stand_in::faults.push_back(std::to_string(stand_in::live.size()) + " buffers left");
        stand_in::live.clear();
        for (const std::string& f : stand_in::faults) printf("%s, allocations %ld, %ld failing: %s\n", name, a, b, f.c_str());
        bad += (int)stand_in::faults.size();
        return stand_in::allocs;
    };
    run(-1, -1);
    for (long a = 1; run(a, -1) >= a; ++a)
        for (long b = a + 1; run(a, b) >= b; ++b) {}
}

static void mlp() {
    const int n = 640, n_in = 3, n_out = 5;
    std::vector<float> x(n * n_in, 0.5f), t(n * n_out, 0.25f), y(n * n_out), g;
    float loss[2];
    phylo_mlp* p = nullptr;
    if (phylo_mlp_create(0, n_in, 8, n_out, 16, 1, &p) != PHYLO_OK) return;
    g.resize(phylo_mlp_n_params(p));
    // training, and gradients and outputs after it, whether it failed or not
    for (int rows : {32, n}) {
        phylo_mlp_set_data(p, rows, x.data(), t.data());
        phylo_mlp_train(p, 2, 16, 1e-3f, 1, loss);
        phylo_mlp_grad(p, 16, x.data(), t.data(), loss, g.data());
        phylo_mlp_forward(p, rows, x.data(), y.data());
    }
    phylo_mlp_destroy(p);
}

struct Tree {
    int n = 0, root = -1;
    std::vector<int32_t> left, right;
    std::vector<double> len;
    // a caterpillar (or, paired, a balanced tree) of n_taxa tips
    Tree(int n_taxa, bool paired) : n(2 * n_taxa - 1), left(n, -1), right(n, -1), len(n, 0.1) {
        std::vector<int> f;
        for (int i = 0; i < n_taxa; ++i) f.push_back(i);
        for (int v = n_taxa; v < n; ++v) {
            left[v] = f[0];
            right[v] = f[1];
            f.erase(f.begin(), f.begin() + 2);
            f.insert(paired ? f.end() : f.begin(), v);
        }
        root = f[0];
    }
};

// one context through new trees, neighbourhoods, simulation and precisions, on
// an alphabet of S states
static void context(int S) {
    const int n = 20, m = 300;
    const std::vector<uint32_t> masks(n * m, 1);
    std::vector<double> Q(S * S, 1.0 / (S - 1)), pi(S, 1.0 / S), site(m), lnl(200), P(8 * S * S), clv(m * 8 * S);
    for (int i = 0; i < S; ++i) Q[i * S + i] = -1.0;
    const double rates[4] = {0.2, 0.6, 1.1, 2.1}, w[4] = {0.25, 0.25, 0.25, 0.25};
    std::vector<uint8_t> states(400 * 50);
    phylo_ctx* c = nullptr;
    if (phylo_create(0, &c) != PHYLO_OK) return;
    double total;
    int nv;
    const Tree small(n, true), other(n, false);
    phylo_set_tips(c, n, m, S, masks.data());
    for (const Tree* t : {&small, &other, &small}) {
        phylo_set_topology(c, t->n, t->root, t->left.data(), t->right.data());
        phylo_set_edge_lengths(c, t->len.data());
        phylo_set_model(c, S, Q.data(), pi.data(), pi.data(), PHYLO_P_EIGEN);
        phylo_set_categories(c, 4, rates, w);
        phylo_loglik(c, site.data(), &total);
        phylo_set_edge_lengths(c, t->len.data());
        phylo_simulate(c, 50, pi.data(), 1, states.data());
        phylo_nni_score(c, 1, 200, lnl.data(), nullptr, nullptr, &nv, nullptr);
        phylo_set_precision(c, t == &other ? PHYLO_PREC_FP32 : PHYLO_PREC_FP64);
        phylo_loglik(c, nullptr, &total);
        phylo_node_partials(c, n + 1, clv.data(), nullptr);
        phylo_get_pmatrix(c, 1, P.data());
    }
    // more taxa, and more again: larger programs, first met by whatever failed
    // above, the ones before perhaps never copied
    const std::vector<uint32_t> more(100 * m, 2);
    for (int taxa : {50, 100}) {
        const Tree t(taxa, true);
        phylo_set_tips(c, taxa, m, S, more.data());
        phylo_set_topology(c, t.n, t.root, t.left.data(), t.right.data());
        phylo_set_edge_lengths(c, t.len.data());
        phylo_loglik(c, site.data(), &total);
        if (taxa == 50) continue;
        phylo_set_edge_lengths(c, t.len.data());
        phylo_simulate(c, 50, pi.data(), 1, states.data());
        phylo_loglik(c, site.data(), &total);
    }
    phylo_destroy(c);
}

static void batch() {
    const int m = 300;
    const std::vector<uint32_t> masks(60 * m, 1);
    std::vector<double> Q(16, 1.0 / 3), w(4, 0.25), tot(3), lnl(400);
    for (int i = 0; i < 4; ++i) Q[5 * i] = -1.0;
    phylo_batch* b = nullptr;
    if (phylo_batch_create(0, 4, PHYLO_PREC_FP32, &b) != PHYLO_OK) return;
    for (int n : {8, 60, 5}) {
        const Tree t(n, n == 60);
        phylo_batch_add(b, n, m, 4, masks.data(), t.n, t.root, t.left.data(), t.right.data(), t.len.data(), Q.data(), w.data(),
                        w.data(), w.data(), w.data(), n == 5 ? -1 : 1, nullptr);
    }
    if (phylo_batch_finalize(b, 1) == PHYLO_OK) phylo_batch_run(b, tot.data(), lnl.data());
    phylo_batch_destroy(b);
}

static int features(int n_align, bool limited) {
    const int n = 6;
    const Tree t(n, true);
    std::vector<int32_t> left, right, roots(n_align, t.root);
    std::vector<double> len, eig(36 * n_align, 0.1), pi(4 * n_align, 0.25), rates(2 * n_align, 1.0);
    for (int k = 0; k < n_align; ++k) {
        left.insert(left.end(), t.left.begin(), t.left.end());
        right.insert(right.end(), t.right.begin(), t.right.end());
        len.insert(len.end(), t.len.begin(), t.len.end());
    }
    std::vector<float> out(256 * n_align);
    std::vector<uint32_t> masks(n_align * n * 40);
    if (limited) host_limit = (size_t)n_align * 256;      // (past the library's small vectors)
    int rc = 1;
    try {
        rc = phylo_sim_features(0, n_align, n, 40, 2, left.data(), right.data(), roots.data(), len.data(), eig.data(), pi.data(),
                                rates.data(), 0.0, 1, out.data(), masks.data());
    } catch (const std::bad_alloc&) {
        stand_in::faults.push_back("an exception left phylo_sim_features");
    }
    host_limit = SIZE_MAX;
    return rc;
}

int main() {
    sequence("mlp", mlp);
    sequence("context, 4 states", [] { context(4); });
    sequence("context, 20 states", [] { context(20); });
    sequence("batch", batch);
    sequence("features", [] { features(64, false); });
    // the copy of its inputs on the host fails
    sequence("features, no host memory", [] {
        if (features(64, true) == PHYLO_OK) stand_in::faults.push_back("no error from phylo_sim_features");
    });
    if (stand_in::launches < 100 || runs < 20) {
        printf("too little ran: %ld launches, %d runs\n", stand_in::launches, runs);
        return 1;
    }
    if (!bad) printf("ok %d runs, %ld launches\n", runs, stand_in::launches);
    return bad ? 1 : 0;
}
