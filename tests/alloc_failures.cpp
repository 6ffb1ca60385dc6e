// Every allocation of a few call sequences made to fail in turn, under a
// stand-in for the HIP runtime (hip_stand_in.h): the call that meets the failure
// returns an error, and it and the calls after it launch nothing on memory that
// is not there.  Prints "ok" or the sequence, the failure and what was launched.
#include "hip_stand_in.h"

#include <functional>

#include "../include/phylo_hip.h"
#include "../include/phylo_learn.h"

static int bad = 0, runs = 0;

// runs body with no failure, then with each of its allocations failing
static void sequence(const char* name, const std::function<void()>& body) {
    for (long k = -1;; k = k < 0 ? 1 : k + 1) {
        stand_in::allocs = 0;
        stand_in::fail_at = k;
        stand_in::faults.clear();
        body();
        ++runs;
        for (const std::string& f : stand_in::faults) {
            printf("%s, allocation %ld failing: %s\n", name, k, f.c_str());
            ++bad;
        }
        if (!stand_in::live.empty()) {
            printf("%s, allocation %ld failing: %zu buffers left\n", name, k, stand_in::live.size());
            ++bad;
            stand_in::live.clear();
        }
        if (k >= 0 && stand_in::allocs < k) return;      // no such allocation any more
    }
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

int main() {
    sequence("mlp", mlp);
    if (stand_in::launches < 100 || runs < 20) {
        printf("too little ran: %ld launches, %d runs\n", stand_in::launches, runs);
        return 1;
    }
    if (!bad) printf("ok %d runs, %ld launches\n", runs, stand_in::launches);
    return bad ? 1 : 0;
}
