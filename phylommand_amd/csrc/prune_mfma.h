// prune_mfma.h -- launches of the matrix-core pruning walker (4 < S <= 32).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "nni.h"
#include "prune_device.h"

// Operand slots that cover S states, four a slot.
__host__ __device__ constexpr int mfma_slots(int S) { return (S + 3) / 4; }

// Taxa whose tip masks a wide-state workgroup stages in LDS.
constexpr int kMfmaTipLdsTaxa = 128;

struct MfmaArgs {
    bool f64 = false;
    int C = 1, S = 0;
    const Op* ops = nullptr;
    const int* prog = nullptr;
    const uint32_t* tips = nullptr;
    void* clv = nullptr;
    int* scl = nullptr;
    const double* Pm = nullptr;
    const double* PTm = nullptr;
    const double* roots = nullptr;
    const double* site_w = nullptr;
    double* site_lnl = nullptr;
    double* partial = nullptr;
    int m = 0, m_pad = 0, n_taxa = 0;
    bool tip_lds = false;              // stage the tips (n_taxa <= kMfmaTipLdsTaxa)
    dim3 grid;
    // work mapping (prune_mfma_kernel)
    int n_main = 0, prog_main = -1, blk0 = 0, prog_piece = 0, tail0 = 0, n_tail = 1;
    unsigned* fold = nullptr;
    double* fold_out = nullptr;
};

hipError_t mfma_launch(const MfmaArgs& a, hipStream_t st);
// Workgroups of the staging walker that one CU holds at once, 0 if unknown.
int mfma_resident(bool f64, int C, int S);
// By value in kernel arguments: nothing to copy to the device beforehand.
struct RootWeights {
    double v[40];      // roots[]: per-state weights, category weights from 32
};
struct PRates {
    double v[8];       // category rates
};

// P, the walkers' operands of it (Pm; PmT of the transpose, where set) and the
// tip columns PTm: from the eigen system (device
// memory) and lengths (device or mapped host memory), or with
// eff null from P as it is (pwide_kernel).
// Writes the root and category weights `roots` to d_roots too.
hipError_t mfma_matrices(const double* V, const double* Vinv, const double* lam, const double* eff, const PRates& rates,
                         const RootWeights& roots, int S, int Sp, int C, int n_nodes, double* P, double* Pm, double* PmT,
                         double* PTm, double* d_roots, hipStream_t st);
// NNI walks (nni.h; a.tips, a.P and the batch members unused).
hipError_t nni_mfma_launch(const NniArgs& a, int S, const uint32_t* tips, const double* Pm, const double* PmT,
                           const double* PTm, hipStream_t st);
