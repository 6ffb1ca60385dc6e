// nni.h -- launches of the NNI neighbourhood walks (nni_program.h).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "nni_program.h"

// One problem's place in the launch's buffers (the arguments of every launch
// are these and base pointers).
struct NniInst {
    long tips_off, clv_off, scl_off, P_off;   // uint8 codes, elements, ints, doubles
    long part_off;                            // into part: [site block][variant]
    int roots_off, m, m_pad, n_taxa, n_var, nblk;
};
// A workgroup of a batch launch: walk `prog` over 64-site block `block`.
struct NniItem {
    int inst, prog, block, pad;
};
// A group of up to kNniSumVars variants of one batch instance to be totalled
// into out[out0 ..].
struct NniSum {
    int inst, var0, out0, pad;
};
constexpr int kNniSumVars = 8;

struct NniArgs {
    bool f64 = false;
    int C = 1;
    const NniOp* ops = nullptr;
    const int* prog = nullptr;         // program p: ops[prog[p] .. prog[p + 1])
    const uint8_t* tips = nullptr;
    const void* clv = nullptr;
    const int* scl = nullptr;
    const double* P = nullptr;
    const double* roots = nullptr;
    const double* site_w = nullptr;
    double2* part = nullptr;
    // one problem (insts == nullptr) or the items of a batch
    NniInst one{};
    int n_prog = 0;
    const NniInst* insts = nullptr;
    const NniItem* items = nullptr;
    int n_items = 0;
    int max_taxa = 0;                  // largest taxon count of the launch
};

// Edges a walk should hold so that the launch has some 12 workgroups per CU
// (site blocks x walks; 5 are resident): each segment repeats the walk from
// the root to its start, so few segments move less memory (128 taxa x 100,000
// sites: 64 edges a walk 0.538 ms, 32 0.585, 16 0.599; 6 to 18 workgroups
// within 2 %), but a launch of few site blocks needs the segments to fill the
// CUs.  One edge a walk where even those leave a CU at most 16 waves (wide
// states: 8): the launch then takes one chain's time whatever else it repeats.  Kernel us, 6
// edges / 1, 4 categories, 8 taxa x 64 sites 14.2 / 8.7, 120 x 500 (15 waves)
// 27.8 / 17.8, 60 x 2000 (30) 21.2 / 22.9; 1 category, 120 x 2000 (15) 28.7 /
// 19.8; 20 states, 8 x 64 26.9 / 14.4, 28 x 250 (7) 33.9 / 27.4, 28 x 500 (14)
// 33.8 / 35.4.
inline int nni_segment_edges(double edge_blocks, int C, bool wide, int n_cu) {
    n_cu = std::max(1, n_cu);
    if (edge_blocks * C <= (wide ? 8.0 : 16.0) * n_cu) return 1;
    const double per = edge_blocks / (12.0 * n_cu);
    return (int)std::min(64.0, std::max(6.0, per));
}

// Launches the walks (DNA, S <= 4; C = 1, 2, 4 or 8).  Writes one (mantissa
// product, exponent) pair per variant and site block, or the weighted sum of
// logarithms where site_w is set.
hipError_t nni4_launch(const NniArgs& a, hipStream_t st);

// Totals of the variants from those pairs, in a fixed order with
// compensation.  A batch's trees are totalled by the same launch: out[k] = sum
// of tree_part[seg[k] .. seg[k + 1]), k < n_seg.
hipError_t nni_sum_launch(const double2* part, bool weighted, const NniInst* insts, const NniInst& one,
                          const NniSum* sums, int n_sums, const double* tree_part, const int* seg, int n_seg, double* out,
                          hipStream_t st);
