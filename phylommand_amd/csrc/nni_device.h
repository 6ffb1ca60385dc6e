// nni_device.h -- reductions of the NNI walks over a wave's sites.
#pragma once

#include "prune_device.h"

namespace {

// Mark of a held edge whose second variant is not scored.
constexpr int kNniSingle = 1 << 30;

// Product over the wave of doubles in [0.5, 1) or 1 (or 0, NaN), in lane 63,
// by DPP row shifts and row broadcasts (lanes without a source multiply by 1);
// the same for sums of integers.
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_mul(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWS, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0x3ff00000, __double2hiint(v), CTRL, ROWS, 0xf, false);
    return v * __hiloint2double(hi, lo);
}
__device__ __forceinline__ double wave_product(double v) {
    v = dpp_mul<0x111, 0xf>(v);   // row_shr 1, 2, 4, 8
    v = dpp_mul<0x112, 0xf>(v);
    v = dpp_mul<0x114, 0xf>(v);
    v = dpp_mul<0x118, 0xf>(v);
    v = dpp_mul<0x142, 0xa>(v);   // row_bcast 15, 31
    return dpp_mul<0x143, 0xc>(v);
}
__device__ __forceinline__ int wave_add(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);
    return v + __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);
}

// The wave's site likelihoods lc 2^sc as (mantissa product, exponent), in
// lane 63.
__device__ __forceinline__ double2 nni_product(double lc, int sc, bool live) {
    int e = 0;
    double mant = 1.0;
    if (live) {
        mant = frexp(lc, &e);
        e += sc;
        // a negative sum has no logarithm: its sign must not cancel in the product
        if (!(lc >= 0.0)) mant = __builtin_nan("");
    }
    mant = wave_product(mant);
    return make_double2(mant, (double)wave_add(e));
}

// The sum of weighted site log-likelihoods instead.
__device__ __forceinline__ double2 nni_weighted(double lc, int sc, double w, bool live) {
    return make_double2(wave_sum(live ? w * (log(lc) + sc * kLn2) : 0.0), 0.0);
}

}  // namespace
