// nni.hip -- NNI neighbourhoods of DNA problems (S <= 4) by outer partials
// (nni_program.h).
#include "nni.h"

#include "nni_device.h"
#include "prune_device.h"

namespace {

// y = P x and y = P^T x for a 4 x 4 P held in scalar registers
__device__ __forceinline__ void matvec4(const double* __restrict__ P, const double (&x)[4], double (&y)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        double a = 0.0;
#pragma unroll
        for (int j = 0; j < 4; ++j) a = fma(P[i * 4 + j], x[j], a);
        y[i] = a;
    }
}
__device__ __forceinline__ void matvec4t(const double* __restrict__ P, const double (&x)[4], double (&y)[4]) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        double a = 0.0;
#pragma unroll
        for (int i = 0; i < 4; ++i) a = fma(P[i * 4 + j], x[i], a);
        y[j] = a;
    }
}

// One workgroup walks one program over 64 sites, wave c computing rate
// category c (P is wave-uniform: scalar loads).  The variants' category sums
// meet in LDS, EV variants at a time, and wave w finishes variant w of them.
// (One wave finishing all of them, a row of 16 lanes a variant, issues a
// third of the instructions but holds the others at the barrier: 0.615
// against 0.585 ms for 250 variants of 128 taxa x 100,000 sites.)
// The 64 site likelihoods of a block are multiplied rather than their
// logarithms added: mantissas in [0.5, 1) cannot underflow over 64 factors,
// the exponents add up as integers, and the one logarithm per (variant, block)
// is left to the summing kernel (a double logarithm costs more than a
// variant's two products).  With site weights the weighted logarithms are
// added here.
// An edge issues about 220 vector instructions, 108 of them the FP64 products,
// and reads two stored partials; issue (58 % busy) and the reads (1.0 GB of
// partials, re-read once for the siblings) bind together, so five waves a
// SIMD are asked for (FP32 80 registers, FP64 94; four 0.69, five 0.52 ms).
// 250 variants of 128 taxa x 100,000 sites: 0.52 to 0.57 ms, 2.206 ms as one
// path-to-root program a variant.  (The FP64 walk with site weights spills 6 to
// 13 of its 96 registers: a call at 128 x 20,000 takes 0.365 ms, 0.336 without
// weights.)
template <typename T, int C, bool TL, bool BATCH, bool WEIGHTED>
__global__ __launch_bounds__(64 * C, 5) void nni4_kernel(
    const NniOp* __restrict__ ops, const int* __restrict__ prog_begin, const NniInst* __restrict__ insts, NniInst one,
    const NniItem* __restrict__ items, int n_prog, const uint8_t* __restrict__ tips_all, const T* __restrict__ clv_all,
    const int* __restrict__ scl_all, const double* __restrict__ P_all, const double* __restrict__ roots_all,
    const double* __restrict__ site_w, double2* __restrict__ part) {
    constexpr int EV = C == 1 ? 2 : C < 4 ? C : 4, EP = EV / 2;    // variants, edges collected
    __shared__ double xr[C > 1 ? EV : 1][C][64];
    __shared__ int xs[C > 1 ? EP : 1][C][64];        // (both variants of an edge have one scaler)
    __shared__ double2 sv[kNniSaves][C][2][64];
    __shared__ int svs[kNniSaves][C][64];
    __shared__ __align__(16) T tipv[TL ? 64 : 1];      // the four 0/1 state values of each code
    static_assert(__alignof__(tipv) >= 16, "read four values at once (load_raw4)");
    extern __shared__ __align__(16) uint8_t tl[];
    const int lane = threadIdx.x & 63;
    const int cat = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int bx, prog;
    NniInst I;
    if constexpr (BATCH) {
        const NniItem w = items[blockIdx.x];
        I = insts[w.inst];
        bx = w.block;
        prog = w.prog;
    } else {
        // workgroup i runs on XCD i % 8: the walks of a site block follow
        // each other on one XCD and share its stored partials in L2
        I = one;
        const int slot = (int)blockIdx.x >> 3;
        prog = slot % n_prog;
        bx = slot / n_prog * 8 + ((int)blockIdx.x & 7);
        if (bx >= I.nblk) return;
    }
    const int m_pad = I.m_pad, s = bx * 64 + lane;
    const int n_taxa = I.n_taxa;
    // uniform bases and the lane's 32-bit offsets: the loads take a scalar
    // base and need no 64-bit address arithmetic per lane
    const uint8_t* tips = tips_all + I.tips_off;
    const size_t slot_stride = (size_t)C * m_pad;      // sites per partial slot, all categories
    const T* clv = clv_all + I.clv_off + (size_t)cat * m_pad * 4;
    const int* scl = scl_all + I.scl_off + (size_t)cat * m_pad;
    const char* Pcat = reinterpret_cast<const char*>(P_all + I.P_off + (size_t)cat * 16);
    const double* roots = roots_all + I.roots_off;
    if constexpr (TL) {
        if (threadIdx.x < 64) tipv[threadIdx.x] = (T)(threadIdx.x >> 2 >> (threadIdx.x & 3) & 1);
        const uint8_t* blk = tips + (size_t)bx * 64;
        for (int i = threadIdx.x; i < n_taxa * 16; i += 64 * C) {
            const uint32_t w = *reinterpret_cast<const uint32_t*>(blk + (size_t)(i >> 4) * m_pad + 4 * (i & 15));
            reinterpret_cast<uint32_t*>(tl)[i] = w;
        }
        __syncthreads();
    }
    double2* const out = part + I.part_off + (size_t)bx * I.n_var;

    const auto P_of = [&](int node) {
        return reinterpret_cast<const double*>(Pcat + (uint32_t)node * (uint32_t)(C * 128));
    };
    // a node's own partial (tip states, a stored partial) as it lies in memory
    const auto fetch = [&](int node, T (&x)[4], int& sc) {
        sc = 0;
        if (node >= n_taxa) {
            const size_t at = (size_t)(node - n_taxa) * slot_stride;
            load_raw4(clv + at * 4 + (uint32_t)s * 4u, x);
            sc = (scl + at)[(uint32_t)s];
        } else if (node >= 0) {
            if constexpr (TL) {
                load_raw4(tipv + 4 * tl[node * 64 + lane], x);
            } else {
                const unsigned code = (tips + (size_t)node * m_pad)[(uint32_t)s];
#pragma unroll
                for (int j = 0; j < 4; ++j) x[j] = (T)(code >> j & 1u);
            }
        }
    };
    // its factor P x (ones for a missing child)
    const auto factor = [&](int node, const T (&x)[4], double (&y)[4]) {
        if (node >= 0) {
            double v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = (double)x[i];
            matvec4(P_of(node), v, y);
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) y[i] = 1.0;
        }
    };
    const bool live = s < I.m;
    // edges held and their output index (an NNI_ROOT op has one variant)
    int n_held = 0, held_var[EP] = {};
    // site values of one variant from the categories' sums, to out[var]
    const auto finish = [&](double lc, int sc, int var) {
        const double2 r = WEIGHTED ? nni_weighted(lc, sc, live ? site_w[s] : 0.0, live) : nni_product(lc, sc, live);
        if (lane == 63) out[var] = r;
    };
    const auto flush = [&]() {
        if constexpr (C > 1) {
            __syncthreads();
            if (cat < 2 * n_held) {
                const int p = cat >> 1;
                int var = held_var[0];
#pragma unroll
                for (int q = 1; q < EP; ++q) var = p == q ? held_var[q] : var;
                int M = xs[p][0][lane];
#pragma unroll
                for (int c = 1; c < C; ++c) M = max(M, xs[p][c][lane]);
                double lc = 0.0;
#pragma unroll
                for (int c = 0; c < C; ++c) lc += ldexp(xr[cat][c][lane], xs[p][c][lane] - M);
                if (!(var & kNniSingle)) finish(lc, M, var + (cat & 1));
                else if (!(cat & 1)) finish(lc, M, var & ~kNniSingle);
            }
            __syncthreads();
            n_held = 0;
        }
    };
    const auto hold = [&](double l0, double l1, int sc, const NniOp& op) {
        const int q = op.flags & NNI_XY ? 1 : 0;
        if constexpr (C == 1) {
            finish(l0, sc, op.var + q);
            if (!(op.flags & NNI_ROOT)) finish(l1, sc, op.var + 1 - q);
        } else {
            xr[2 * n_held + q][cat][lane] = l0;
            xr[2 * n_held + 1 - q][cat][lane] = l1;
            xs[n_held][cat][lane] = sc;
#pragma unroll
            for (int p = 0; p < EP; ++p)
                if (n_held == p) held_var[p] = op.var | (op.flags & NNI_ROOT ? kNniSingle : 0);
            ++n_held;
        }
    };

    // An op's operands are fetched during the op before it; after a program's
    // last op those of the next program, but in a batch none: it may be
    // another tree's.
    double O[4] = {}, B[4] = {};
    int sO = 0, sB = 0;
    const int k0 = prog_begin[prog], k1 = prog_begin[prog + 1];
    NniOp nx = ops[k0];
    T rx[4] = {}, ry[4] = {};
    int rsx, rsy;
    fetch(nx.x, rx, rsx);
    fetch(nx.y, ry, rsy);
    for (int k = k0; k < k1; ++k) {
        const NniOp op = nx;
        nx = BATCH ? nni_ahead(ops, k, k1) : ops[k + 1];
        double X[4], Y[4];
        factor(op.x, rx, X);
        factor(op.y, ry, Y);
        const int sX = rsx, sY = rsy;
        fetch(nx.x, rx, rsx);
        fetch(nx.y, ry, rsy);
        if (op.flags & NNI_INIT) {
            const double w = roots[kRootCatOff + cat];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                O[i] = roots[i] * w;
                B[i] = Y[i];
            }
            sO = 0;
            sB = sY;
            continue;
        }
        if (op.flags & NNI_POP) {
            const int l = nni_pop_slot(op.flags);
            const double2 a = sv[l][cat][0][lane], b = sv[l][cat][1][lane];
            O[0] = a.x; O[1] = a.y; O[2] = b.x; O[3] = b.y;
            sO = svs[l][cat][lane];
        }
        if (op.flags & NNI_FETCH_S) {
            T z[4] = {};
            fetch(op.s, z, sB);
            factor(op.s, z, B);
        }
        if (op.flags & NNI_SAVE) {
            const int l = nni_save_slot(op.flags);
            sv[l][cat][0][lane] = make_double2(O[0], O[1]);
            sv[l][cat][1][lane] = make_double2(O[2], O[3]);
            svs[l][cat][lane] = sO;
        }
        int sc = sO + sX + sY;
        if (op.flags & NNI_ROOT) {
            // in the pair's terms below: S = the factor of c, X = P_s (X x D)
            T z[4] = {};
            double f[4];
            int sD;
            fetch(op.d, z, sD);
            factor(op.d, z, f);
            sc += sD;
#pragma unroll
            for (int i = 0; i < 4; ++i) f[i] *= X[i];
            matvec4(P_of(op.s), f, X);
            fetch(op.c, z, sB);
            factor(op.c, z, B);
        }
        const double* Pv = P_of(op.v);
        if (op.flags & (NNI_PAIR | NNI_ROOT)) {
            double x[4], u[4], l0 = 0.0, l1 = 0.0;
#pragma unroll
            for (int i = 0; i < 4; ++i) x[i] = B[i] * Y[i];
            matvec4(Pv, x, u);
#pragma unroll
            for (int i = 0; i < 4; ++i) l0 = fma(O[i] * X[i], u[i], l0);
#pragma unroll
            for (int i = 0; i < 4; ++i) x[i] = B[i] * X[i];
            matvec4(Pv, x, u);
#pragma unroll
            for (int i = 0; i < 4; ++i) l1 = fma(O[i] * Y[i], u[i], l1);
            hold(l0, l1, sc + sB, op);
        }
        if (op.flags & NNI_DESC) {
            double x[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) x[i] = O[i] * B[i];
            matvec4t(Pv, x, O);
            sO += sB;
            if (max_hi_word(O) < kLazyRescaleHi) {
                const int e = max_exponent(O);
                sO += e;
#pragma unroll
                for (int i = 0; i < 4; ++i) O[i] = ldexp(O[i], -e);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) B[i] = Y[i];
            sB = sY;
        }
        // (only O and B are live across a group's reductions)
        if (C > 1 && n_held == EP) flush();
    }
    if (C > 1 && n_held) flush();    // (uniform per workgroup)
}

// total = sum over site blocks of log(mantissa product) + exponent ln 2 (or
// of the weighted sums): 256 / W slices of a variant's blocks, W variants side by
// side; Kahan within a slice, then two-sums over the slices in a fixed order
// (infinite values as in block_total).
// Bound by a slice's chain of loads and logarithms where there are few
// workgroups (250 variants x 1564 blocks: W = 8 30 us, 4 17, 2 10.9; 74 x 640:
// 6.8, 5.0, 3.8), by the width of its loads (16 W bytes) where there are many
// (5200 variants of 24 alignments: 8.4, 9.1, 11.1).  A batch's tree totals come
// along (their own launch added 5 to 8 us to every run, most of it the gap).
template <int W>
__global__ __launch_bounds__(256) void nni_sum_kernel(const double2* __restrict__ part, int weighted,
                                                      const NniInst* __restrict__ insts, NniInst one,
                                                      const NniSum* __restrict__ sums, int n_sums,
                                                      const double* __restrict__ tree_part, const int* __restrict__ seg,
                                                      double* __restrict__ out) {
    constexpr int SL = 256 / W;
    static_assert(64 % W == 0, "a wave holds whole slices");
    if ((int)blockIdx.x >= n_sums) {      // a batch's trees, after the variants
        const int k = (int)blockIdx.x - n_sums;
        const double t = block_total(tree_part + seg[k], seg[k + 1] - seg[k]);
        if (threadIdx.x == 0) out[k] = t;
        return;
    }
    __shared__ double hi[4][W], lo[4][W];
    NniSum g{0, (int)blockIdx.x * W, (int)blockIdx.x * W, 0};
    NniInst I = one;
    if (sums) {
        g = sums[blockIdx.x];
        I = insts[g.inst];
    }
    const int w = threadIdx.x % W, sl = threadIdx.x / W, var = g.var0 + w;
    const double2* p = part + I.part_off + var;
    const int nblk = var < I.n_var ? I.nblk : 0;
    const auto value = [&](double2 v) { return weighted ? v.x : log(v.x) + v.y * kLn2; };
    double s = 0.0, comp = 0.0;
    for (int b0 = sl; b0 < nblk; b0 += 4 * SL) {
        double2 v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int b = b0 + u * SL;
            v[u] = b < nblk ? p[(size_t)b * I.n_var] : make_double2(weighted ? 0.0 : 1.0, 0.0);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const double x = value(v[u]) - comp;
            const double t = s + x;
            comp = (t - s) - x;
            s = t;
        }
    }
    double h = s, l = -comp;
#pragma unroll
    for (int o = W; o < 64; o <<= 1) two_sum_add(h, l, __shfl_xor(h, o, 64), __shfl_xor(l, o, 64));
    if (__any(!(h + l == h + l))) {
        double q = 0.0;
        for (int b = sl; b < nblk; b += SL) q += value(p[(size_t)b * I.n_var]);
#pragma unroll
        for (int o = W; o < 64; o <<= 1) q += __shfl_xor(q, o, 64);
        if (!(h + l == h + l)) {
            h = q;
            l = 0.0;
        }
    }
    if ((threadIdx.x & 63) < W) {
        hi[threadIdx.x >> 6][w] = h;
        lo[threadIdx.x >> 6][w] = l;
    }
    __syncthreads();
    if (threadIdx.x < W && var < I.n_var) {
        for (int q = 1; q < 4; ++q) two_sum_add(h, l, hi[q][w], lo[q][w]);
        const double t = h + l;
        out[g.out0 + w] = t == t ? t : (hi[0][w] + hi[1][w]) + (hi[2][w] + hi[3][w]);
    }
}

template <typename T, int C, bool TL, bool BATCH, bool W>
void launch_k(const NniArgs& a, hipStream_t st) {
    const dim3 grid(BATCH ? a.n_items : (a.one.nblk + 7) / 8 * 8 * a.n_prog);
    hipLaunchKernelGGL((nni4_kernel<T, C, TL, BATCH, W>), grid, dim3(64 * C), TL ? tip_lds_bytes(a.max_taxa) : 0, st,
                       a.ops, a.prog, a.insts, a.one, a.items, a.n_prog, a.tips, static_cast<const T*>(a.clv), a.scl,
                       a.P, a.roots, a.site_w, a.part);
}

template <typename T, int C>
void launch_c(const NniArgs& a, hipStream_t st) {
    const bool tl = a.max_taxa <= kTipLdsTaxa;
    if (a.items) tl ? launch_k<T, C, true, true, false>(a, st) : launch_k<T, C, false, true, false>(a, st);
    else if (a.site_w) tl ? launch_k<T, C, true, false, true>(a, st) : launch_k<T, C, false, false, true>(a, st);
    else tl ? launch_k<T, C, true, false, false>(a, st) : launch_k<T, C, false, false, false>(a, st);
}

template <typename T>
void launch_t(const NniArgs& a, hipStream_t st) {
    switch (a.C) {
    case 1: launch_c<T, 1>(a, st); break;
    case 2: launch_c<T, 2>(a, st); break;
    case 4: launch_c<T, 4>(a, st); break;
    default: launch_c<T, 8>(a, st); break;
    }
}

}  // namespace

hipError_t nni4_launch(const NniArgs& a, hipStream_t st) {
    if (a.f64) launch_t<double>(a, st);
    else launch_t<float>(a, st);
    return hipGetLastError();
}

hipError_t nni_sum_launch(const double2* part, bool weighted, const NniInst* insts, const NniInst& one,
                          const NniSum* sums, int n_sums, const double* tree_part, const int* seg, int n_seg, double* out,
                          hipStream_t st) {
    static_assert(kSumThreads == 256, "trees and variants by the same workgroups");
    const auto launch = [&](auto* kernel, int n) {
        hipLaunchKernelGGL(kernel, dim3(n + n_seg), dim3(256), 0, st, part, weighted ? 1 : 0, insts, one, sums, n, tree_part,
                           seg, out);
    };
    // one neighbourhood: narrow groups until they alone fill the chip
    if (sums || n_seg) launch(nni_sum_kernel<kNniSumVars>, n_sums);
    else if (one.n_var <= 1024) launch(nni_sum_kernel<2>, (one.n_var + 1) / 2);
    else launch(nni_sum_kernel<kNniSumVars>, (one.n_var + kNniSumVars - 1) / kNniSumVars);
    return hipGetLastError();
}
