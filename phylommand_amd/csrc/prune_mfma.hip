// prune_mfma.hip -- the pruning walker for alphabets wider than 4 states
// (prune_mfma.h).
#include "prune_mfma.h"

#include "nni.h"
#include "nni_device.h"
#include "prune_device.h"

namespace {

// ---------------------------------------------------------------------------
// Wide-state walker on the matrix cores (4 < S <= 32, FP64 arithmetic).
//
// One wave = G groups of 16 sites x one rate category; a workgroup holds the
// C category waves of the same G site groups.  Each child product is a GEMM
//     out[state row][site] = sum_k P[row][k] * L[k][site]
// done as v_mfma_f64_16x16x4f64 steps (A = P: 16 rows x 4 k, B = L: 4 k x 16
// sites, D = 16 rows x 16 sites; D[i][j] sits in lane j + 16 (i % 4),
// register i / 4).  Lane l serves site l % 16 and lane group g = l / 16; slot
// t of a lane holds state 4t + g, and row i of tile T is state 16T + i, so an
// MFMA result (tile T, register r) is slot 4T + r of the next op's operand
// with no shuffles.  V = ceil(S / 4) slots cover the S states; tile 1 exists
// for S > 16 (for 17..20 states as v_mfma_f64_4x4x4f64 blocks, see
// pwide_kernel).  Partials are stored as [slot][cat][site group][V][64 lanes]
// (every load and store a full row), P as [node][cat][tile][V][64] doubles
// (pwide_kernel).  FP64 matrix cores rather than FP32 ones: the FP32 MFMA
// dot products truncate small addends (about -0.1 ulp per 5-step chain on
// transition-matrix-shaped operands), which biases every site the same way.
// Scalers as in the DNA walker: one int32 power of two per (node, category,
// site), the categories meeting only at the root.
// ---------------------------------------------------------------------------

typedef double mfma_d4 __attribute__((ext_vector_type(4)));

// The P matrices of one (node, category) a workgroup, in every form the walkers
// read, from one pass: P itself, the matrix-core operands, the tip columns.
//
// P[i][j] = sum_k V[i][k] exp(lam_k r_c t_node) Vinv[k][j], the exponentials
// taken once (eff set), or P as it lies in memory (eff null: built on the host).
//
// Pm[node][cat][T][t][lane] = P[16T + lane % 16][4t + lane / 16] (0 outside S),
// the A operand of v_mfma_f64_16x16x4f64 for row tile T and K-step t.  With
// V = 5 (17..20 states) tile 1 holds only rows 16..19 and is instead the A
// operand of v_mfma_f64_4x4x4f64 (four 4x4 blocks, one per 4 sites): lane l
// = 4b + 16k + i holds P[16 + i][4t + k] for every block b.  That product
// lands as D[lane j + 16 i] = row 16 + i of site j, the operand slot of
// states 16..19, with no padded rows.  PmT (where set): the same of P's
// transpose.
//
// PTm[node][cat][k][i] = P[i][k] for k < S, PTm[..][S][i] = sum_q P[i][q]
// (the product with an all-states tip), i < 4V (0 for i >= S): the columns a
// single-state or all-states tip selects.
//
// Bound by the chain exp -> V exp -> S fma -> layouts and the launch, not by its
// few MB of stores: 7.2 us for the 127 nodes and 4 categories of a 64-taxon
// 20-state tree.  As three launches, each entry of P with its own S
// exponentials, the same took 18 us and two more gaps.
__global__ __launch_bounds__(256) void pwide_kernel(const double* __restrict__ eig_V, const double* __restrict__ eig_Vinv,
                                                    const double* __restrict__ lam, const double* __restrict__ eff,
                                                    const PRates rates, const RootWeights roots, int S, int Sp, int C,
                                                    int V, int TN, double* P, double* __restrict__ Pm,
                                                    double* __restrict__ PmT, double* __restrict__ PTm,
                                                    double* __restrict__ d_roots) {
    __shared__ double ex[32], ve[32 * 32], vi[32 * 32], p[32][33];
    const int mat = blockIdx.x, c = mat % C, node = mat / C;      // node * C + cat
    const int tid = threadIdx.x;
    double* Pg = P + (size_t)mat * Sp * Sp;
    if (mat == 0 && tid < kRootDoubles) d_roots[tid] = roots.v[tid];
    if (eff) {
        const double t = eff[node] * rates.v[c];
        if (tid < S) ex[tid] = exp(lam[tid] * t);
        __syncthreads();
        for (int i = tid; i < S * S; i += 256) {
            ve[i] = eig_V[i] * ex[i % S];
            vi[i] = eig_Vinv[i];
        }
        __syncthreads();
        for (int e = tid; e < Sp * Sp; e += 256) {
            const int i = e / Sp, j = e % Sp;
            double v = 0.0;
            if (i < S && j < S)
                for (int k = 0; k < S; ++k) v = fma(ve[i * S + k], vi[k * S + j], v);
            p[i][j] = v;
            Pg[e] = v;
        }
    } else {
        for (int e = tid; e < Sp * Sp; e += 256) p[e / Sp][e % Sp] = Pg[e];
    }
    __syncthreads();
    double* pm = Pm + (size_t)mat * TN * V * 64;
    double* pmt = PmT ? PmT + (size_t)mat * TN * V * 64 : nullptr;
    for (int e = tid; e < TN * V * 64; e += 256) {
        const int l = e % 64, t = e / 64 % V, T = e / (64 * V);
        const bool short_tile = V == 5 && T == 1;
        const int row = 16 * T + (short_tile ? l % 4 : l % 16), col = 4 * t + l / 16;
        const bool in = row < S && col < S;
        pm[e] = in ? p[row][col] : 0.0;
        if (pmt) pmt[e] = in ? p[col][row] : 0.0;
    }
    const int W = 4 * V;
    double* pt = PTm + (size_t)mat * (S + 1) * W;
    for (int e = tid; e < (S + 1) * W; e += 256) {
        const int i = e % W, k = e / W;
        double v = 0.0;
        if (i < S) {
            if (k < S) v = p[i][k];
            else
                for (int q = 0; q < S; ++q) v += p[i][q];
        }
        pt[e] = v;
    }
}

__device__ inline double to_d(float x) { return (double)x; }
__device__ inline double to_d(double x) { return x; }

// Largest state value of a site in the matrix walker's layout (states 4t + g
// in slot t of lane group g, so the maximum runs over the slots and then the
// four lane groups: lanes l ^ 16, l ^ 32), and its frexp exponent (0 when no
// state is positive).  Every lane of the wave must take part.
template <int V>
__device__ inline double site_max(const double (&v)[V]) {
    double mx = 0.0;
#pragma unroll
    for (int t = 0; t < V; ++t) mx = fmax(mx, v[t]);
    mx = fmax(mx, __shfl_xor(mx, 16, 64));
    return fmax(mx, __shfl_xor(mx, 32, 64));
}
template <int V>
__device__ inline int site_exponent(const double (&v)[V]) {
    const double mx = site_max<V>(v);
    int e = 0;
    if (mx > 0.0) (void)frexp(mx, &e);
    return e;
}

// One child for the G site groups of a wave: acc[q][T] = P . x for tile T,
// x in operand order.  The P operand of each K-step is loaded once and used by
// every group.
template <typename T, int C, int V, int G, bool TL>
__device__ inline void mfma_child(int kind, int idx, int node, int cat, const int (&s)[G], int sg0, int n_sg,
                                  int lane, int g, int m_pad, int S, uint32_t full,
                                  const uint32_t* __restrict__ tips, const uint32_t* tl, const T* clv,
                                  size_t slot_stride,
                                  const int* scl, const double* __restrict__ Pm, const double* __restrict__ PTm,
                                  const double (&cA)[G][V], const int (&sA)[G], const double* cB,
                                  const int (&sB)[G], mfma_d4 (&acc)[G][2], int (&sc)[G]) {
    constexpr int TN = V > 4 ? 2 : 1;
    double x[G][V];
    if (kind == SRC_TIP) {
        uint32_t mk[G];
        bool simple = true;
#pragma unroll
        for (int q = 0; q < G; ++q) {
            mk[q] = TL ? tl[idx * 16 * G + 16 * q + (lane & 15)] : tips[(size_t)idx * m_pad + s[q]];
            simple = simple && (mk[q] == full || __popc(mk[q]) == 1);
        }
        // a wave whose sites are all single states or gaps selects columns of P
        if (__all(simple)) {
            const double* base = PTm + ((size_t)node * C + cat) * (S + 1) * (4 * V) + g;
#pragma unroll
            for (int q = 0; q < G; ++q) {
                const int col = mk[q] == full ? S : __ffs(mk[q]) - 1;
                const double* pt = base + (size_t)col * (4 * V);
#pragma unroll
                for (int t = 0; t < V; ++t) acc[q][t / 4][t % 4] = pt[4 * t];
            }
            return;
        }
#pragma unroll
        for (int q = 0; q < G; ++q)
#pragma unroll
            for (int t = 0; t < V; ++t) x[q][t] = (mk[q] >> (4 * t + g)) & 1u ? 1.0 : 0.0;
    } else if (kind == SRC_CLV) {
#pragma unroll
        for (int q = 0; q < G; ++q) {
            const T* src = clv + (size_t)idx * slot_stride + ((size_t)cat * n_sg + sg0 + q) * V * 64 + lane;
#pragma unroll
            for (int t = 0; t < V; ++t) x[q][t] = to_d(src[t * 64]);
            sc[q] += scl[((size_t)idx * C + cat) * m_pad + s[q]];
        }
    } else if (kind == SRC_CARRY_A) {
#pragma unroll
        for (int q = 0; q < G; ++q) {
#pragma unroll
            for (int t = 0; t < V; ++t) x[q][t] = to_d(cA[q][t]);
            sc[q] += sA[q];
        }
    } else {
#pragma unroll
        for (int q = 0; q < G; ++q) {
#pragma unroll
            for (int t = 0; t < V; ++t) x[q][t] = cB[(q * V + t) * 64];
            sc[q] += sB[q];
        }
    }
    const double* pm = Pm + ((size_t)node * C + cat) * TN * V * 64 + lane;
#pragma unroll
    for (int T2 = 0; T2 < TN; ++T2) {
#pragma unroll
        for (int q = 0; q < G; ++q) acc[q][T2] = mfma_d4{0.0, 0.0, 0.0, 0.0};
        if (V == 5 && T2 == 1) {
            // states 16..19: four 4x4x4 blocks give exactly the 4 rows
            double d[G];
#pragma unroll
            for (int q = 0; q < G; ++q) d[q] = 0.0;
#pragma unroll
            for (int t = 0; t < V; ++t) {
                const double a = pm[(V + t) * 64];
#pragma unroll
                for (int q = 0; q < G; ++q) d[q] = __builtin_amdgcn_mfma_f64_4x4x4f64(a, x[q][t], d[q], 0, 0, 0);
            }
#pragma unroll
            for (int q = 0; q < G; ++q) acc[q][1][0] = d[q];
            continue;
        }
#pragma unroll
        for (int t = 0; t < V; ++t) {
            const double a = pm[(T2 * V + t) * 64];
#pragma unroll
            for (int q = 0; q < G; ++q)
                acc[q][T2] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, x[q][t], acc[q][T2], 0, 0, 0);
        }
    }
}

// The P operand of one child for every row tile and K-step (Pm order: tile
// T, K-step t at register T V + t).
template <int C, int V>
__device__ __forceinline__ void load_pm(int node, int cat, int lane, const double* __restrict__ Pm,
                                        double (&pf)[(V > 4 ? 2 : 1) * V]) {
    constexpr int TN = V > 4 ? 2 : 1;
    const double* pm = Pm + ((size_t)node * C + cat) * TN * V * 64 + lane;
#pragma unroll
    for (int i = 0; i < TN * V; ++i) pf[i] = pm[i * 64];
}

// r = P . x for the G site groups with the P operand in registers: the same
// matrix instructions in the same order as mfma_child; r[q][t] is state
// 4t + g of group q's site.
template <int V, int G>
__device__ __forceinline__ void mfma_products(const double (&pf)[(V > 4 ? 2 : 1) * V], const double (&x)[G][V],
                                              double (&r)[G][V]) {
    constexpr int TN = V > 4 ? 2 : 1;
    mfma_d4 acc[G][2];
#pragma unroll
    for (int T2 = 0; T2 < TN; ++T2) {
        if (V == 5 && T2 == 1) {
            double d[G];
#pragma unroll
            for (int q = 0; q < G; ++q) d[q] = 0.0;
#pragma unroll
            for (int t = 0; t < V; ++t)
#pragma unroll
                for (int q = 0; q < G; ++q) d[q] = __builtin_amdgcn_mfma_f64_4x4x4f64(pf[V + t], x[q][t], d[q], 0, 0, 0);
#pragma unroll
            for (int q = 0; q < G; ++q) acc[q][1][0] = d[q];
            continue;
        }
#pragma unroll
        for (int q = 0; q < G; ++q) acc[q][T2] = mfma_d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int t = 0; t < V; ++t)
#pragma unroll
            for (int q = 0; q < G; ++q)
                acc[q][T2] = __builtin_amdgcn_mfma_f64_16x16x4f64(pf[T2 * V + t], x[q][t], acc[q][T2], 0, 0, 0);
    }
#pragma unroll
    for (int q = 0; q < G; ++q)
#pragma unroll
        for (int t = 0; t < V; ++t) r[q][t] = acc[q][t / 4][t % 4];
}

// A tip child's state masks for the G site groups, and whether every site of
// the wave is a single state or a gap (then the child's factor is a column
// of P).
template <int G, bool TL>
__device__ __forceinline__ bool tip_masks(int idx, const int (&s)[G], int lane, int m_pad, uint32_t full,
                                          const uint32_t* __restrict__ tips, const uint32_t* tl, uint32_t (&mk)[G]) {
    bool simple = true;
#pragma unroll
    for (int q = 0; q < G; ++q) {
        mk[q] = TL ? tl[idx * 16 * G + 16 * q + (lane & 15)] : tips[(size_t)idx * m_pad + s[q]];
        simple = simple && (mk[q] == full || __popc(mk[q]) == 1);
    }
    return __all(simple);
}

// One child's factor in a shape-specialised op: a tip's P columns (col) or
// products with its state indicators, a stored or carried partial's products.
template <int K, typename T, int C, int V, int G>
__device__ __forceinline__ void mfma_factor(bool col, const double (&cols)[G][V], const uint32_t (&mk)[G], int node,
                                            int cat, int lane, int g, const double* __restrict__ Pm,
                                            const double (&pf)[(V > 4 ? 2 : 1) * V], const T (&xr)[G][V],
                                            const double (&cA)[G][V], const double* cB, double (&r)[G][V]) {
    if constexpr (K == SRC_TIP) {
        if (col) {
#pragma unroll
            for (int q = 0; q < G; ++q)
#pragma unroll
                for (int t = 0; t < V; ++t) r[q][t] = cols[q][t];
            return;
        }
        double pt[(V > 4 ? 2 : 1) * V], x[G][V];
        load_pm<C, V>(node, cat, lane, Pm, pt);
#pragma unroll
        for (int q = 0; q < G; ++q)
#pragma unroll
            for (int t = 0; t < V; ++t) x[q][t] = (mk[q] >> (4 * t + g)) & 1u ? 1.0 : 0.0;
        mfma_products<V, G>(pt, x, r);
    } else if constexpr (K == SRC_CLV) {
        double x[G][V];
#pragma unroll
        for (int q = 0; q < G; ++q)
#pragma unroll
            for (int t = 0; t < V; ++t) x[q][t] = to_d(xr[q][t]);
        mfma_products<V, G>(pf, x, r);
    } else if constexpr (K == SRC_CARRY_A) {
        mfma_products<V, G>(pf, cA, r);
    } else {
        double x[G][V];
#pragma unroll
        for (int q = 0; q < G; ++q)
#pragma unroll
            for (int t = 0; t < V; ++t) x[q][t] = cB[(q * V + t) * 64];
        mfma_products<V, G>(pf, x, r);
    }
}

// An op of child shape (LK, RK) (kind order, RK != SRC_NONE): the tip masks
// are read first, then every load of the op (P operands, stored partials and
// their scalers, tip columns) is issued before the first product, so the two
// children's memory latencies overlap.  val = left factor x right factor and
// sc = the children's scalers, as the generic op computes them.
template <int LK, int RK, typename T, int C, int V, int G, bool TL>
__device__ __forceinline__ void mfma_shape(const Op& op, int cat, const int (&s)[G], int sg0, int n_sg, int lane,
                                           int g, int m_pad, int S, uint32_t full, const uint32_t* __restrict__ tips,
                                           const uint32_t* tl, const T* clv, size_t slot_stride, const int* scl,
                                           const double* __restrict__ Pm, const double* __restrict__ PTm,
                                           const double (&cA)[G][V], const int (&sA)[G], const double* cB,
                                           const int (&sB)[G], double (&val)[G][V], int (&sc)[G]) {
    constexpr int TNV = (V > 4 ? 2 : 1) * V;
    uint32_t mkL[G], mkR[G];
    bool colL = false, colR = false;
    if constexpr (LK == SRC_TIP) colL = tip_masks<G, TL>(op.l_idx, s, lane, m_pad, full, tips, tl, mkL);
    if constexpr (RK == SRC_TIP) colR = tip_masks<G, TL>(op.r_idx, s, lane, m_pad, full, tips, tl, mkR);
    double pL[TNV], pR[TNV];
    if constexpr (LK != SRC_TIP) load_pm<C, V>(op.l_node, cat, lane, Pm, pL);
    T xL[G][V], xR[G][V];
    const auto load_stored = [&](int idx, T (&xr)[G][V]) {
#pragma unroll
        for (int q = 0; q < G; ++q) {
            const T* src = clv + (size_t)idx * slot_stride + ((size_t)cat * n_sg + sg0 + q) * V * 64 + lane;
#pragma unroll
            for (int t = 0; t < V; ++t) xr[q][t] = src[t * 64];
            sc[q] += scl[((size_t)idx * C + cat) * m_pad + s[q]];
        }
    };
    if constexpr (LK == SRC_CLV) load_stored(op.l_idx, xL);
    if constexpr (RK == SRC_CLV) load_stored(op.r_idx, xR);
    double gL[G][V], gR[G][V];
    const auto tip_columns = [&](int node, const uint32_t (&mk)[G], double (&cols)[G][V]) {
        const double* base = PTm + ((size_t)node * C + cat) * (S + 1) * (4 * V) + g;
#pragma unroll
        for (int q = 0; q < G; ++q) {
            const int col = mk[q] == full ? S : __ffs(mk[q]) - 1;
            const double* pt = base + (size_t)col * (4 * V);
#pragma unroll
            for (int t = 0; t < V; ++t) cols[q][t] = pt[4 * t];
        }
    };
    if constexpr (LK == SRC_TIP)
        if (colL) tip_columns(op.l_node, mkL, gL);
    if constexpr (RK == SRC_TIP)
        if (colR) tip_columns(op.r_node, mkR, gR);
#pragma unroll
    for (int q = 0; q < G; ++q) {
        if constexpr (LK == SRC_CARRY_A || RK == SRC_CARRY_A) sc[q] += sA[q];
        if constexpr (LK == SRC_CARRY_B || RK == SRC_CARRY_B) sc[q] += sB[q];
    }
    mfma_factor<LK, T, C, V, G>(colL, gL, mkL, op.l_node, cat, lane, g, Pm, pL, xL, cA, cB, val);
    if constexpr (RK != SRC_TIP) load_pm<C, V>(op.r_node, cat, lane, Pm, pR);
    double r[G][V];
    mfma_factor<RK, T, C, V, G>(colR, gR, mkR, op.r_node, cat, lane, g, Pm, pR, xR, cA, cB, r);
#pragma unroll
    for (int q = 0; q < G; ++q)
#pragma unroll
        for (int t = 0; t < V; ++t) val[q][t] *= r[q][t];
}

// grid = (m_pad / (16 G), n_programs), block = 64 * C: wave c computes
// category c of the G 16-site groups starting at group G * x of site block
// x (blockIdx.x in a plain launch; the tail-split mapping of prune4_kernel
// otherwise).
// TL (n_taxa <= kMfmaTipLdsTaxa): the workgroup first copies the tip masks of
// its 16 G sites into LDS (tl[16 G t + site]).
template <typename T, int C, int V, int G, bool TL>
__global__ __launch_bounds__(64 * C, (V <= 5 ? 3 : 1)) void prune_mfma_kernel(
    const Op* __restrict__ ops, const int* __restrict__ prog_begin, const uint32_t* __restrict__ tips, T* clv,
    int* scl, const double* __restrict__ Pm, const double* __restrict__ PTm, const double* __restrict__ roots,
    const double* __restrict__ site_w, double* __restrict__ site_lnl, double* __restrict__ partial, int m, int m_pad,
    int S, uint32_t full, int n_taxa, int n_main, int prog_main, int blk0, int prog_piece, int tail0, int n_tail,
    unsigned* fold_counter, double* fold_out) {
    __shared__ int xsc[C][16 * G];
    __shared__ double xroot[C][16 * G];
    __shared__ uint32_t tl[TL ? kMfmaTipLdsTaxa * 16 * G : 1];
    __shared__ double xb[C][G * V * 64];    // each wave's carry B (LDS keeps the registers for the products)
    // work mapping as in prune4_kernel (plain or tail-split launch)
    const int y = blockIdx.y;
    int bx = blockIdx.x, prog = y;
    bool has_root = true;
    if (prog_main >= 0) {
        if ((int)blockIdx.x < n_main) {
            bx = blk0 + (int)blockIdx.x;
            prog = prog_main;
        } else {
            const int r = (int)blockIdx.x - n_main;
            bx = tail0 + r % n_tail;
            prog = prog_piece + r / n_tail;
            has_root = false;
        }
    }
    if (TL) {
        const uint32_t* blk = tips + (size_t)bx * 16 * G;
        for (int i = threadIdx.x; i < n_taxa * 16 * G; i += 64 * C)
            tl[i] = blk[(size_t)(i / (16 * G)) * m_pad + i % (16 * G)];
        __syncthreads();
    }
    const int lane = threadIdx.x & 63;
    const int g = lane >> 4, j = lane & 15;
    const int cat = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int sg0 = bx * G, n_sg = m_pad >> 4;
    int s[G];
#pragma unroll
    for (int q = 0; q < G; ++q) s[q] = (sg0 + q) * 16 + j;
    const int k0 = prog_begin[prog], k1 = prog_begin[prog + 1];
    const size_t slot_stride = (size_t)C * m_pad * 4 * V;
    // carried results stay in FP64 and are rescaled lazily, as in the DNA
    // walker; only stored partials are rounded to T
    double cA[G][V];
    int sA[G], sB[G];
    double* const cB = &xb[cat][lane];      // carry B: (group q, slot t) at cB[64 (q V + t)]
#pragma unroll
    for (int q = 0; q < G; ++q) {
#pragma unroll
        for (int t = 0; t < V; ++t) { cA[q][t] = 0.0; cB[(q * V + t) * 64] = 0.0; }
        sA[q] = 0;
        sB[q] = 0;
    }
    double lnl[G];
#pragma unroll
    for (int q = 0; q < G; ++q) lnl[q] = 0.0;
    Op nxt = ops[k0];
    for (int k = k0; k < k1; ++k) {
        const Op op = nxt;
        nxt = ops[k + 1];     // in flight during this op (an op buffer ends with one pad op)
        int sc[G];
#pragma unroll
        for (int q = 0; q < G; ++q) sc[q] = 0;
        double val[G][V];
#define PHYLO_MFMA_SHAPE(LK, RK)                                                                                     \
    mfma_shape<LK, RK, T, C, V, G, TL>(op, cat, s, sg0, n_sg, lane, g, m_pad, S, full, tips, tl, clv, slot_stride, \
                                       scl, Pm, PTm, cA, sA, cB, sB, val, sc)
        if (op.flags & OP_SH_AT) PHYLO_MFMA_SHAPE(SRC_CARRY_A, SRC_TIP);
        else if (op.flags & OP_SH_TT) PHYLO_MFMA_SHAPE(SRC_TIP, SRC_TIP);
        else if (op.flags & OP_SH_AB) PHYLO_MFMA_SHAPE(SRC_CARRY_A, SRC_CARRY_B);
        else if (op.flags & OP_SH_AC) PHYLO_MFMA_SHAPE(SRC_CARRY_A, SRC_CLV);
        else {
#undef PHYLO_MFMA_SHAPE
            // the other shapes: one child at a time, kinds read at run time
            mfma_d4 acc[G][2];
            mfma_child<T, C, V, G, TL>(op.l_kind, op.l_idx, op.l_node, cat, s, sg0, n_sg, lane, g, m_pad, S, full,
                                       tips, tl, clv, slot_stride, scl, Pm, PTm, cA, sA, cB, sB, acc, sc);
#pragma unroll
            for (int q = 0; q < G; ++q)
#pragma unroll
                for (int t = 0; t < V; ++t) val[q][t] = acc[q][t / 4][t % 4];
            if (op.r_kind != SRC_NONE) {
                mfma_child<T, C, V, G, TL>(op.r_kind, op.r_idx, op.r_node, cat, s, sg0, n_sg, lane, g, m_pad, S,
                                           full, tips, tl, clv, slot_stride, scl, Pm, PTm, cA, sA, cB, sB, acc, sc);
#pragma unroll
                for (int q = 0; q < G; ++q)
#pragma unroll
                    for (int t = 0; t < V; ++t) val[q][t] *= acc[q][t / 4][t % 4];
            }
        }
        // Lazy rescale: only when a site's largest state falls below 2^-256
        // (a site's states are spread over the lane groups, so its maximum
        // takes two cross-lane steps; every lane holding part of such a site
        // has its own largest state below the threshold, so those steps run
        // only when some lane of the wave has).
        bool low = false;
#pragma unroll
        for (int q = 0; q < G; ++q) {
            int h = __double2hiint(val[q][0]);     // the lane's largest state of the site, as a high word
#pragma unroll
            for (int t = 1; t < V; ++t) h = max(h, __double2hiint(val[q][t]));
            low |= h < kLazyRescaleHi;
        }
        if (__builtin_amdgcn_ballot_w64(low) != 0) {
#pragma unroll
            for (int q = 0; q < G; ++q) {
                const int e = site_exponent<V>(val[q]);
                const double mx = site_max<V>(val[q]);
                if (mx < 0x1p-256) {
                    sc[q] += e;
#pragma unroll
                    for (int t = 0; t < V; ++t) val[q][t] = ldexp(val[q][t], -e);
                }
            }
        }
#pragma unroll
        for (int q = 0; q < G; ++q) {
            if (op.out_slot >= 0) {
                // stored: brought to [0.5, 1) with its own scaler, then rounded
                // to T with per-state random bits
                const int e = site_exponent<V>(val[q]);
                const uint32_t key = round_key(s[q], op, cat) + 0x9e3779b9u * (8u * (uint32_t)g);
                T* dst = clv + (size_t)op.out_slot * slot_stride + ((size_t)cat * n_sg + sg0 + q) * V * 64 + lane;
#pragma unroll
                for (int t = 0; t < V; ++t)
                    dst[t * 64] = (T)round_cut(ldexp(val[q][t], -e), key + 0x9e3779b9u * t, T());
                if (g == 0) scl[((size_t)op.out_slot * C + cat) * m_pad + s[q]] = sc[q] + e;
            }
            if (op.flags & OP_TO_B) {
#pragma unroll
                for (int t = 0; t < V; ++t) cB[(q * V + t) * 64] = val[q][t];
                sB[q] = sc[q];
            } else {
#pragma unroll
                for (int t = 0; t < V; ++t) cA[q][t] = val[q][t];
                sA[q] = sc[q];
            }
        }
        if (op.flags & OP_ROOT) {
            double lc[G];
#pragma unroll
            for (int q = 0; q < G; ++q) {
                // the root partial brought to [0.5, 1) first (as in walk4)
                const int e = site_exponent<V>(val[q]);
                sc[q] += e;
#pragma unroll
                for (int t = 0; t < V; ++t) val[q][t] = ldexp(val[q][t], -e);
                lc[q] = 0.0;
#pragma unroll
                for (int t = 0; t < V; ++t) lc[q] = fma(roots[4 * t + g], val[q][t], lc[q]);
                lc[q] += __shfl_xor(lc[q], 16, 64);
                lc[q] += __shfl_xor(lc[q], 32, 64);
                lc[q] *= roots[kRootCatOff + cat];
            }
            if (C > 1) {
                // the categories' sums at their largest exponent
                if (g == 0) {
#pragma unroll
                    for (int q = 0; q < G; ++q) {
                        xroot[cat][16 * q + j] = lc[q];
                        xsc[cat][16 * q + j] = sc[q];
                    }
                }
                __syncthreads();
#pragma unroll
                for (int q = 0; q < G; ++q) {
                    int M = xsc[0][16 * q + j];
#pragma unroll
                    for (int c = 1; c < C; ++c) M = max(M, xsc[c][16 * q + j]);
                    lc[q] = 0.0;
#pragma unroll
                    for (int c = 0; c < C; ++c) lc[q] += ldexp(xroot[c][16 * q + j], xsc[c][16 * q + j] - M);
                    sc[q] = M;
                }
                __syncthreads();
            }
#pragma unroll
            for (int q = 0; q < G; ++q) lnl[q] = log(lc[q]) + sc[q] * kLn2;
        }
    }
    if (!has_root) return;    // a piece: its stores are its result (uniform per workgroup)
    double sum = 0.0;
#pragma unroll
    for (int q = 0; q < G; ++q) {
        const bool live = s[q] < m && cat == 0 && g == 0;
        if (live && site_lnl) site_lnl[(size_t)y * m + s[q]] = lnl[q];
        if (live) sum += (site_w ? site_w[s[q]] : 1.0) * lnl[q];
    }
    block_sum_store(sum, partial + (prog_main >= 0 ? (size_t)bx : (size_t)y * gridDim.x + blockIdx.x));
    if (64 * C == kSumThreads && fold_counter) fold_total(partial, blk0 + n_main, fold_counter, fold_out);
}

// One workgroup walks one NNI program (nni_program.h) over 16 G sites, wave c
// computing rate category c: the DNA walk of nni.hip with the products on
// the matrix cores.  P_v serves both variants from one load; its transpose
// (PmT, the same operand order) carries the outer partial down.  The outer
// partial and one child factor stay in registers between edges.  One site
// group a wave: two need 168 registers and spill 188 in the loop, one fits 128
// (up to 20 states), four waves a SIMD to hide the chain of dependent products
// that binds it (29 to 32 states: 168 registers at three waves, 8 to 10 spilled).
// 74 variants of 40 taxa x 5,000 sites, 20 states: 0.18 ms, 0.44 ms as one
// path-to-root program a variant.
template <typename T, int C, int V, int G>
__global__ __launch_bounds__(64 * C, (V <= 5 ? 4 : 3)) void nni_mfma_kernel(
    const NniOp* __restrict__ ops, const int* __restrict__ prog_begin, int n_prog, const uint32_t* __restrict__ tips,
    const T* __restrict__ clv, const int* __restrict__ scl, const double* __restrict__ Pm,
    const double* __restrict__ PmT, const double* __restrict__ PTm, const double* __restrict__ roots,
    const double* __restrict__ site_w, double2* __restrict__ part, int m, int m_pad, int S, uint32_t full, int n_taxa,
    int nblk, int n_var, int tip_lds) {
    constexpr int EV = C == 1 ? 2 : C < 4 ? C : 4, EP = EV / 2, TNV = (V > 4 ? 2 : 1) * V;
    __shared__ double xr[EV][C][16 * G];
    __shared__ int xs[EP][C][16 * G];
    static_assert(kNniSaves == 1, "one save slot");
    __shared__ double sv[C][G * V * 64];
    __shared__ int svs[C][G][64];
    extern __shared__ uint32_t tl[];        // n_taxa x 16 G masks (tip_lds)
    const int slot = (int)blockIdx.x >> 3;
    const int prog = slot % n_prog, bx = slot / n_prog * 8 + ((int)blockIdx.x & 7);
    if (bx >= nblk) return;
    if (tip_lds) {
        const uint32_t* blk = tips + (size_t)bx * 16 * G;
        for (int i = threadIdx.x; i < n_taxa * 16 * G; i += 64 * C)
            tl[i] = blk[(size_t)(i / (16 * G)) * m_pad + i % (16 * G)];
        __syncthreads();
    }
    const int lane = threadIdx.x & 63, g = lane >> 4, j = lane & 15;
    const int cat = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int sg0 = bx * G, n_sg = m_pad >> 4;
    const size_t slot_stride = (size_t)C * m_pad * 4 * V;
    double2* const out = part + (size_t)bx * n_var;

    // a node's own partial: tip masks (col: all single states or gaps) or a stored partial
    const auto fetch = [&](int node, T (&x)[G][V], uint32_t (&mk)[G], bool& col, int (&sc)[G]) {
#pragma unroll
        for (int q = 0; q < G; ++q) sc[q] = 0;
        col = false;
        if (node >= n_taxa) {
            const size_t idx = node - n_taxa;
#pragma unroll
            for (int q = 0; q < G; ++q) {
                const T* src = clv + idx * slot_stride + ((size_t)cat * n_sg + sg0 + q) * V * 64 + lane;
#pragma unroll
                for (int t = 0; t < V; ++t) x[q][t] = src[t * 64];
                sc[q] = scl[(idx * C + cat) * m_pad + (sg0 + q) * 16 + j];
            }
        } else if (node >= 0) {
            bool simple = true;
#pragma unroll
            for (int q = 0; q < G; ++q) {
                mk[q] = tip_lds ? tl[node * 16 * G + 16 * q + j] : tips[(size_t)node * m_pad + (sg0 + q) * 16 + j];
                simple = simple && (mk[q] == full || __popc(mk[q]) == 1);
            }
            col = __all(simple);
        }
    };
    // its factor P x (ones for a missing child)
    const auto factor = [&](int node, const T (&x)[G][V], const uint32_t (&mk)[G], bool col, double (&f)[G][V]) {
        if (node < 0) {
#pragma unroll
            for (int q = 0; q < G; ++q)
#pragma unroll
                for (int t = 0; t < V; ++t) f[q][t] = 1.0;
        } else if (col) {
            const double* base = PTm + ((size_t)node * C + cat) * (S + 1) * (4 * V) + g;
#pragma unroll
            for (int q = 0; q < G; ++q) {
                const int c = mk[q] == full ? S : __ffs(mk[q]) - 1;
                const double* pt = base + (size_t)c * (4 * V);
#pragma unroll
                for (int t = 0; t < V; ++t) f[q][t] = pt[4 * t];
            }
        } else {
            double p[TNV], v[G][V];
            load_pm<C, V>(node, cat, lane, Pm, p);
            const bool tip = node < n_taxa;
#pragma unroll
            for (int q = 0; q < G; ++q)
#pragma unroll
                for (int t = 0; t < V; ++t)
                    v[q][t] = tip ? ((mk[q] >> (4 * t + g)) & 1u ? 1.0 : 0.0) : to_d(x[q][t]);
            mfma_products<V, G>(p, v, f);
        }
    };
    int n_held = 0, held_var[EP] = {};
    const auto flush = [&]() {
        __syncthreads();
#pragma unroll
        for (int r = 0; r < (EV + C - 1) / C; ++r) {
            const int w = cat + r * C;
            if (w >= 2 * n_held) continue;
            const int p = w >> 1, i = lane % (16 * G);
            int var = held_var[0];
#pragma unroll
            for (int q = 1; q < EP; ++q) var = p == q ? held_var[q] : var;
            int M = xs[p][0][i];
#pragma unroll
            for (int c = 1; c < C; ++c) M = max(M, xs[p][c][i]);
            double lc = 0.0;
#pragma unroll
            for (int c = 0; c < C; ++c) lc += ldexp(xr[w][c][i], xs[p][c][i] - M);
            const int s = sg0 * 16 + lane;
            const bool live = lane < 16 * G && s < m;
            const double2 res = site_w ? nni_weighted(lc, M, live ? site_w[s] : 0.0, live) : nni_product(lc, M, live);
            if (lane == 63) {
                if (!(var & kNniSingle)) out[var + (w & 1)] = res;
                else if (!(w & 1)) out[var & ~kNniSingle] = res;
            }
        }
        __syncthreads();
        n_held = 0;
    };
    // l[q]: a site's sum over its states, still spread over the lane groups
    const auto hold = [&](const double (&l0)[G], const double (&l1)[G], const int (&sc)[G], const NniOp& op) {
        const int k = 2 * n_held + (op.flags & NNI_XY ? 1 : 0);
#pragma unroll
        for (int q = 0; q < G; ++q) {
            double a = l0[q], b = l1[q];
            a += __shfl_xor(a, 16, 64);
            b += __shfl_xor(b, 16, 64);
            a += __shfl_xor(a, 32, 64);
            b += __shfl_xor(b, 32, 64);
            if (g == 0) {
                xr[k][cat][16 * q + j] = a;
                xr[k ^ 1][cat][16 * q + j] = b;
                xs[n_held][cat][16 * q + j] = sc[q];
            }
        }
#pragma unroll
        for (int p = 0; p < EP; ++p)
            if (n_held == p) held_var[p] = op.var | (op.flags & NNI_ROOT ? kNniSingle : 0);
        ++n_held;
    };

    double O[G][V] = {}, B[G][V] = {};
    int sO[G] = {}, sB[G] = {};
    const int k0 = prog_begin[prog], k1 = prog_begin[prog + 1];
    NniOp nx = ops[k0];
    for (int k = k0; k < k1; ++k) {
        const NniOp op = nx;
        nx = ops[k + 1];
        double X[G][V], Y[G][V];
        int sX[G], sY[G];
        {
            T rx[G][V] = {}, ry[G][V] = {};
            uint32_t mx[G] = {}, my[G] = {};
            bool cx, cy;
            fetch(op.x, rx, mx, cx, sX);
            fetch(op.y, ry, my, cy, sY);
            factor(op.x, rx, mx, cx, X);
            factor(op.y, ry, my, cy, Y);
        }
        if (op.flags & NNI_INIT) {
            const double w = roots[kRootCatOff + cat];
#pragma unroll
            for (int q = 0; q < G; ++q) {
#pragma unroll
                for (int t = 0; t < V; ++t) {
                    O[q][t] = roots[4 * t + g] * w;
                    B[q][t] = Y[q][t];
                }
                sO[q] = 0;
                sB[q] = sY[q];
            }
            continue;
        }
        if (op.flags & NNI_POP) {
#pragma unroll
            for (int q = 0; q < G; ++q) {
#pragma unroll
                for (int t = 0; t < V; ++t) O[q][t] = sv[cat][(q * V + t) * 64 + lane];
                sO[q] = svs[cat][q][lane];
            }
        }
        if (op.flags & NNI_FETCH_S) {
            T r[G][V] = {};
            uint32_t mk[G] = {};
            bool col;
            fetch(op.s, r, mk, col, sB);
            factor(op.s, r, mk, col, B);
        }
        if (op.flags & NNI_SAVE) {
#pragma unroll
            for (int q = 0; q < G; ++q) {
#pragma unroll
                for (int t = 0; t < V; ++t) sv[cat][(q * V + t) * 64 + lane] = O[q][t];
                svs[cat][q][lane] = sO[q];
            }
        }
        if (op.flags & NNI_ROOT) {
            // in the pair's terms below: S = the factor of c, X = P_s (X x D)
            T r[G][V] = {};
            uint32_t mk[G] = {};
            bool col;
            int sD[G];
            double f[G][V], p[TNV];
            fetch(op.d, r, mk, col, sD);
            factor(op.d, r, mk, col, f);
#pragma unroll
            for (int q = 0; q < G; ++q) {
                sX[q] += sD[q];
#pragma unroll
                for (int t = 0; t < V; ++t) f[q][t] *= X[q][t];
            }
            load_pm<C, V>(op.s, cat, lane, Pm, p);
            mfma_products<V, G>(p, f, X);
            fetch(op.c, r, mk, col, sB);
            factor(op.c, r, mk, col, B);
        }
        if (op.flags & (NNI_PAIR | NNI_ROOT)) {
            double p[TNV], v[G][V], u[G][V], l0[G], l1[G];
            int sc[G];
            load_pm<C, V>(op.v, cat, lane, Pm, p);
#pragma unroll
            for (int q = 0; q < G; ++q)
#pragma unroll
                for (int t = 0; t < V; ++t) v[q][t] = B[q][t] * Y[q][t];
            mfma_products<V, G>(p, v, u);
#pragma unroll
            for (int q = 0; q < G; ++q) {
                l0[q] = 0.0;
#pragma unroll
                for (int t = 0; t < V; ++t) l0[q] = fma(O[q][t] * X[q][t], u[q][t], l0[q]);
#pragma unroll
                for (int t = 0; t < V; ++t) v[q][t] = B[q][t] * X[q][t];
            }
            mfma_products<V, G>(p, v, u);
#pragma unroll
            for (int q = 0; q < G; ++q) {
                l1[q] = 0.0;
#pragma unroll
                for (int t = 0; t < V; ++t) l1[q] = fma(O[q][t] * Y[q][t], u[q][t], l1[q]);
                sc[q] = sO[q] + sB[q] + sX[q] + sY[q];
            }
            hold(l0, l1, sc, op);
        }
        if (op.flags & NNI_DESC) {
            double p[TNV], v[G][V];
            load_pm<C, V>(op.v, cat, lane, PmT, p);
#pragma unroll
            for (int q = 0; q < G; ++q)
#pragma unroll
                for (int t = 0; t < V; ++t) v[q][t] = O[q][t] * B[q][t];
            mfma_products<V, G>(p, v, O);
            // lazy rescale, as in the pruning walker
            bool low = false;
#pragma unroll
            for (int q = 0; q < G; ++q) {
                sO[q] += sB[q];
                int h = __double2hiint(O[q][0]);
#pragma unroll
                for (int t = 1; t < V; ++t) h = max(h, __double2hiint(O[q][t]));
                low |= h < kLazyRescaleHi;
            }
            if (__builtin_amdgcn_ballot_w64(low) != 0) {
#pragma unroll
                for (int q = 0; q < G; ++q) {
                    const int e = site_exponent<V>(O[q]);
                    const double mx = site_max<V>(O[q]);
                    if (mx < 0x1p-256) {
                        sO[q] += e;
#pragma unroll
                        for (int t = 0; t < V; ++t) O[q][t] = ldexp(O[q][t], -e);
                    }
                }
            }
#pragma unroll
            for (int q = 0; q < G; ++q) {
#pragma unroll
                for (int t = 0; t < V; ++t) B[q][t] = Y[q][t];
                sB[q] = sY[q];
            }
        }
        if (n_held == EP) flush();
    }
    if (n_held) flush();    // (uniform per workgroup)
}

template <typename T, int C, int V>
void launch_nni_v(const NniArgs& a, int S, const uint32_t* tips, const double* Pm, const double* PmT, const double* PTm,
                  hipStream_t st) {
    const uint32_t full = S == 32 ? 0xFFFFFFFFu : ((1u << S) - 1u);
    const bool tl = a.max_taxa <= kMfmaTipLdsTaxa;
    hipLaunchKernelGGL((nni_mfma_kernel<T, C, V, kNniGroups>), dim3((a.one.nblk + 7) / 8 * 8 * a.n_prog), dim3(64 * C),
                       tl ? (size_t)a.max_taxa * 16 * kNniGroups * sizeof(uint32_t) : 0, st, a.ops, a.prog, a.n_prog,
                       tips, static_cast<const T*>(a.clv), a.scl, Pm, PmT, PTm, a.roots, a.site_w, a.part, a.one.m,
                       a.one.m_pad, S, full, a.one.n_taxa, a.one.nblk, a.one.n_var, tl ? 1 : 0);
}

template <typename T, int C, int V>
void launch_v(const MfmaArgs& a, hipStream_t st) {
    const uint32_t full = a.S == 32 ? 0xFFFFFFFFu : ((1u << a.S) - 1u);
    T* clv = static_cast<T*>(a.clv);
#define PHYLO_MFMA_LAUNCH(K)                                                                                           \
    hipLaunchKernelGGL(K, a.grid, dim3(64 * C), 0, st, a.ops, a.prog, a.tips, clv, a.scl, a.Pm, a.PTm, a.roots, a.site_w, \
                       a.site_lnl, a.partial, a.m, a.m_pad, a.S, full, a.n_taxa, a.n_main, a.prog_main, a.blk0,        \
                       a.prog_piece, a.tail0, a.n_tail, a.fold, a.fold_out)
    if (a.tip_lds) PHYLO_MFMA_LAUNCH((prune_mfma_kernel<T, C, V, kMfmaGroups, true>));
    else PHYLO_MFMA_LAUNCH((prune_mfma_kernel<T, C, V, kMfmaGroups, false>));
#undef PHYLO_MFMA_LAUNCH
}

template <typename T, int C, int V>
int resident_v() {
    int n = 0;
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, prune_mfma_kernel<T, C, V, kMfmaGroups, true>, 64 * C, 0) ==
                   hipSuccess ? n : 0;
}

// f(storage type, categories, operand slots) for a context's values
template <typename T, int C, class F>
void with_v(int S, F&& f) {
    switch (mfma_slots(S)) {
    case 2: f(T(), std::integral_constant<int, C>(), std::integral_constant<int, 2>()); break;
    case 3: f(T(), std::integral_constant<int, C>(), std::integral_constant<int, 3>()); break;
    case 4: f(T(), std::integral_constant<int, C>(), std::integral_constant<int, 4>()); break;
    case 5: f(T(), std::integral_constant<int, C>(), std::integral_constant<int, 5>()); break;
    case 6: f(T(), std::integral_constant<int, C>(), std::integral_constant<int, 6>()); break;
    case 7: f(T(), std::integral_constant<int, C>(), std::integral_constant<int, 7>()); break;
    default: f(T(), std::integral_constant<int, C>(), std::integral_constant<int, 8>()); break;
    }
}
template <typename T, class F>
void with_c(int C, int S, F&& f) {
    switch (C) {
    case 1: with_v<T, 1>(S, f); break;
    case 2: with_v<T, 2>(S, f); break;
    case 4: with_v<T, 4>(S, f); break;
    case 8: with_v<T, 8>(S, f); break;
    default: break;
    }
}
template <class F>
void with_kernel(bool f64, int C, int S, F&& f) {
    if (f64) with_c<double>(C, S, f);
    else with_c<float>(C, S, f);
}

}  // namespace

hipError_t mfma_launch(const MfmaArgs& a, hipStream_t st) {
    with_kernel(a.f64, a.C, a.S, [&](auto t, auto c, auto v) { launch_v<decltype(t), c(), v()>(a, st); });
    return hipGetLastError();
}

int mfma_resident(bool f64, int C, int S) {
    int n = 0;
    with_kernel(f64, C, S, [&](auto t, auto c, auto v) { n = resident_v<decltype(t), c(), v()>(); });
    return n;
}

hipError_t nni_mfma_launch(const NniArgs& a, int S, const uint32_t* tips, const double* Pm, const double* PmT,
                           const double* PTm, hipStream_t st) {
    with_kernel(a.f64, a.C, S, [&](auto t, auto c, auto v) {
        launch_nni_v<decltype(t), c(), v()>(a, S, tips, Pm, PmT, PTm, st);
    });
    return hipGetLastError();
}

hipError_t mfma_matrices(const double* V, const double* Vinv, const double* lam, const double* eff, const PRates& rates,
                         const RootWeights& roots, int S, int Sp, int C, int n_nodes, double* P, double* Pm, double* PmT,
                         double* PTm, double* d_roots, hipStream_t st) {
    const int slots = mfma_slots(S);
    hipLaunchKernelGGL(pwide_kernel, dim3(n_nodes * C), dim3(256), 0, st, V, Vinv, lam, eff, rates, roots, S, Sp, C, slots,
                       slots > 4 ? 2 : 1, P, Pm, PmT, PTm, d_roots);
    return hipGetLastError();
}
