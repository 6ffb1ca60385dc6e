// prune_device.h -- what the pruning kernels of libphylo_hip share: the op
// format of the compiled programs, loads and stores of partials, stochastic
// rounding, power-of-two scaling and the fixed-order compensated sums.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

enum SrcKind : int { SRC_TIP = 0, SRC_CLV = 1, SRC_CARRY_A = 2, SRC_CARRY_B = 3, SRC_NONE = 4 };
// OP_SWAP: the children were swapped into kind order (order_children); the
// stochastic rounding of a stored result is keyed by them in their original
// order.
// OP_SH_*: one-hot hints for the four commonest child shapes (children in
// kind order), set by order_children; the DNA walker tests them before its
// switch, the matrix walker runs a specialised op for each.
enum OpFlags : int {
    OP_ROOT = 1, OP_TO_B = 2, OP_SWAP = 4,
    OP_SH_AT = 8, OP_SH_TT = 16, OP_SH_AB = 32, OP_SH_AC = 64,
    OP_SH_ALL = OP_SH_AT | OP_SH_TT | OP_SH_AB | OP_SH_AC
};

struct alignas(16) Op {
    int l_node, r_node;   // child node ids: P matrices are per (child node, category)
    int l_kind, r_kind;   // SrcKind
    int l_idx, r_idx;     // tip row or partial slot
    int out_slot;         // slot to store the result in, -1 for none
    int flags;            // OpFlags
};

namespace {

constexpr int kBlock = 256;
constexpr int kMaxCat = 8;
constexpr int kMaxStates = 32;
constexpr double kLn2 = 0.69314718055994530942;
constexpr int kRootCatOff = 32;   // roots[]: per-state weights [0, 32), category weights after
constexpr int kRootDoubles = kRootCatOff + kMaxCat;

// Workgroups per CU below which a whole-tree launch has too few waves to
// hide its dependent chain: every site block is then walked as subtree
// pieces plus the top program (the tail split applied to all blocks), which
// multiplies the independent waves by the number of pieces.
constexpr int kSplitAllBelowPerCu = 4;

// Site groups per wave of the MFMA walker: two independent MFMA chains per
// wave share each P operand load and overlap their memory latency.
constexpr int kMfmaGroups = 2;

// Site groups per wave of the matrix-core NNI walk.
constexpr int kNniGroups = 1;

// ---------------------------------------------------------------------------
// Device helpers
// ---------------------------------------------------------------------------

__device__ inline void load4(const float* p, double v[4]) {
    const float4 x = *reinterpret_cast<const float4*>(p);
    v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w;
}
__device__ inline void load4(const double* p, double v[4]) {
    const double2 a = reinterpret_cast<const double2*>(p)[0];
    const double2 b = reinterpret_cast<const double2*>(p)[1];
    v[0] = a.x; v[1] = a.y; v[2] = b.x; v[3] = b.y;
}
__device__ inline void load_raw4(const float* p, float v[4]) {
    const float4 x = *reinterpret_cast<const float4*>(p);
    v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w;
}
__device__ inline void load_raw4(const double* p, double v[4]) { load4(p, v); }
__device__ inline void store4(float* p, const float v[4]) {
    *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
}
__device__ inline void store4(double* p, const double v[4]) {
    reinterpret_cast<double2*>(p)[0] = make_double2(v[0], v[1]);
    reinterpret_cast<double2*>(p)[1] = make_double2(v[2], v[3]);
}

// 32-bit integer hash (Wellons' "lowbias32" xorshift-multiply mix).
__device__ inline uint32_t mix32(uint32_t x) {
    x ^= x >> 16;
    x *= 0x7feb352du;
    x ^= x >> 15;
    x *= 0x846ca68bu;
    x ^= x >> 16;
    return x;
}

// Rounding of a partial (x >= 0) to the storage type.  FP32 storage rounds
// stochastically: 29 random bits are added below the float's last mantissa
// bit of the FP64 value and the bits a float does not hold are cut off, so x
// rounds up with probability equal to its distance from the float below.  A
// subtree with few tips produces the same few values at every site, so
// round-to-nearest would repeat the same error at thousands of sites and the
// total lnL would drift (+4.6e-3 at 128 taxa x 100,000 sites); with
// per-site random bits the errors average out.  The bits come from a hash of
// (site, node, category) stepped by a Weyl sequence per state, so results
// are reproducible and the same node rounds the same way in every program
// that computes it.  (Zero stays zero; values below the float normal range
// end as the nearest float of the truncated value.)
// The dithered cut and the power-of-two scaling commute (the cut reads only
// mantissa bits), so a walker may cut before or after scaling a partial.
__device__ inline double round_cut(double x, uint32_t bits, float) {
    // 64-bit add of the 29 dither bits, written on 32-bit halves
    const uint32_t lo = (uint32_t)__double2loint(x);
    const uint32_t sum = lo + (bits >> 3);
    const uint32_t hi = (uint32_t)__double2hiint(x) + (sum < lo ? 1u : 0u);
    return __hiloint2double((int)hi, (int)(sum & 0xe0000000u));   // <= 24 significant bits
}
__device__ inline double round_cut(double x, uint32_t, double) { return x; }

// Random bits for the partials of one (site, node, category); state i uses
// key + i * 0x9e3779b9.  The node is identified by its two children, in the
// order the program builder gave them.
__device__ inline uint32_t round_key(int s, int l_node, int r_node, int cat) {
    return mix32((uint32_t)s * 0x9e3779b1u ^ ((uint32_t)l_node * 0x85ebca77u + (uint32_t)r_node * 0x27d4eb2fu +
                                              (uint32_t)cat * 0xc2b2ae3du));
}
__device__ inline uint32_t round_key(int s, const Op& op, int cat) {
    return (op.flags & OP_SWAP) ? round_key(s, op.r_node, op.l_node, cat) : round_key(s, op.l_node, op.r_node, cat);
}

__device__ inline double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Compensated sum of partial[0, n) by one wave in a fixed order: lane l adds
// partial[l], partial[l + 64], ... with Kahan compensation, then the lanes'
// (sum, error) pairs meet in a two-sum butterfly.  Every lane returns the
// same total (two-sum gives the exact error whichever operand comes first).
// Adds b + bl to the compensated pair (hi, lo) by Knuth's two-sum.
__device__ inline void two_sum_add(double& hi, double& lo, double b, double bl) {
    const double t = hi + b;
    const double bb = t - hi;
    const double err = (hi - (t - bb)) + (b - bb);
    hi = t;
    lo = (lo + bl) + err;
}

// Threads of the compensated sum: one workgroup per program.
constexpr int kSumThreads = 256;
static_assert(kSumThreads == 4 * 64, "block_total: four waves");

// Compensated fixed-order sum of partial[0, n) by the first kSumThreads
// threads of one workgroup.  Each thread issues its loads eight at a time before adding
// them (Kahan), so their latencies overlap instead of queueing; the threads'
// (sum, error) pairs then meet by two-sum, in a butterfly within each wave
// and in LDS across the waves.  Thread 0 returns the total.
// An infinite value (a site of likelihood zero) has no compensation: inf - inf
// is no number.  With INF a wave that ends with none adds its values again
// without, and so do the waves' sums.
template <bool INF = true>
__device__ inline double block_total(const double* partial, int n) {
    double s = 0.0, comp = 0.0;
    for (int base = threadIdx.x < kSumThreads ? (int)threadIdx.x : n; base < n; base += 8 * kSumThreads) {
        double v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int i = base + u * kSumThreads;
            v[u] = i < n ? partial[i] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            if (base + u * kSumThreads < n) {
                const double x = v[u] - comp;
                const double t = s + x;
                comp = (t - s) - x;
                s = t;
            }
        }
    }
    double hi = s, lo = -comp;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) two_sum_add(hi, lo, __shfl_xor(hi, o, 64), __shfl_xor(lo, o, 64));
    if (INF && !(hi + lo == hi + lo)) {      // (the same in every lane)
        hi = lo = 0.0;
        for (int i = threadIdx.x; i < n; i += kSumThreads) hi += partial[i];
        hi = wave_sum(hi);
    }
    __shared__ double red_hi[kSumThreads / 64], red_lo[kSumThreads / 64];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane == 0 && wid < kSumThreads / 64) { red_hi[wid] = hi; red_lo[wid] = lo; }
    __syncthreads();
    hi = red_hi[0];
    lo = red_lo[0];
#pragma unroll
    for (int w = 1; w < kSumThreads / 64; ++w) two_sum_add(hi, lo, red_hi[w], red_lo[w]);
    const double t = hi + lo;
    return !INF || t == t ? t : (red_hi[0] + red_hi[1]) + (red_hi[2] + red_hi[3]);
}

// Sums v over the workgroup (any multiple of 64 threads); thread 0 stores it.
__device__ inline void block_sum_store(double v, double* dst) {
    __shared__ double red[16];
    v = wave_sum(v);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane == 0) red[wid] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int w = 0; w < (int)(blockDim.x >> 6); ++w) t += red[w];
        *dst = t;
    }
}

// The top launch of a tail split (its workgroups are the last blocks to
// finish an evaluation) folds in the final sum: each workgroup, once its
// partial is stored, counts itself in; the last one sums every block's
// partial in block_total's order (so the total equals final_sum_kernel's),
// writes it to the host-mapped total and returns the counter to zero.  The
// fences publish the few partials this launch wrote and drop stale copies
// before the sum reads them.  Workgroups of kSumThreads threads or more only.
// (Without block_total's second pass over infinite values: the host sums again
// where the total is no number, and the walkers stay as they are.)
__device__ inline void fold_total(const double* partial, int n_part, unsigned* counter, double* total) {
    __shared__ int last;
    if (threadIdx.x == 0) {
        __threadfence();
        last = atomicAdd(counter, 1u) == gridDim.x - 1;
        if (last) __threadfence();
    }
    __syncthreads();
    if (last) {
        const double t = block_total<false>(partial, n_part);
        if (threadIdx.x == 0) {
            *total = t;
            *counter = 0u;
        }
    }
}

// Bit j of a tip's state set as 1.0 or 0.0: a bit-field extract and an
// integer-to-double conversion.  (Building the double's high word from a
// mask needs a third instruction to copy the zero low word into each
// register pair; the conversion form ran the C2 kernel 1 % faster.)
template <int J>
__device__ inline double tip_bit(unsigned code) {
    return (double)((code >> J) & 1u);
}

// frexp exponent of the largest of four values (0 if none is positive): as
// signed integers the high words of positive doubles order like the values,
// and those of negative ones (P(t) from the eigen system can leave tiny
// negative partials) are negative, so they never win.
__device__ inline int max_exponent(const double (&L)[4]) {
    const int h = max(max(__double2hiint(L[0]), __double2hiint(L[1])), max(__double2hiint(L[2]), __double2hiint(L[3])));
    int e = (h >> 20) - 1022;
    if (h < 0x00100000) {   // no positive normal value: zero, subnormal or negative maximum
        const double mx = fmax(fmax(L[0], L[1]), fmax(L[2], L[3]));
        e = 0;
        if (mx > 0.0) (void)frexp(mx, &e);
    }
    return e;
}

// The largest high word of four doubles, as signed integers: for positive
// values it orders like the values (negative ones never win).
__device__ inline int max_hi_word(const double (&L)[4]) {
    return max(max(__double2hiint(L[0]), __double2hiint(L[1])), max(__double2hiint(L[2]), __double2hiint(L[3])));
}

// High word of 2^-256: carried DNA partials whose largest entry is below it
// are rescaled (walk4).
constexpr int kLazyRescaleHi = (1023 - 256) << 20;

// Taxa whose tip codes a DNA workgroup stages in LDS (one byte per site,
// sized at launch).
constexpr int kTipLdsTaxa = 256;
inline size_t tip_lds_bytes(int n_taxa) { return (size_t)n_taxa * 64; }

}  // namespace
