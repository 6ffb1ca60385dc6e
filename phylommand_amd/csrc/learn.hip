// learn.hip -- learned starting values for the model fit: a GPU forward
// simulator fused with site-pattern / pairwise-distance feature extraction,
// and a small MLP (FP32) trained with hand-written forward / backward
// kernels.  The simulator extends simpleML::simulate_chars
// (simpleML.cpp:233-292) with gamma rate categories, gaps and a seeded
// counter-based RNG.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <memory>
#include <new>
#include <random>
#include <string>
#include <vector>

#include "../../include/phylo_hip.h"
#include "../../include/phylo_learn.h"

namespace {

constexpr int kSimThreads = 512;
constexpr int kMaxSimTaxa = 32;
constexpr int kMaxSimNodes = 2 * kMaxSimTaxa - 1;
constexpr int kMaxSimCat = 8;
constexpr int kSimPairs = (kMaxSimTaxa * (kMaxSimTaxa - 1) / 2 + kSimThreads - 1) / kSimThreads;   // a thread, at most
constexpr int kFeat = 256;

__device__ inline uint64_t mix64(uint64_t z) {
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
}
// uniform in [0, 1) from a counter
__device__ inline float urand(uint64_t seed, uint64_t a, uint64_t b, uint64_t c) {
    const uint64_t h = mix64(seed ^ mix64(a * 0x9e3779b97f4a7c15ull ^ mix64(b * 0xc2b2ae3d27d4eb4full ^ (c + 1))));
    return (float)(h >> 40) * (1.0f / 16777216.0f);
}

// One workgroup per alignment.  Per-alignment inputs (eig = V[16], Vinv[16],
// lam[4]; pi[4]; cat_rates[C]) give P(t) = V exp(lam r t) Vinv in LDS as
// cumulative rows; walk holds the nodes in preorder as node | parent << 8.
// Each thread simulates one site of a chunk down the tree; a tip's states leave
// as four ballot words a wave (one bit a site and state), so the joint state
// counts of a pair of taxa are 16 popcounts of ANDed words per 64 sites.  (A
// byte a site, counted site by site into an array indexed at run time, which
// lies in scratch memory, took 1.42 ms for 512 alignments of 32 taxa x 2,000
// sites.)  Bound by the generator, three 64-bit mixes a draw, 94 draws a site,
// and by the chain of states down the tree behind it: eight waves a workgroup,
// so that 512 alignments give every SIMD four (four waves, two a SIMD, 0.40 ms;
// eight 0.31; sixteen 0.34, half of them without a pair to count).  A table of
// the innermost mixes, which the alignments share, made the kernel a tenth
// faster and its own launch and allocation took that back.
__global__ __launch_bounds__(kSimThreads) void sim_features_kernel(
    int n_taxa, int n_sites, int n_cat, const int* __restrict__ walk, const double* __restrict__ blen,
    const double* __restrict__ eig, const double* __restrict__ pi_all, const double* __restrict__ cat_all,
    float gap_frac, uint64_t seed, float* __restrict__ feat, uint32_t* __restrict__ masks_out) {
    const int a = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n_nodes = 2 * n_taxa - 1;
    extern __shared__ __align__(16) float cumP[];       // [n_nodes][n_cat][4][4]
    __shared__ unsigned char st[kMaxSimNodes - kMaxSimTaxa][kSimThreads];   // inner nodes' states
    __shared__ uint64_t tip[kMaxSimTaxa][kSimThreads / 16 + 1];    // [taxon][wave, state]; odd rows: no bank conflicts
    __shared__ float cum_pi[4];
    __shared__ int h_site[4 + 32 + 32];
    __shared__ float h_pair[16 + 32 + 32 + 32 + 8];
    __shared__ int base[4];
    __shared__ int invariant;
    const double* bl = blen + (size_t)a * n_nodes;
    const double* V = eig + (size_t)a * 36;
    const double* Vi = V + 16;
    const double* lam = V + 32;
    walk += (size_t)a * n_nodes;
    for (int i = tid; i < 4 + 32 + 32; i += kSimThreads) h_site[i] = 0;
    for (int i = tid; i < 16 + 32 + 32 + 32 + 8; i += kSimThreads) h_pair[i] = 0.f;
    if (tid < 4) base[tid] = 0;
    if (tid == 0) {
        invariant = 0;
        double c = 0.0;
        for (int i = 0; i < 4; ++i) { c += pi_all[(size_t)a * 4 + i]; cum_pi[i] = (float)c; }
        cum_pi[3] = 1.0f;
    }
    // cumulative P rows: cumP[(v, c)][i][j] = sum_{j' <= j} P_ij'
    for (int e = tid; e < n_nodes * n_cat * 4; e += kSimThreads) {
        const int i = e % 4, c = (e / 4) % n_cat, v = e / (4 * n_cat);
        const double t = bl[v] * cat_all[(size_t)a * n_cat + c];
        float* row = cumP + (size_t)e * 4;
        double acc = 0.0;
        float r[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            double p = 0.0;
#pragma unroll
            for (int k = 0; k < 4; ++k) p += V[i * 4 + k] * exp(lam[k] * t) * Vi[k * 4 + j];
            acc += p > 0.0 ? p : 0.0;
            r[j] = (float)acc;
        }
        const float tot = r[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) row[j] = r[j] / tot;
        row[3] = 1.0f;
    }
    __syncthreads();
    // pair ownership: thread owns pairs p = tid, tid + kSimThreads, ... (496 pairs for 32 taxa)
    const int n_pairs = n_taxa * (n_taxa - 1) / 2;
    int pa[kSimPairs], pb[kSimPairs];
#pragma unroll
    for (int q = 0; q < kSimPairs; ++q) {
        pa[q] = pb[q] = -1;
        int p = tid + q * kSimThreads;
        if (p >= n_pairs) continue;
        int i = 0;
        while (p >= n_taxa - 1 - i) { p -= n_taxa - 1 - i; ++i; }
        pa[q] = i;
        pb[q] = i + 1 + p;
    }
    int joint[kSimPairs][16];
#pragma unroll
    for (int q = 0; q < kSimPairs; ++q)
#pragma unroll
        for (int c = 0; c < 16; ++c) joint[q][c] = 0;
    int base_count = 0;      // threads < 4 n_taxa: state tid % 4 of taxon tid / 4
    for (int s0 = 0; s0 < n_sites; s0 += kSimThreads) {
        const int s = s0 + tid, waves = min(kSimThreads / 64, (n_sites - s0 + 63) / 64);    // (that have a site)
        const bool live = s < n_sites;      // (its wave's other lanes draw too: the ballots need every lane)
        if (wave < waves) {
            const int cat = n_cat > 1 ? min(n_cat - 1, (int)(urand(seed, a, s, 1u << 20) * n_cat)) : 0;
            const float u = urand(seed, a, s, (1u << 20) + 1);
            // the first state whose cumulative value exceeds u (3 at the end)
            int rs = !(u < cum_pi[0]);
            rs += rs == 1 && !(u < cum_pi[1]);
            rs += rs == 2 && !(u < cum_pi[2]);
            st[walk[0] - n_taxa][tid] = (unsigned char)rs;
            uint32_t cnt = 0;        // tips per state, a byte each
            for (int k = 1; k < n_nodes; ++k) {
                const int w = walk[k], v = w & 255;
                const int anc = st[(w >> 8) - n_taxa][tid];
                const float r = urand(seed, a, s, (uint64_t)v);
                const float4 row = *reinterpret_cast<const float4*>(cumP + (((size_t)v * n_cat + cat) * 4 + anc) * 4);
                int x = !(r < row.x);
                x += x == 1 && !(r < row.y);
                x += x == 2 && !(r < row.z);
                if (v >= n_taxa) {
                    st[v - n_taxa][tid] = (unsigned char)x;
                    continue;
                }
                // a tip: gaps, its states' words
                const bool ok = live && !(gap_frac > 0.f && urand(seed, a, s, (2u << 20) + v) < gap_frac);
                cnt += ok ? 1u << (8 * x) : 0u;
                const uint64_t m0 = __ballot(ok && x == 0), m1 = __ballot(ok && x == 1), m2 = __ballot(ok && x == 2),
                               m3 = __ballot(ok && x == 3);
                if (lane < 4) tip[v][4 * wave + lane] = lane == 0 ? m0 : lane == 1 ? m1 : lane == 2 ? m2 : m3;
                if (masks_out && live) masks_out[((size_t)a * n_taxa + v) * n_sites + s] = ok ? 1u << x : 15u;
            }
            if (live) {
                int distinct = 0, mx = 0, sq = 0, n_ok = 0;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int c = cnt >> (8 * j) & 255;
                    n_ok += c;
                    distinct += c > 0;
                    mx = max(mx, c);
                    sq += c * c;
                }
                if (distinct > 0) atomicAdd(&h_site[distinct - 1], 1);
                if (distinct == 1) atomicAdd(&invariant, 1);
                // minor-allele fraction (n - max) / n in bins of 1/64 and
                // Gini-Simpson diversity 1 - sum f^2 in bins of 3/128, both from
                // integers so the bin edges are exact
                const int nn2 = n_ok * n_ok;
                atomicAdd(&h_site[4 + (n_ok ? min(31, 64 * (n_ok - mx) / n_ok) : 0)], 1);
                atomicAdd(&h_site[36 + (n_ok ? min(31, 128 * (nn2 - sq) / (3 * nn2)) : 0)], 1);
            }
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < kSimPairs; ++q) {
            if (pa[q] < 0) continue;
            for (int w = 0; w < waves; ++w) {
                uint64_t x[4], y[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) { x[j] = tip[pa[q]][4 * w + j]; y[j] = tip[pb[q]][4 * w + j]; }
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j) joint[q][i * 4 + j] += __popcll(x[i] & y[j]);
            }
        }
        if (tid < 4 * n_taxa)
            for (int w = 0; w < waves; ++w) base_count += __popcll(tip[tid >> 2][4 * w + (tid & 3)]);
        __syncthreads();
    }
    // pair statistics
#pragma unroll
    for (int q = 0; q < kSimPairs; ++q) {
        if (pa[q] < 0) continue;
        int n = 0;
#pragma unroll
        for (int c = 0; c < 16; ++c) n += joint[q][c];
        if (n == 0) continue;
        const float inv = 1.f / n;
        const int same = joint[q][0] + joint[q][5] + joint[q][10] + joint[q][15];
        const int ts = joint[q][1] + joint[q][4] + joint[q][11] + joint[q][14];     // A<->G, C<->T
        const int tv = n - same - ts;
        const float pd = (n - same) * inv, pts = ts * inv, ptv = tv * inv;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                atomicAdd(&h_pair[i * 4 + j], 0.5f * (joint[q][i * 4 + j] + joint[q][j * 4 + i]) * inv / n_pairs);
        // p-distance in bins of 1/40, transition and transversion distances
        // in bins of 1/80 (integer bin edges)
        atomicAdd(&h_pair[16 + min(31, 40 * (n - same) / n)], 1.f / n_pairs);
        atomicAdd(&h_pair[48 + min(31, 80 * ts / n)], 1.f / n_pairs);
        atomicAdd(&h_pair[80 + min(31, 80 * tv / n)], 1.f / n_pairs);
        atomicAdd(&h_pair[112], pd / n_pairs);
        atomicAdd(&h_pair[113], pd * pd / n_pairs);
        atomicAdd(&h_pair[114], pts / n_pairs);
        atomicAdd(&h_pair[115], ptv / n_pairs);
        // Jukes-Cantor distance capped at 3
        const float jc = fminf(3.f, -0.75f * logf(fmaxf(1e-6f, 1.f - pd / 0.75f)));
        atomicAdd(&h_pair[116], jc / n_pairs);
    }
    if (tid < 4 * n_taxa) atomicAdd(&base[tid & 3], base_count);
    __syncthreads();
    float* f = feat + (size_t)a * kFeat;
    for (int i = tid; i < kFeat; i += kSimThreads) {
        float v = 0.f;
        const int nb = base[0] + base[1] + base[2] + base[3];
        if (i < 4) v = nb ? (float)base[i] / nb : 0.f;
        else if (i < 20) v = h_pair[i - 4];
        else if (i < 116) v = h_pair[16 + (i - 20)];
        else if (i < 120) v = (float)h_site[i - 116] / n_sites;
        else if (i < 184) v = (float)h_site[4 + (i - 120)] / n_sites;
        else if (i == 184) v = h_pair[112];
        else if (i == 185) v = sqrtf(fmaxf(0.f, h_pair[113] - h_pair[112] * h_pair[112]));
        else if (i == 186) v = h_pair[114];
        else if (i == 187) v = h_pair[115];
        else if (i == 188) v = (float)(n_sites * n_taxa - nb) / ((float)n_sites * n_taxa);
        else if (i == 189) v = h_pair[116];
        else if (i == 190) v = fminf(20.f, h_pair[114] / fmaxf(1e-6f, h_pair[115]));
        else if (i == 191) v = (float)invariant / n_sites;
        f[i] = v;
    }
}

// ---------------------------------------------------------------------------
// MLP kernels (FP32)
//
// A training step is six launches: two hidden layers forward (bias and ReLU
// in the product's epilogue, the minibatch's rows gathered as they are read),
// the output layer with the loss and its gradient, the gradients of the second
// and the first layer's pre-activations, and all weight and bias
// gradients with their Adam updates.  Every sum runs over k in ascending order
// by fused multiply-adds, one accumulator an output: Adam divides a gradient
// by its own magnitude, so another order (split sums, the matrix cores) moves
// a few weights by whole steps, although its gradients are as accurate.
// The products are a few tens of MFLOP, too few waves to hide a load behind
// another wave's work, so what binds is the chain of loads and dependent
// multiply-adds.  A workgroup of two waves owns a 16 x 32 tile (256 of them for
// 256 x 512 outputs, 2 x 2 a thread) and stages 64 k of both operands in LDS
// while the next two pieces are on their way into registers (what a launch reads
// was written by the launch before, on other XCDs, so it comes from beyond L2):
// 13.2 us for 256 x 512 x 512.  (Rows by scalar loads and columns from L1 waited
// in every 16-long piece: 18 us.)
// Wide layers and batches take 64 x 64 tiles, 4 x 4 a thread (large_tiles): the
// same sums in the same order.
// ---------------------------------------------------------------------------

constexpr int kTileK = 64;

// R x R outputs a thread, 16 threads a tile row.
template <int R_, int THREADS_>
struct Tile {
    static constexpr int R = R_, THREADS = THREADS_, M = THREADS_ / 16 * R_, N = 16 * R_;
    static constexpr int U = R_ == 2 ? 16 : 4;       // k read ahead of their sums
    struct alignas(16) Lds {
        float a[kTileK][M + R_];
        float b[kTileK][N];
    };
    static_assert(alignof(Lds) >= R_ * sizeof(float), "read R values at once");
};
typedef Tile<2, 128> Small;      // 16 x 32
typedef Tile<4, 256> Large;      // 64 x 64

__device__ __forceinline__ void read_values(const float* p, float (&v)[2]) {
    const float2 x = *reinterpret_cast<const float2*>(p);
    v[0] = x.x; v[1] = x.y;
}
__device__ __forceinline__ void read_values(const float* p, float (&v)[4]) {
    const float4 x = *reinterpret_cast<const float4*>(p);
    v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w;
}

// The thread's sums over k (ascending) of A(row, k) B(k, col) for rows
// row0 + R p .. and columns col0 + R q .. (p = thread / 16, q = thread % 16).
// A is row-major (K_MINOR: element (row, k) at A[row * lda + k], storage row
// rows[row] where set) or its transpose (A[k * lda + row], storage row rows[k]).
// B(k, col) is B[k * ldb + col].  Rows past M and columns past N repeat the last.
template <class T, bool K_MINOR>
__device__ __forceinline__ void tile_products(typename T::Lds& t, const float* __restrict__ A, int lda,
                                              const int* __restrict__ rows, int row0, int M, int K,
                                              const float* __restrict__ B, int ldb, int col0, int N,
                                              float (&acc)[T::R][T::R]) {
    constexpr int R = T::R, NA = T::M * kTileK / T::THREADS, NB = T::N * kTileK / T::THREADS;
    constexpr int SA = K_MINOR ? T::THREADS / 64 : T::THREADS / T::M, SB = T::THREADS / T::N;   // rows a step
    const int tid = threadIdx.x;
    // staging: A by k runs of 64 (K_MINOR: a wave's rows are its own, so their
    // addresses are uniform) or rows of the tile, B by rows of the tile.  A load
    // is a uniform base and the thread's own offset, so that a piece's addresses
    // cost the vector unit one instruction each.  Rows are reached in 64 bits:
    // those of a minibatch may lie anywhere in the training set.
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ak = K_MINOR ? tid & 63 : tid / T::M, ar = K_MINOR ? wave : tid % T::M;
    const int bk = tid / T::N, bc = min(col0 + tid % T::N, N - 1);
    const float* arow[K_MINOR ? NA : 1];
    if constexpr (K_MINOR) {
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            const int r = min(row0 + wave + SA * i, M - 1);
            arow[i] = A + (size_t)(rows ? rows[r] : r) * lda;
        }
    }
    const size_t aoff = (size_t)ak * lda + min(row0 + ar, M - 1), boff = (size_t)bk * ldb + bc;
    float ra[2][NA], rb[2][NB];
    const auto load = [&](int k0, int h) {
        if (k0 + kTileK <= K) {
#pragma unroll
            for (int i = 0; i < NA; ++i) {
                if constexpr (K_MINOR) ra[h][i] = (arow[i] + k0)[ak];
                else if (rows) ra[h][i] = A[(size_t)rows[k0 + ak + SA * i] * lda + min(row0 + ar, M - 1)];
                else ra[h][i] = (A + (size_t)(k0 + SA * i) * lda)[aoff];
            }
#pragma unroll
            for (int i = 0; i < NB; ++i) rb[h][i] = (B + (size_t)(k0 + SB * i) * ldb)[boff];
        } else {
#pragma unroll
            for (int i = 0; i < NA; ++i) {
                if constexpr (K_MINOR) {
                    ra[h][i] = arow[i][min(k0 + ak, K - 1)];
                } else {
                    const int k = min(k0 + ak + SA * i, K - 1);
                    ra[h][i] = A[(size_t)(rows ? rows[k] : k) * lda + min(row0 + ar, M - 1)];
                }
            }
#pragma unroll
            for (int i = 0; i < NB; ++i) rb[h][i] = B[(size_t)min(k0 + bk + SB * i, K - 1) * ldb + bc];
        }
    };
    const int p = tid >> 4, q = tid & 15;
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
        for (int j = 0; j < R; ++j) acc[i][j] = 0.f;
    const auto add = [&](const float (&x)[R], const float (&y)[R]) {
#pragma unroll
        for (int i = 0; i < R; ++i)
#pragma unroll
            for (int j = 0; j < R; ++j) acc[i][j] = fmaf(x[i], y[j], acc[i][j]);
    };
    const auto piece = [&](int k0, int h) {
        if (k0) __syncthreads();
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            if constexpr (K_MINOR) t.a[ak][ar + SA * i] = ra[h][i];
            else t.a[ak + SA * i][ar] = ra[h][i];
        }
#pragma unroll
        for (int i = 0; i < NB; ++i) t.b[bk + SB * i][tid % T::N] = rb[h][i];
        __syncthreads();
        if (k0 + 2 * kTileK < K) load(k0 + 2 * kTileK, h);
        const int n = min(kTileK, K - k0);
        if (n == kTileK) {
            // U k read ahead of their sums (few waves a SIMD: each read waited
            // for by itself costs the LDS latency, 3.3 us a piece of 64)
            constexpr int U = T::U;
            float x[2][U][R], y[2][U][R];
            const auto read = [&](int k, int h) {
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    read_values(&t.a[k + u][R * p], x[h][u]);
                    read_values(&t.b[k + u][R * q], y[h][u]);
                }
            };
            read(0, 0);
#pragma unroll
            for (int k = 0; k < kTileK; k += U) {
                const int h = k / U % 2;
                if (k + U < kTileK) read(k + U, 1 - h);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int u = 0; u < U; ++u) add(x[h][u], y[h][u]);
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
            for (int k = 0; k < n; ++k) {
                float x[R], y[R];
                read_values(&t.a[k][R * p], x);
                read_values(&t.b[k][R * q], y);
                add(x, y);
            }
        }
    };
    load(0, 0);
    if (kTileK < K) load(kTileK, 1);
    for (int k0 = 0; k0 < K; k0 += 2 * kTileK) {
        piece(k0, 0);
        if (k0 + kTileK < K) piece(k0 + kTileK, 1);
    }
}

// epi(row, col, value) for the thread's elements inside M x N
template <int R, class Epi>
__device__ __forceinline__ void tile_out(const float (&acc)[R][R], int row0, int M, int col0, int N, Epi&& epi) {
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
        for (int j = 0; j < R; ++j) {
            const int r = row0 + R * (threadIdx.x >> 4) + i, c = col0 + R * (threadIdx.x & 15) + j;
            if (r < M && c < N) epi(r, c, acc[i][j]);
        }
}

// H = relu(X W + b), X's rows through `rows` where set.
template <class T>
__global__ __launch_bounds__(T::THREADS) void layer_kernel(int M, int N, int K, const float* __restrict__ X,
                                                             const int* __restrict__ rows, const float* __restrict__ W,
                                                             const float* __restrict__ b, float* __restrict__ H) {
    __shared__ typename T::Lds t;
    const int nx = (N + T::N - 1) / T::N, row0 = blockIdx.x / nx * T::M, col0 = blockIdx.x % nx * T::N;
    float acc[T::R][T::R];
    tile_products<T, true>(t, X, K, rows, row0, M, K, W, N, col0, N, acc);
    tile_out(acc, row0, M, col0, N, [&](int r, int c, float v) { H[(size_t)r * N + c] = fmaxf(v + b[c], 0.f); });
}

// dZ = (dY W^T) x (H > 0), from the transposed weights WT: the gradient
// through a layer and its input's ReLU.
template <class T>
__global__ __launch_bounds__(T::THREADS) void back_kernel(int M, int N, int K, const float* __restrict__ dY,
                                                            const float* __restrict__ WT, const float* __restrict__ H,
                                                            float* __restrict__ dZ) {
    __shared__ typename T::Lds t;
    const int nx = (N + T::N - 1) / T::N, row0 = blockIdx.x / nx * T::M, col0 = blockIdx.x % nx * T::N;
    float acc[T::R][T::R];
    tile_products<T, true>(t, dY, K, nullptr, row0, M, K, WT, N, col0, N, acc);
    tile_out(acc, row0, M, col0, N, [&](int r, int c, float v) {
        const size_t i = (size_t)r * N + c;
        dZ[i] = H[i] > 0.f ? v : 0.f;
    });
}

// The output layer: Y = H W + b; with targets also dY = 2 (Y - T) / (M N) and
// the workgroup's share of the loss.
__global__ __launch_bounds__(Small::THREADS) void output_kernel(int M, int N, int K, const float* __restrict__ H,
                                                              const float* __restrict__ W, const float* __restrict__ b,
                                                              const float* __restrict__ T, const int* __restrict__ rows,
                                                              float* __restrict__ Y, float* __restrict__ dY,
                                                              float* __restrict__ loss_part) {
    __shared__ Small::Lds t;
    __shared__ float wave_loss[2];
    const int nx = (N + Small::N - 1) / Small::N, row0 = blockIdx.x / nx * Small::M, col0 = blockIdx.x % nx * Small::N;
    float acc[2][2], loss = 0.f;
    tile_products<Small, true>(t, H, K, nullptr, row0, M, K, W, N, col0, N, acc);
    tile_out(acc, row0, M, col0, N, [&](int r, int c, float v) {
        const float y = v + b[c];
        Y[(size_t)r * N + c] = y;
        if (T) {
            const float d = y - T[(size_t)(rows ? rows[r] : r) * N + c];
            dY[(size_t)r * N + c] = 2.f * d / ((float)M * N);
            loss += d * d / ((float)M * N);
        }
    });
    if (!T) return;
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) loss += __shfl_xor(loss, d, 64);
    if ((threadIdx.x & 63) == 0) wave_loss[threadIdx.x >> 6] = loss;
    __syncthreads();
    if (threadIdx.x == 0) loss_part[blockIdx.x] = wave_loss[0] + wave_loss[1];
}

// dZ = (dY W^T) x (H > 0) for the few outputs of the last layer (M x n_out by
// n_out x N, W stored N x n_out): eight rows and 64 units a wave, dY uniform.
__global__ __launch_bounds__(64) void output_back_kernel(int M, int N, int n_out, const float* __restrict__ dY,
                                                         const float* __restrict__ W, const float* __restrict__ H,
                                                         float* __restrict__ dZ) {
    constexpr int R = 8;
    const int nx = (N + 63) / 64, row0 = blockIdx.x / nx * R, c = blockIdx.x % nx * 64 + threadIdx.x;
    if (c >= N) return;
    float z[R] = {};
#pragma unroll 4
    for (int o = 0; o < n_out; ++o) {
        const float w = W[(size_t)c * n_out + o];
#pragma unroll
        for (int r = 0; r < R; ++r) z[r] = fmaf(dY[(size_t)min(row0 + r, M - 1) * n_out + o], w, z[r]);
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
        if (row0 + r < M) {
            const size_t i = (size_t)(row0 + r) * N + c;
            dZ[i] = H[i] > 0.f ? z[r] : 0.f;
        }
}

// WT = W^T (n x n)
__global__ __launch_bounds__(256) void transpose_kernel(int n, const float* __restrict__ W, float* __restrict__ WT) {
    __shared__ float t[32][33];
    const int nb = (n + 31) / 32, r0 = blockIdx.x / nb * 32, c0 = blockIdx.x % nb * 32;
    const int x = threadIdx.x & 31, y = threadIdx.x >> 5;
    for (int i = y; i < 32; i += 8)
        if (r0 + i < n && c0 + x < n) t[i][x] = W[(size_t)(r0 + i) * n + c0 + x];
    __syncthreads();
    for (int i = y; i < 32; i += 8)
        if (c0 + i < n && r0 + x < n) WT[(size_t)(c0 + i) * n + r0 + x] = t[x][i];
}

struct Adam {
    float lr, b1, b2, eps, c1, c2;
    float *w, *m, *v;      // null w: gradients only
};
__device__ __forceinline__ void put_gradient(const Adam& a, float* __restrict__ g, size_t i, float gi) {
    if (!a.w) {
        g[i] = gi;
        return;
    }
    const float mi = a.b1 * a.m[i] + (1.f - a.b1) * gi;
    const float vi = a.b2 * a.v[i] + (1.f - a.b2) * gi * gi;
    a.m[i] = mi;
    a.v[i] = vi;
    a.w[i] -= a.lr * (mi / a.c1) / (sqrtf(vi / a.c2) + a.eps);
}

// Every weight gradient A^T dZ and bias gradient (column sums of dZ) of the
// step, and the Adam updates (and W2's transpose kept up with them).
// Workgroups: the layers' tiles in turn, then a thread a bias column.
struct GradArgs {
    int n_in, n_hid, n_out, M;
    int tile[3], bias[3];              // first workgroup of each layer's tiles, of its biases
    size_t w_off[3], b_off[3];
};
template <class T>
__global__ __launch_bounds__(T::THREADS) void gradient_kernel(
    GradArgs a, const float* __restrict__ X, const int* __restrict__ rows, const float* __restrict__ H1,
    const float* __restrict__ H2, const float* __restrict__ dZ1, const float* __restrict__ dZ2,
    const float* __restrict__ dY, Adam adam, float* __restrict__ g, float* __restrict__ W2T) {
    __shared__ typename T::Lds t;
    const int blk = blockIdx.x;
    if (blk < a.bias[0]) {
        const int l = blk >= a.tile[2] ? 2 : blk >= a.tile[1] ? 1 : 0;
        const float* A = l == 0 ? X : l == 1 ? H1 : H2;
        const float* D = l == 0 ? dZ1 : l == 1 ? dZ2 : dY;
        const int n_a = l == 0 ? a.n_in : a.n_hid, n_d = l == 2 ? a.n_out : a.n_hid;
        const int nx = (n_d + T::N - 1) / T::N, tile = blk - a.tile[l];
        const int row0 = tile / nx * T::M, col0 = tile % nx * T::N;
        float acc[T::R][T::R];
        tile_products<T, false>(t, A, n_a, l == 0 ? rows : nullptr, row0, n_a, a.M, D, n_d, col0, n_d, acc);
        tile_out(acc, row0, n_a, col0, n_d, [&](int r, int c, float v) {
            const size_t i = a.w_off[l] + (size_t)r * n_d + c;
            put_gradient(adam, g, i, v);
            if (l == 1 && adam.w) W2T[(size_t)c * n_d + r] = adam.w[i];
        });
        return;
    }
    const int l = blk >= a.bias[2] ? 2 : blk >= a.bias[1] ? 1 : 0;
    const float* D = l == 0 ? dZ1 : l == 1 ? dZ2 : dY;
    const int n_d = l == 2 ? a.n_out : a.n_hid, j = (blk - a.bias[l]) * T::THREADS + threadIdx.x;
    if (j >= n_d) return;
    float s = 0.f;
    int i = 0;
    for (; i + 32 <= a.M; i += 32) {
        float x[32];
#pragma unroll
        for (int u = 0; u < 32; ++u) x[u] = D[(size_t)(i + u) * n_d + j];
#pragma unroll
        for (int u = 0; u < 32; ++u) s += x[u];
    }
    for (; i < a.M; ++i) s += D[(size_t)i * n_d + j];
    put_gradient(adam, g, a.b_off[l] + j, s);
}

}  // namespace

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------

struct phylo_mlp {
    int device = 0, n_cu = 0;
    int n_in = 0, n_hid = 0, n_out = 0, max_batch = 0;
    long n_params = 0;
    hipStream_t stream = nullptr;
    std::string err;
    float* d_w = nullptr;       // [W1 | b1 | W2 | b2 | W3 | b3]
    float* d_g = nullptr;
    float* d_m = nullptr;
    float* d_v = nullptr;
    float* d_x = nullptr;       // batch buffers
    float* d_t = nullptr;
    float* d_h1 = nullptr;
    float* d_h2 = nullptr;
    float* d_y = nullptr;
    float* d_dh1 = nullptr;
    float* d_dh2 = nullptr;
    float* d_dy = nullptr;
    float* d_loss = nullptr;
    float* d_w2t = nullptr;     // W2 transposed
    int* d_idx = nullptr;
    float* d_data_x = nullptr;  // training set
    float* d_data_t = nullptr;
    size_t data_x_cap = 0, data_t_cap = 0, loss_cap = 0, idx_cap = 0;
    int n_data = 0;
    long step = 0;
};

namespace {

int mfail(phylo_mlp* p, int code, const std::string& m) {
    if (p) p->err = m;
    return code;
}
#define MCHK(p, expr)                                                                            \
    do {                                                                                         \
        hipError_t e_ = (expr);                                                                  \
        if (e_ != hipSuccess) return mfail((p), PHYLO_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
    } while (0)

// Parameter views inside the flat buffer.
struct Views {
    float *W1, *b1, *W2, *b2, *W3, *b3;
};
Views views(phylo_mlp* p, float* base) {
    Views v;
    v.W1 = base;
    v.b1 = v.W1 + (size_t)p->n_in * p->n_hid;
    v.W2 = v.b1 + p->n_hid;
    v.b2 = v.W2 + (size_t)p->n_hid * p->n_hid;
    v.W3 = v.b2 + p->n_hid;
    v.b3 = v.W3 + (size_t)p->n_hid * p->n_out;
    return v;
}

unsigned tiles(int n, int t) { return (unsigned)((n + t - 1) / t); }

// Workgroups of the output layer, each with a part of the loss.
unsigned loss_parts(const phylo_mlp* p, int B) { return tiles(B, Small::M) * tiles(p->n_out, Small::N); }

// Whether an M x N product takes the large tiles: from one a CU on.  They read A
// half and B a quarter as often, which is what binds there; with fewer, CUs stand
// idle.  Kernel us, small / large, of the second layer: batch 1024 x 512 hidden
// (128 tiles) 24 / 32, 256 x 4096 (256) 318 / 231, 1024 x 1024 (256) 97 / 63,
// 1024 x 4096 1200 / 589; of the gradients at batch 1024: 512 hidden (64) 66 / 134,
// 1024 (256) 144 / 137, 4096 1830 / 978.
bool large_tiles(const phylo_mlp* p, int M, int N) {
    return (size_t)tiles(M, Large::M) * tiles(N, Large::N) >= (size_t)p->n_cu;
}

// One pass over B rows of X (through `rows` where set): the forward layers
// and the output; with targets also the loss parts and the gradients of the
// pre-activations (d_dy, d_dh2, d_dh1; d_w2t holds W2's transpose).
void pass(phylo_mlp* p, int B, const float* X, const int* rows, const float* T, float* loss) {
    const Views w = views(p, p->d_w);
    const int H = p->n_hid;
    const bool large = large_tiles(p, B, H);
    const dim3 grid(large ? tiles(H, Large::N) * tiles(B, Large::M) : tiles(H, Small::N) * tiles(B, Small::M));
    const dim3 block(large ? Large::THREADS : Small::THREADS);
    const auto layer = [&](int n_in, const float* in, const int* in_rows, const float* W, const float* b, float* out) {
        hipLaunchKernelGGL(large ? layer_kernel<Large> : layer_kernel<Small>, grid, block, 0, p->stream, B, H, n_in, in, in_rows,
                           W, b, out);
    };
    layer(p->n_in, X, rows, w.W1, w.b1, p->d_h1);
    layer(H, p->d_h1, nullptr, w.W2, w.b2, p->d_h2);
    hipLaunchKernelGGL(output_kernel, dim3(loss_parts(p, B)), dim3(Small::THREADS), 0, p->stream, B, p->n_out, H, p->d_h2, w.W3,
                       w.b3, T, rows, p->d_y, p->d_dy, loss);
    if (!T) return;
    hipLaunchKernelGGL(output_back_kernel, dim3(tiles(H, 64) * tiles(B, 8)), dim3(64), 0, p->stream, B, H, p->n_out, p->d_dy,
                       w.W3, p->d_h2, p->d_dh2);
    hipLaunchKernelGGL(large ? back_kernel<Large> : back_kernel<Small>, grid, block, 0, p->stream, B, H, H, p->d_dh2, p->d_w2t, p->d_h1, p->d_dh1);
}

void transpose_w2(phylo_mlp* p) {
    hipLaunchKernelGGL(transpose_kernel, dim3(tiles(p->n_hid, 32) * tiles(p->n_hid, 32)), dim3(256), 0, p->stream, p->n_hid,
                       views(p, p->d_w).W2, p->d_w2t);
}

// The step's gradients: into d_g (adam.w null) or straight into the weights.
void gradients(phylo_mlp* p, int B, const float* X, const int* rows, const Adam& adam) {
    const Views o = views(p, p->d_w);
    const auto off = [&](const float* q) { return (size_t)(q - p->d_w); };
    GradArgs a{p->n_in, p->n_hid, p->n_out, B, {}, {}, {off(o.W1), off(o.W2), off(o.W3)}, {off(o.b1), off(o.b2), off(o.b3)}};
    const int n_a[3] = {p->n_in, p->n_hid, p->n_hid}, n_d[3] = {p->n_hid, p->n_hid, p->n_out};
    const bool large = large_tiles(p, p->n_hid, p->n_hid);
    const int tile_m = large ? Large::M : Small::M, tile_n = large ? Large::N : Small::N;
    const int threads = large ? Large::THREADS : Small::THREADS;
    int n = 0;
    for (int l = 0; l < 3; ++l) {
        a.tile[l] = n;
        n += tiles(n_a[l], tile_m) * tiles(n_d[l], tile_n);
    }
    for (int l = 0; l < 3; ++l) {
        a.bias[l] = n;
        n += tiles(n_d[l], threads);
    }
    hipLaunchKernelGGL(large ? gradient_kernel<Large> : gradient_kernel<Small>, dim3(n), dim3(threads), 0, p->stream, a, X, rows, p->d_h1, p->d_h2, p->d_dh1, p->d_dh2,
                       p->d_dy, adam, p->d_g, p->d_w2t);
}

// The loss of a step from its parts.
float sum_loss(const float* part, unsigned n) {
    double s = 0.0;
    for (unsigned i = 0; i < n; ++i) s += part[i];
    return (float)s;
}

// Grows a device buffer to n elements; the old one stays if there is no memory
// for the new (the loss parts serve phylo_mlp_grad too).
template <typename T>
hipError_t grow(T*& d, size_t& have, size_t n) {
    if (n <= have) return hipSuccess;
    T* bigger = nullptr;
    const hipError_t e = hipMalloc(reinterpret_cast<void**>(&bigger), n * sizeof(T));
    if (e != hipSuccess) return e;
    if (d) (void)hipFree(d);
    d = bigger;
    have = n;
    return hipSuccess;
}

}  // namespace

extern "C" {

int phylo_sim_features(int device, int n_align, int n_taxa, int n_sites, int n_cat, const int32_t* left,
                       const int32_t* right, const int32_t* roots, const double* blen, const double* eig,
                       const double* pi, const double* cat_rates, double gap_frac, uint64_t seed, float* features,
                       uint32_t* masks) {
    if (n_align < 1 || n_taxa < 4 || n_taxa > kMaxSimTaxa || n_sites < 1 || n_sites > (1 << 20) || n_cat < 1 ||
        n_cat > kMaxSimCat ||
        !left || !right || !roots || !blen || !eig || !pi || !cat_rates || !features || gap_frac < 0 || gap_frac >= 1)
        return PHYLO_ERR_ARG;
    const int nn = 2 * n_taxa - 1;
    for (long i = 0; i < (long)n_align * nn; ++i)
        if (left[i] < -1 || left[i] >= nn || right[i] < -1 || right[i] >= nn) return PHYLO_ERR_ARG;
    // every tree must be a rooted binary tree over nodes 0..nn-1 with the tips
    // 0..n_taxa-1 childless: the kernel's walk and state table are sized by
    // that.  The walk lists the nodes in preorder with their parents.
    std::vector<int> n_par(nn), stack;
    // one device block for every input, the features and the masks, filled by one copy
    size_t off = 0;
    const auto take = [&](size_t bytes) {
        const size_t at = off;
        off += (bytes + 255) & ~size_t(255);
        return at;
    };
    const size_t N = (size_t)n_align;
    const size_t o_walk = take(N * nn * sizeof(int)), o_blen = take(N * nn * sizeof(double));
    const size_t o_eig = take(N * 36 * sizeof(double)), o_pi = take(N * 4 * sizeof(double));
    const size_t o_cat = take(N * n_cat * sizeof(double)), in_bytes = off;
    const size_t o_feat = take(N * kFeat * sizeof(float));
    const size_t o_mask = take(masks ? N * n_taxa * n_sites * sizeof(uint32_t) : 0);
    const std::unique_ptr<unsigned char[]> in(new (std::nothrow) unsigned char[in_bytes]);
    if (!in) return PHYLO_ERR_HIP;
    int* walk = reinterpret_cast<int*>(in.get() + o_walk);
    for (int k = 0; k < n_align; ++k) {
        const int32_t* L = left + (size_t)k * nn;
        const int32_t* R = right + (size_t)k * nn;
        if (roots[k] < n_taxa || roots[k] >= nn) return PHYLO_ERR_ARG;
        std::fill(n_par.begin(), n_par.end(), 0);
        for (int v = 0; v < nn; ++v) {
            const bool tip = v < n_taxa;
            if (tip != (L[v] < 0) || tip != (R[v] < 0)) return PHYLO_ERR_ARG;
            if (!tip) {
                ++n_par[L[v]];
                ++n_par[R[v]];
            }
        }
        for (int v = 0; v < nn; ++v)
            if (n_par[v] != (v == roots[k] ? 0 : 1)) return PHYLO_ERR_ARG;
        // connected: every node is reached from the root
        int* out = walk + (size_t)k * nn;
        int seen = 0;
        stack.assign(1, roots[k]);
        while (!stack.empty()) {
            const int w = stack.back(), v = w & 255;
            stack.pop_back();
            if (seen == nn) return PHYLO_ERR_ARG;
            out[seen++] = w;
            if (L[v] >= 0) {
                stack.push_back(R[v] | v << 8);
                stack.push_back(L[v] | v << 8);
            }
        }
        if (seen != nn) return PHYLO_ERR_ARG;
    }
    std::memcpy(in.get() + o_blen, blen, N * nn * sizeof(double));
    std::memcpy(in.get() + o_eig, eig, N * 36 * sizeof(double));
    std::memcpy(in.get() + o_pi, pi, N * 4 * sizeof(double));
    std::memcpy(in.get() + o_cat, cat_rates, N * n_cat * sizeof(double));
    if (hipSetDevice(device) != hipSuccess) return PHYLO_ERR_HIP;
    const hipStream_t st = hipStreamPerThread;     // (a stream of its own a call, and the staging buffer zeroed, took 80 us)
    int rc = PHYLO_OK;
    unsigned char* d = nullptr;
    if (hipMalloc(reinterpret_cast<void**>(&d), off) != hipSuccess ||
        hipMemcpyAsync(d, in.get(), in_bytes, hipMemcpyHostToDevice, st) != hipSuccess) {
        rc = PHYLO_ERR_HIP;
    } else {
        const auto dbl = [&](size_t o) { return reinterpret_cast<const double*>(d + o); };
        float* df = reinterpret_cast<float*>(d + o_feat);
        uint32_t* dm = masks ? reinterpret_cast<uint32_t*>(d + o_mask) : nullptr;
        hipLaunchKernelGGL(sim_features_kernel, dim3(n_align), dim3(kSimThreads), (size_t)nn * n_cat * 16 * sizeof(float), st,
                           n_taxa, n_sites, n_cat, reinterpret_cast<const int*>(d + o_walk), dbl(o_blen), dbl(o_eig),
                           dbl(o_pi), dbl(o_cat), (float)gap_frac, seed, df, dm);
        if (hipGetLastError() != hipSuccess ||
            hipMemcpyAsync(features, df, N * kFeat * sizeof(float), hipMemcpyDeviceToHost, st) != hipSuccess ||
            (masks && hipMemcpyAsync(masks, dm, N * n_taxa * n_sites * sizeof(uint32_t), hipMemcpyDeviceToHost, st) !=
                          hipSuccess) ||
            hipStreamSynchronize(st) != hipSuccess)
            rc = PHYLO_ERR_HIP;
    }
    if (d) (void)hipFree(d);
    return rc;
}

int phylo_mlp_create(int device, int n_in, int n_hidden, int n_out, int max_batch, uint64_t seed, phylo_mlp** out) {
    if (!out || n_in < 1 || n_hidden < 1 || n_out < 1 || max_batch < 1) return PHYLO_ERR_ARG;
    *out = nullptr;
    phylo_mlp* p = new phylo_mlp();
    p->device = device;
    p->n_in = n_in;
    p->n_hid = n_hidden;
    p->n_out = n_out;
    p->max_batch = max_batch;
    p->n_params = (long)n_in * n_hidden + n_hidden + (long)n_hidden * n_hidden + n_hidden + (long)n_hidden * n_out + n_out;
    auto alloc = [&](auto*& d, size_t n) { return hipMalloc(reinterpret_cast<void**>(&d), n * sizeof(*d)) == hipSuccess; };
    const size_t B = max_batch;
    if (hipSetDevice(device) != hipSuccess || hipStreamCreateWithFlags(&p->stream, hipStreamNonBlocking) != hipSuccess ||
        hipDeviceGetAttribute(&p->n_cu, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess ||
        !alloc(p->d_w, p->n_params) || !alloc(p->d_g, p->n_params) || !alloc(p->d_m, p->n_params) ||
        !alloc(p->d_v, p->n_params) || !alloc(p->d_x, B * n_in) || !alloc(p->d_t, B * n_out) ||
        !alloc(p->d_h1, B * n_hidden) || !alloc(p->d_h2, B * n_hidden) || !alloc(p->d_y, B * n_out) ||
        !alloc(p->d_dh1, B * n_hidden) || !alloc(p->d_dh2, B * n_hidden) || !alloc(p->d_dy, B * n_out) ||
        !alloc(p->d_w2t, (size_t)n_hidden * n_hidden) || grow(p->d_loss, p->loss_cap, loss_parts(p, max_batch)) != hipSuccess) {
        phylo_mlp_destroy(p);
        return PHYLO_ERR_HIP;
    }
    // He-normal weights, zero biases
    std::vector<float> w(p->n_params, 0.f);
    std::mt19937_64 rng(seed);
    std::normal_distribution<float> N01(0.f, 1.f);
    Views hv;
    hv.W1 = w.data();
    hv.b1 = hv.W1 + (size_t)n_in * n_hidden;
    hv.W2 = hv.b1 + n_hidden;
    hv.b2 = hv.W2 + (size_t)n_hidden * n_hidden;
    hv.W3 = hv.b2 + n_hidden;
    hv.b3 = hv.W3 + (size_t)n_hidden * n_out;
    for (long i = 0; i < (long)n_in * n_hidden; ++i) hv.W1[i] = N01(rng) * std::sqrt(2.f / n_in);
    for (long i = 0; i < (long)n_hidden * n_hidden; ++i) hv.W2[i] = N01(rng) * std::sqrt(2.f / n_hidden);
    for (long i = 0; i < (long)n_hidden * n_out; ++i) hv.W3[i] = N01(rng) * std::sqrt(1.f / n_hidden);
    std::vector<float> zero(p->n_params, 0.f);
    if (hipMemcpy(p->d_w, w.data(), w.size() * sizeof(float), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(p->d_m, zero.data(), zero.size() * sizeof(float), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(p->d_v, zero.data(), zero.size() * sizeof(float), hipMemcpyHostToDevice) != hipSuccess) {
        phylo_mlp_destroy(p);
        return PHYLO_ERR_HIP;
    }
    *out = p;
    return PHYLO_OK;
}

const char* phylo_mlp_last_error(const phylo_mlp* p) { return p ? p->err.c_str() : "null mlp"; }

long phylo_mlp_n_params(const phylo_mlp* p) { return p ? p->n_params : 0; }

int phylo_mlp_params(phylo_mlp* p, float* get, const float* set) {
    if (!p) return PHYLO_ERR_ARG;
    MCHK(p, hipSetDevice(p->device));
    if (set) MCHK(p, hipMemcpy(p->d_w, set, p->n_params * sizeof(float), hipMemcpyHostToDevice));
    if (get) MCHK(p, hipMemcpy(get, p->d_w, p->n_params * sizeof(float), hipMemcpyDeviceToHost));
    return PHYLO_OK;
}

int phylo_mlp_forward(phylo_mlp* p, int batch, const float* x, float* y) {
    if (!p || !x || !y || batch < 1) return PHYLO_ERR_ARG;
    MCHK(p, hipSetDevice(p->device));
    for (int b0 = 0; b0 < batch; b0 += p->max_batch) {
        const int B = std::min(p->max_batch, batch - b0);
        MCHK(p, hipMemcpyAsync(p->d_x, x + (size_t)b0 * p->n_in, (size_t)B * p->n_in * sizeof(float),
                               hipMemcpyHostToDevice, p->stream));
        pass(p, B, p->d_x, nullptr, nullptr, nullptr);
        MCHK(p, hipGetLastError());
        MCHK(p, hipMemcpyAsync(y + (size_t)b0 * p->n_out, p->d_y, (size_t)B * p->n_out * sizeof(float),
                               hipMemcpyDeviceToHost, p->stream));
    }
    MCHK(p, hipStreamSynchronize(p->stream));
    return PHYLO_OK;
}

int phylo_mlp_grad(phylo_mlp* p, int batch, const float* x, const float* t, float* loss, float* grad) {
    if (!p || !x || !t || batch < 1 || batch > p->max_batch) return PHYLO_ERR_ARG;
    MCHK(p, hipSetDevice(p->device));
    MCHK(p, hipMemcpyAsync(p->d_x, x, (size_t)batch * p->n_in * sizeof(float), hipMemcpyHostToDevice, p->stream));
    MCHK(p, hipMemcpyAsync(p->d_t, t, (size_t)batch * p->n_out * sizeof(float), hipMemcpyHostToDevice, p->stream));
    transpose_w2(p);
    pass(p, batch, p->d_x, nullptr, p->d_t, p->d_loss);
    gradients(p, batch, p->d_x, nullptr, Adam{});
    MCHK(p, hipGetLastError());
    std::vector<float> part(loss_parts(p, batch));
    if (loss) MCHK(p, hipMemcpyAsync(part.data(), p->d_loss, part.size() * sizeof(float), hipMemcpyDeviceToHost, p->stream));
    if (grad) MCHK(p, hipMemcpyAsync(grad, p->d_g, p->n_params * sizeof(float), hipMemcpyDeviceToHost, p->stream));
    MCHK(p, hipStreamSynchronize(p->stream));
    if (loss) *loss = sum_loss(part.data(), (unsigned)part.size());
    return PHYLO_OK;
}

int phylo_mlp_set_data(phylo_mlp* p, int n, const float* x, const float* t) {
    if (!p || n < 1 || !x || !t) return PHYLO_ERR_ARG;
    MCHK(p, hipSetDevice(p->device));
    p->n_data = 0;
    // (a larger set needs no room beside the one it replaces)
    const auto make_room = [](float*& d, size_t& have, size_t n) {
        if (n <= have) return;
        if (d) (void)hipFree(d);
        d = nullptr;
        have = 0;
    };
    make_room(p->d_data_x, p->data_x_cap, (size_t)n * p->n_in);
    make_room(p->d_data_t, p->data_t_cap, (size_t)n * p->n_out);
    MCHK(p, grow(p->d_data_x, p->data_x_cap, (size_t)n * p->n_in));
    MCHK(p, grow(p->d_data_t, p->data_t_cap, (size_t)n * p->n_out));
    MCHK(p, hipMemcpy(p->d_data_x, x, (size_t)n * p->n_in * sizeof(float), hipMemcpyHostToDevice));
    MCHK(p, hipMemcpy(p->d_data_t, t, (size_t)n * p->n_out * sizeof(float), hipMemcpyHostToDevice));
    p->n_data = n;
    return PHYLO_OK;
}

// Epochs of minibatch Adam over the stored training set (shuffled per epoch).
int phylo_mlp_train(phylo_mlp* p, int epochs, int batch, float lr, uint64_t seed, float* loss_per_epoch) {
    if (!p || epochs < 1 || batch < 1 || batch > p->max_batch || !p->d_data_x || p->n_data < 1)
        return PHYLO_ERR_ARG;
    MCHK(p, hipSetDevice(p->device));
    std::mt19937_64 rng(seed);
    std::vector<int> perm(p->n_data);
    const float b1 = 0.9f, b2 = 0.999f;
    // an epoch is enqueued whole: the shuffled order goes over once, the steps'
    // loss parts come back together
    const unsigned n_part = loss_parts(p, batch);
    const int steps = p->n_data / batch;
    MCHK(p, grow(p->d_idx, p->idx_cap, (size_t)p->n_data));
    MCHK(p, grow(p->d_loss, p->loss_cap, (size_t)std::max(1, steps) * n_part));
    std::vector<float> part((size_t)steps * n_part);
    transpose_w2(p);      // (kept up by the steps)
    for (int ep = 0; ep < epochs; ++ep) {
        for (int i = 0; i < p->n_data; ++i) perm[i] = i;
        std::shuffle(perm.begin(), perm.end(), rng);
        MCHK(p, hipMemcpyAsync(p->d_idx, perm.data(), perm.size() * sizeof(int), hipMemcpyHostToDevice, p->stream));
        for (int k = 0; k < steps; ++k) {
            const int* rows = p->d_idx + (size_t)k * batch;
            pass(p, batch, p->d_data_x, rows, p->d_data_t, p->d_loss + (size_t)k * n_part);
            ++p->step;
            const float c1 = 1.f - std::pow(b1, (float)p->step), c2 = 1.f - std::pow(b2, (float)p->step);
            gradients(p, batch, p->d_data_x, rows, Adam{lr, b1, b2, 1e-8f, c1, c2, p->d_w, p->d_m, p->d_v});
            MCHK(p, hipGetLastError());
        }
        if (steps)
            MCHK(p, hipMemcpyAsync(part.data(), p->d_loss, part.size() * sizeof(float), hipMemcpyDeviceToHost, p->stream));
        MCHK(p, hipStreamSynchronize(p->stream));
        double lsum = 0.0;
        for (int k = 0; k < steps; ++k) lsum += sum_loss(part.data() + (size_t)k * n_part, n_part);
        if (loss_per_epoch) loss_per_epoch[ep] = steps ? (float)(lsum / steps) : NAN;
    }
    return PHYLO_OK;
}

void phylo_mlp_destroy(phylo_mlp* p) {
    if (!p) return;
    (void)hipSetDevice(p->device);
    if (p->stream) (void)hipStreamSynchronize(p->stream);
    void* bufs[] = {p->d_w, p->d_g, p->d_m, p->d_v, p->d_x, p->d_t, p->d_h1, p->d_h2, p->d_y,
                    p->d_dh1, p->d_dh2, p->d_dy, p->d_loss, p->d_w2t, p->d_idx, p->d_data_x, p->d_data_t};
    for (void* b : bufs)
        if (b) (void)hipFree(b);
    if (p->stream) (void)hipStreamDestroy(p->stream);
    delete p;
}

}  // extern "C"
