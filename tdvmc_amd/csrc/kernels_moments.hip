// TDVP moments of one sampling stage:
//   <O>, <E_R>, <E_I>, S = <O O^T> - <O><O>^T, F = <O E> - <O><E>
// (the sums of src/TDVMC.cpp:1103-1109 combined as in :1506-1537).
//
// The walker-by-parameter matrix X = [O | E_R | E_I] (W x Pa, Pa = P + 2) is
// centred column-wise (two passes: column means in FP64, then centring while
// packing), and S_aug = Xc^T Xc / W is a dense contraction over walkers:
//   mode 0 (FP64):  v_mfma_f64_16x16x4 on FP64 operands;
//   mode 1 (mixed): every centred entry (rounded to FP32) is split into
//                   three bf16 terms x = x0 + x1 + x2 (exact: 24 significant
//                   bits) and each product is formed from the split terms on
//                   v_mfma_f32_32x32x16_bf16: x0*y0 + x0*y1 + x1*y0 (the
//                   "bf16x3" products) + x1*y1 + x0*y2 + x2*y0 (together
//                   "bf16x6", Henry, Tang, Heinecke, ARITH 2019), leaving out
//                   terms of relative size 2^-24 and below.  With two-term
//                   splits (16 bits) the per-entry residual of ~2^-18 left
//                   F = <O E> - <O><E> 1.4e-6 off FP64 on sampled N = 343
//                   data, where O and E_L correlate weakly.  FP32
//                   accumulation is folded into FP64 registers every 256
//                   walkers, and the walker slices are reduced in FP64.
// Only tiles on or above the diagonal are computed; F is column Pa-2 / Pa-1.
//
// Folded columns (MomentsWork::cols): the contraction runs over a subset of
// O's columns (one column per group of identical ones, such as the two slots
// of a k / -k pair that share |rho_k|^2), and the results are written to
// every full index of the group (MomentsWork::outmap).  Rows and columns of
// such a group are then bit-identical in S and F, so the directions along
// which S is singular by construction stay exactly singular in both
// precisions (the Tikhonov term then holds them at eps).

#include "common.hpp"
#include "kernels.hpp"

namespace tdvmc {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef double double4v __attribute__((ext_vector_type(4)));

constexpr int kColBlock = 256;
constexpr int kChunkRows = 64;     // walkers per column-sum chunk (fewer only past kMaxChunks chunks)
constexpr int kMaxChunks = 1024;

inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

struct Geometry {
    int P, Pa, tile, Pp, nb, ntiles, groups;
    int64_t W, Wp, ksteps;   // Wp: padded walkers; ksteps: MFMA k-steps over Wp
    int chunks;
};

Geometry geometry(int64_t W, int P, int mode)
{
    Geometry g;
    g.P = P;
    g.Pa = P + 2;
    g.tile = mode == 0 ? 16 : 32;
    g.Pp = (int)ceil_div(g.Pa, g.tile) * g.tile;
    g.nb = g.Pp / g.tile;
    g.ntiles = g.nb * (g.nb + 1) / 2;
    const int kstep = mode == 0 ? 4 : 16;
    const int fold = 256;                               // walkers per FP32 fold (mode 1)
    g.W = W;
    g.Wp = ceil_div(W, fold) * fold;
    g.ksteps = g.Wp / kstep;
    int64_t groups = g.Wp / fold;
    const int64_t cap = mode == 0 ? 64 : 32;
    if (groups > cap) groups = cap;
    if (groups < 1) groups = 1;
    g.groups = (int)groups;
    int64_t ch = ceil_div(W, kChunkRows);
    g.chunks = (int)(ch > kMaxChunks ? kMaxChunks : (ch < 1 ? 1 : ch));
    return g;
}

// O column of computed column c (c < P): cols[c], or c; ld is O's row stride
struct ColSrc {
    const int* cols;
    int ld;
    __device__ __forceinline__ int operator()(int c) const { return cols ? cols[c] : c; }
};

// ---- pass 1: column sums of X in FP64, per row chunk
template <typename TO>
__global__ void colsum_kernel(const TO* __restrict__ O, const double* __restrict__ ER, const double* __restrict__ EI,
                              int64_t W, int P, ColSrc cs, int chunks, double* __restrict__ part)
{
    const int Pa = P + 2;
    const int c = blockIdx.x * kColBlock + threadIdx.x;
    const int ch = blockIdx.y;
    const int64_t rows = (W + chunks - 1) / chunks;
    const int64_t w0 = ch * rows, w1 = min(W, w0 + rows);
    if (c >= Pa) return;
    double s = 0.0;
    if (c < P) {
        const int oc = cs(c);
        // independent loads in flight; the sum keeps walker order
#pragma unroll 8
        for (int64_t w = w0; w < w1; w++) s += (double)O[w * cs.ld + oc];
    } else if (c == P)
        for (int64_t w = w0; w < w1; w++) s += ER[w];
    else
        for (int64_t w = w0; w < w1; w++) s += EI[w];
    part[(size_t)ch * Pa + c] = s;
}

// one workgroup of 256 threads per column: strided partial sums, then a fixed
// reduction tree (wavefront butterflies, then the 4 wavefronts in order)
__global__ __launch_bounds__(256) void colmean_kernel(const double* __restrict__ part, int chunks, int Pa, int64_t W,
                                                      double* __restrict__ mean, const int* __restrict__ outmap,
                                                      int P_full, double* __restrict__ mean_full)
{
    __shared__ double red[4];
    const int c = blockIdx.x, tid = threadIdx.x;
    double s = 0.0;
    for (int ch = tid; ch < chunks; ch += 256) s += part[(size_t)ch * Pa + c];
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if ((tid & 63) == 0) red[tid >> 6] = s;
    __syncthreads();
    if (tid == 0) {
        const double m = (((red[0] + red[1]) + red[2]) + red[3]) / (double)W;
        mean[c] = m;
        if (outmap) {
            // computed column c -> its full indices; E_R, E_I -> P_full, P_full + 1
            const int Pc = Pa - 2;
            if (c < Pc) {
                for (int k = 0; k < 2; k++)
                    if (outmap[2 * c + k] >= 0) mean_full[outmap[2 * c + k]] = m;
            } else {
                mean_full[P_full + (c - Pc)] = m;
            }
        }
    }
}

__device__ __forceinline__ double xval(const float* O, const double* ER, const double* EI, int64_t W, int P,
                                       ColSrc cs, const double* mean, int64_t w, int c)
{
    if (w >= W || c >= P + 2) return 0.0;
    const double v = c < P ? (double)O[w * cs.ld + cs(c)] : (c == P ? ER[w] : EI[w]);
    return v - mean[c];
}
__device__ __forceinline__ double xval(const double* O, const double* ER, const double* EI, int64_t W, int P,
                                       ColSrc cs, const double* mean, int64_t w, int c)
{
    if (w >= W || c >= P + 2) return 0.0;
    const double v = c < P ? O[w * cs.ld + cs(c)] : (c == P ? ER[w] : EI[w]);
    return v - mean[c];
}

// ---- pass 2a (mode 0): pack centred FP64 operands as [cb][s][kk][pp]
//      column c = 16 cb + pp, walker w = 4 s + kk
template <typename TO>
__global__ void pack64_kernel(const TO* __restrict__ O, const double* __restrict__ ER, const double* __restrict__ EI,
                              int64_t W, int P, ColSrc cs, const double* __restrict__ mean, int64_t Wp, int Pp,
                              double* __restrict__ xt)
{
    const int64_t total = Wp * Pp;
    const int64_t S4 = Wp / 4;
    for (int64_t idx = threadIdx.x + (int64_t)blockIdx.x * blockDim.x; idx < total;
         idx += (int64_t)blockDim.x * gridDim.x) {
        // idx enumerates the packed layout; recover (w, c)
        const int pp = (int)(idx & 15);
        const int kk = (int)((idx >> 4) & 3);
        const int64_t rest = idx >> 6;
        const int64_t s = rest % S4;
        const int cb = (int)(rest / S4);
        const int64_t w = 4 * s + kk;
        const int c = 16 * cb + pp;
        xt[idx] = xval(O, ER, EI, W, P, cs, mean, w, c);
    }
}

// ---- pass 2b (mode 1): pack centred operands split into three bf16 terms as
//      [cb][s][part][h][l32][j], column c = 32 cb + l32, walker w = 16 s + 8 h + j
constexpr int kSplit = 3;
template <typename TO>
__global__ void pack_bf16_kernel(const TO* __restrict__ O, const double* __restrict__ ER, const double* __restrict__ EI,
                                 int64_t W, int P, ColSrc cs, const double* __restrict__ mean, int64_t Wp, int Pp,
                                 __bf16* __restrict__ xt)
{
    // one thread per (cb, s, h, l32): 8 walkers of one column
    const int64_t S16 = Wp / 16;
    const int64_t total = (int64_t)(Pp / 32) * S16 * 64;
    for (int64_t idx = threadIdx.x + (int64_t)blockIdx.x * blockDim.x; idx < total;
         idx += (int64_t)blockDim.x * gridDim.x) {
        const int l32 = (int)(idx & 31);
        const int h = (int)((idx >> 5) & 1);
        const int64_t rest = idx >> 6;
        const int64_t s = rest % S16;
        const int cb = (int)(rest / S16);
        const int c = 32 * cb + l32;
        __bf16* base = xt + ((((size_t)cb * S16 + s) * kSplit) * 64) * 8;
        // 8 walkers of each term: one 16-byte store per term
        bf16x8 v[kSplit];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int64_t w = 16 * s + 8 * h + j;
            float x = (float)xval(O, ER, EI, W, P, cs, mean, w, c);
#pragma unroll
            for (int q = 0; q < kSplit; q++) {
                const __bf16 xq = (__bf16)x;
                v[q][j] = xq;
                x -= (float)xq;   // exact: the remainder has at most 16 significant bits
            }
        }
#pragma unroll
        for (int q = 0; q < kSplit; q++)
            *reinterpret_cast<bf16x8*>(base + ((size_t)q * 64 + h * 32 + l32) * 8) = v[q];
    }
}

__device__ __forceinline__ void tile_of(int t, int nb, int* I, int* J)
{
    // t enumerates the upper triangle row by row
    int i = 0;
    while (t >= nb - i) {
        t -= nb - i;
        i++;
    }
    *I = i;
    *J = i + t;
}

// Workgroup -> (tile t, walker group g).  Consecutive workgroups go to the 8
// XCDs in turn (workgroup b runs on XCD b mod 8), each with its own L2: the
// blocks of XCD x are given a contiguous range of the group-major order, so
// every tile of a walker group reads that group's rows through one L2 and
// the rows come from HBM about once instead of once per XCD.
__device__ __forceinline__ void tile_group_of(int b, int ntiles, int groups, int* t, int* g)
{
    const int nblk = ntiles * groups;
    const int x = b & 7, k = b >> 3;
    const int per = nblk >> 3, extra = nblk & 7;
    const int lin = x * per + min(x, extra) + k;
    *g = lin / ntiles;
    *t = lin - *g * ntiles;
}

// ---- pass 3a (mode 0): FP64 MFMA over walker slices, one wave per (tile, group)
__global__ __launch_bounds__(64) void gemm64_kernel(const double* __restrict__ xt, int64_t ksteps, int nb, int groups,
                                                    double* __restrict__ partial)
{
    const int lane = threadIdx.x, ntiles = nb * (nb + 1) / 2;
    int t, g, I, J;
    tile_group_of(blockIdx.x, ntiles, groups, &t, &g);
    tile_of(t, nb, &I, &J);
    const int64_t per = (ksteps + groups - 1) / groups;
    const int64_t s0 = g * per, s1 = min(ksteps, s0 + per);
    const double* A = xt + (size_t)I * ksteps * 64;
    const double* B = xt + (size_t)J * ksteps * 64;
    double4v acc = {0.0, 0.0, 0.0, 0.0};
    // 8 k-steps' operands in flight: one step at a time the products waited
    // for memory
    int64_t s = s0;
    for (; s + 8 <= s1; s += 8) {
        double a[8], b[8];
#pragma unroll
        for (int q = 0; q < 8; q++) {
            a[q] = A[(s + q) * 64 + lane];
            b[q] = B[(s + q) * 64 + lane];
        }
#pragma unroll
        for (int q = 0; q < 8; q++) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[q], b[q], acc, 0, 0, 0);
    }
    for (; s < s1; s++) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(A[s * 64 + lane], B[s * 64 + lane], acc, 0, 0, 0);
    // D[i][j]: j = lane % 16, i = 4 v + lane / 16
    double* out = partial + (((size_t)g * ntiles + t) * 256);
#pragma unroll
    for (int v = 0; v < 4; v++) out[(4 * v + lane / 16) * 16 + (lane % 16)] = acc[v];
}

// ---- pass 3b (mode 1): split-bf16 MFMA, six products per k-step
__global__ __launch_bounds__(64) void gemm_bf16x6_kernel(const __bf16* __restrict__ xt, int64_t ksteps, int nb,
                                                         int groups, double* __restrict__ partial)
{
    const int lane = threadIdx.x, ntiles = nb * (nb + 1) / 2;
    int t, g, I, J;
    tile_group_of(blockIdx.x, ntiles, groups, &t, &g);
    tile_of(t, nb, &I, &J);
    // per k-step block: kSplit parts x 64 lanes x 8 bf16
    const size_t step_elems = kSplit * 64 * 8;
    const bf16x8* A = reinterpret_cast<const bf16x8*>(xt + (size_t)I * ksteps * step_elems);
    const bf16x8* B = reinterpret_cast<const bf16x8*>(xt + (size_t)J * ksteps * step_elems);
    // groups split the k-steps in whole folds of 16 steps (256 walkers)
    const int64_t folds = ksteps / 16;
    const int64_t per = (folds + groups - 1) / groups;
    const int64_t f0 = g * per, f1 = min(folds, f0 + per);
    double acc64[16];
#pragma unroll
    for (int v = 0; v < 16; v++) acc64[v] = 0.0;
    // The leading term x0*y0 carries nearly all of each product: its 16-walker
    // MFMA sums go to FP64 at every k-step, so FP32 rounds only one MFMA's sum
    // of it (a 256-walker FP32 accumulator left S errors of ~1e-4 absolute on
    // entries ~1e5, enough to make S + eps I indefinite at eps = 1e-4).  The
    // five smaller terms (2^-8 of it and below) share an FP32 accumulator
    // folded every 256 walkers.
    const floatx16 zero = {};
    for (int64_t f = f0; f < f1; f++) {
        floatx16 acc = zero;
        for (int64_t s = f * 16; s < f * 16 + 16; s++) {
            const bf16x8* a = A + s * (kSplit * 64) + lane;
            const bf16x8* b = B + s * (kSplit * 64) + lane;
            const bf16x8 a0 = a[0], a1 = a[64], a2 = a[128];
            const bf16x8 b0 = b[0], b1 = b[64], b2 = b[128];
            const floatx16 lead = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, b0, zero, 0, 0, 0);
            // smallest terms first
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, b2, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a2, b0, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, b1, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, b1, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, b0, acc, 0, 0, 0);
#pragma unroll
            for (int v = 0; v < 16; v++) acc64[v] += (double)lead[v];
        }
#pragma unroll
        for (int v = 0; v < 16; v++) acc64[v] += (double)acc[v];
    }
    // D[i][j]: j = lane % 32, i = 8 (v / 4) + 4 (lane / 32) + (v % 4)
    double* out = partial + (((size_t)g * ntiles + t) * 1024);
#pragma unroll
    for (int v = 0; v < 16; v++) out[(8 * (v / 4) + 4 * (lane / 32) + (v % 4)) * 32 + (lane % 32)] = acc64[v];
}

// s = cov(computed columns i, j), i <= j, to every full index: S (both
// triangles) for two operators, F for an operator and an energy
__device__ __forceinline__ void store_cov(double s, int i, int j, int P, const int* __restrict__ outmap, int P_full,
                                          double* __restrict__ S, double* __restrict__ F)
{
    // full indices of computed columns i and j (one, or two for a folded group)
    int fi[2] = {i, -1}, fj[2] = {j, -1};
    if (outmap) {
        if (i < P) fi[0] = outmap[2 * i], fi[1] = outmap[2 * i + 1];
        if (j < P) fj[0] = outmap[2 * j], fj[1] = outmap[2 * j + 1];
    }
    if (i < P && j < P) {
        for (int a = 0; a < 2; a++)
            for (int b = 0; b < 2; b++)
                if (fi[a] >= 0 && fj[b] >= 0) {
                    S[(size_t)fi[a] * P_full + fj[b]] = s;
                    S[(size_t)fj[b] * P_full + fi[a]] = s;
                }
    } else if (i < P && (j == P || j == P + 1)) {
        for (int a = 0; a < 2; a++)
            if (fi[a] >= 0) F[(size_t)(j - P) * P_full + fi[a]] = s;
    }
}

// ---- pass 4: sum slices, scale 1/W, scatter to S (both triangles) and F.
// One tile element per thread, its slices loaded 16 at a time and added in
// order: with 4 elements per thread and one load at a time the latency of 128
// loads was 18 to 37 us (W = 8192 .. 131072).
__global__ __launch_bounds__(256) void reduce_tiles_kernel(const double* __restrict__ partial, int ntiles, int nb,
                                                           int tile, int groups, int P, int64_t W,
                                                           const int* __restrict__ outmap, int P_full,
                                                           double* __restrict__ S, double* __restrict__ F)
{
    const int t = blockIdx.x;
    int I, J;
    tile_of(t, nb, &I, &J);
    const int tt = tile * tile;
    const int e = blockIdx.y * 256 + threadIdx.x;   // tt is a multiple of 256
    // diagonal tiles: take the upper element for both triangles
    if (I == J && e / tile > e % tile) return;
    const double* p = partial + (size_t)t * tt + e;
    const size_t stride = (size_t)ntiles * tt;
    double s = 0.0;
#pragma unroll 16
    for (int g = 0; g < groups; g++) s += p[g * stride];
    s *= 1.0 / (double)W;
    store_cov(s, I * tile + e / tile, J * tile + e % tile, P, outmap, P_full, S, F);
}

// ---- few columns, few walkers (FP64): two launches instead of five.
// Workgroup c centres a chunk of kSmallRows walkers on the chunk's own means
// in LDS and forms its products on FP64 MFMA; the second kernel combines the
// chunks by the parallel-variance formula, sum_c (M_c + n_c d_c d_c^T) with
// d_c = mean_c - mean, so nothing is subtracted that is larger than the
// spread of the samples.
constexpr int kSmallRows = 64, kSmallCols = 64, kSmallChunks = 512;
static_assert(kSmallRows == kChunkRows && kSmallChunks <= kMaxChunks, "chunk means fit the column sums' buffer");

inline bool moments_small(int64_t W, int P, int mode)
{
    // sums, means, packing, products and reduction are a launch each, 41 to
    // 62 us together at these sizes whatever the work; the two launches take
    // 9 us (16 columns, 1024 walkers) to 14 us (34 columns, 16384 walkers).
    // More columns or chunks would outgrow the LDS of the combination.
    return mode == 0 && P + 2 <= kSmallCols && W <= (int64_t)kSmallRows * kSmallChunks;
}
inline int small_chunks(int64_t W) { return (int)ceil_div(W, kSmallRows); }

template <typename TO>
__global__ __launch_bounds__(256) void small_partial_kernel(const TO* __restrict__ O, const double* __restrict__ ER,
                                                            const double* __restrict__ EI, int64_t W, int P, ColSrc cs,
                                                            int nb, double* __restrict__ mean, double* __restrict__ part)
{
    // 68 doubles a row: the rows of an MFMA operand (16 doubles each) start 8 banks
    // apart, so two that are read together share 24 of 32 banks, where 64 doubles
    // would put them in the same ones
    constexpr int LD = kSmallCols + 4;
    __shared__ double X[kSmallRows * LD];
    __shared__ double m[4][kSmallCols];
    const int tid = threadIdx.x, Pa = P + 2, Pp = nb * 16;
    const int64_t w0 = (int64_t)blockIdx.x * kSmallRows;
    const int n = (int)min((int64_t)kSmallRows, W - w0);
    const int c = tid & 63, q = tid >> 6;   // this thread's column and rows q, q + 4, ...
    const int oc = c < P ? cs(c) : 0;
    double v[kSmallRows / 4];
    double s = 0.0;
#pragma unroll
    for (int i = 0; i < kSmallRows / 4; i++) {
        const int64_t w = w0 + q + 4 * i;
        v[i] = 0.0;
        if (q + 4 * i < n && c < Pa) v[i] = c < P ? (double)O[w * cs.ld + oc] : (c == P ? ER[w] : EI[w]);
    }
#pragma unroll
    for (int i = 0; i < kSmallRows / 4; i++) s += v[i];
    m[q][c] = s;
    __syncthreads();
    const double mc = (((m[0][c] + m[1][c]) + m[2][c]) + m[3][c]) / (double)n;
    if (q == 0 && c < Pa) mean[(size_t)blockIdx.x * Pa + c] = mc;
#pragma unroll
    for (int i = 0; i < kSmallRows / 4; i++)
        if (c < Pp) X[(q + 4 * i) * LD + c] = (q + 4 * i < n && c < Pa) ? v[i] - mc : 0.0;
    __syncthreads();
    const int lane = tid & 63, pp = lane & 15, kk = lane >> 4;
    const int ntiles = nb * (nb + 1) / 2;
    for (int t = q; t < ntiles; t += 4) {
        int I, J;
        tile_of(t, nb, &I, &J);
        double4v acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int k = 0; k < kSmallRows; k += 4)
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(X[(k + kk) * LD + 16 * I + pp], X[(k + kk) * LD + 16 * J + pp], acc,
                                                       0, 0, 0);
        double* out = part + ((size_t)blockIdx.x * ntiles + t) * 256;
#pragma unroll
        for (int u = 0; u < 4; u++) out[(4 * u + kk) * 16 + pp] = acc[u];
    }
}

__global__ __launch_bounds__(1024) void small_combine_kernel(const double* __restrict__ cmean,
                                                             const double* __restrict__ part, int chunks, int64_t W,
                                                             int P, int nb, const int* __restrict__ outmap, int P_full,
                                                             double* __restrict__ mean, double* __restrict__ S,
                                                             double* __restrict__ F)
{
    __shared__ double cm[kSmallChunks * 32];   // chunk means of the tile's 16 + 16 columns
    __shared__ double red[1024];
    __shared__ double mt[32];
    const int t = blockIdx.x, tid = threadIdx.x, Pa = P + 2, ntiles = gridDim.x;
    int I, J;
    tile_of(t, nb, &I, &J);
    auto rows = [&](int k) { return (double)min((int64_t)kSmallRows, W - (int64_t)k * kSmallRows); };
    // total means of the 32 columns: 32 strided sums each, then a fixed tree
    {
        const int u = tid & 31, col = u < 16 ? 16 * I + u : 16 * J + u - 16;
        double s = 0.0;
#pragma unroll 4
        for (int k = tid >> 5; k < chunks; k += 32) {
            const double v = col < Pa ? cmean[(size_t)k * Pa + col] : 0.0;
            cm[k * 32 + u] = v;
            s += rows(k) * v;
        }
        red[tid] = s;
        __syncthreads();
        for (int o = 16; o > 0; o >>= 1) {
            if ((tid >> 5) < o) red[tid] += red[tid + 32 * o];
            __syncthreads();
        }
        if (tid < 32) {
            const double m = red[tid] / (double)W;
            mt[tid] = m;
            // the diagonal tiles hold every column once
            if (I == J && blockIdx.y == 0 && tid < 16 && col < Pa) {
                if (col >= P)
                    mean[P_full + (col - P)] = m;
                else if (!outmap)
                    mean[col] = m;
                else
                    for (int k = 0; k < 2; k++)
                        if (outmap[2 * col + k] >= 0) mean[outmap[2 * col + k]] = m;
            }
        }
        __syncthreads();
    }
    // element (i, j) of the tile, 64 a workgroup: chunks tid / 64, + 16, ..., then
    // the 16 sums (a workgroup for all 256 elements had four times the loads in a
    // row: 16 against 8.6 us at 34 columns and 256 chunks)
    const int e = blockIdx.y * 64 + (tid & 63), i = e >> 4, j = e & 15;
    const double mi = mt[i], mj = mt[16 + j];
    double s = 0.0;
#pragma unroll 8
    for (int k = tid >> 6; k < chunks; k += 16)
        s += part[((size_t)k * ntiles + t) * 256 + e] + rows(k) * (cm[k * 32 + i] - mi) * (cm[k * 32 + 16 + j] - mj);
    red[tid] = s;
    __syncthreads();
    if (tid < 64 && !(I == J && i > j)) {
        s = 0.0;
#pragma unroll
        for (int q = 0; q < 16; q++) s += red[tid + 64 * q];
        store_cov(s * (1.0 / (double)W), 16 * I + i, 16 * J + j, P, outmap, P_full, S, F);
    }
}

}  // namespace

void moments_work_bytes(int64_t W, int P, int mode, size_t* xt, size_t* partial, size_t* colsum)
{
    Geometry g = geometry(W, P, mode);
    if (mode == 0)
        *xt = (size_t)g.Wp * g.Pp * sizeof(double);
    else
        *xt = (size_t)g.Wp * g.Pp * kSplit * sizeof(__bf16);
    *partial = (size_t)g.groups * g.ntiles * g.tile * g.tile * sizeof(double);
    *colsum = (size_t)g.chunks * g.Pa * sizeof(double);
    // (the small form keeps its chunks' means where the column sums go, a chunk
    // being a column-sum chunk, and their tiles, 32 nb (nb + 1) / 2 bytes a sample
    // against 128 nb packed, where the packed operands go)
}

template <typename TO>
hipError_t launch_moments(const TO* O, const double* ER, const double* EI, int64_t W, int P, int mode,
                          const MomentsWork& wk, double* mean, double* S, double* F, hipStream_t st)
{
    if (W <= 0) return hipErrorInvalidValue;
    // computed columns: all P of O, or the wk.P_cols of a fold
    const bool fold = wk.cols != nullptr;
    if (fold && (!wk.outmap || !wk.mean_cols || wk.P_cols < 1 || wk.P_cols > P)) return hipErrorInvalidValue;
    const int Pc = fold ? wk.P_cols : P;
    const ColSrc cs{wk.cols, P};
    double* mc = fold ? wk.mean_cols : mean;   // means of the computed columns
    Geometry g = geometry(W, Pc, mode);
    size_t xb, pb, cb;
    moments_work_bytes(W, Pc, mode, &xb, &pb, &cb);
    if (wk.xt_bytes < xb || wk.partial_bytes < pb || wk.colsum_bytes < cb) return hipErrorInvalidValue;

    if (moments_small(W, Pc, mode)) {
        const int chunks = small_chunks(W);
        double* tiles = static_cast<double*>(wk.xt);
        hipLaunchKernelGGL(small_partial_kernel<TO>, dim3(chunks), dim3(256), 0, st, O, ER, EI, W, Pc, cs, g.nb, wk.colsum,
                           tiles);
        hipLaunchKernelGGL(small_combine_kernel, dim3(g.ntiles, 4), dim3(1024), 0, st, wk.colsum, tiles, chunks, W, Pc, g.nb,
                           wk.outmap, P, mean, S, F);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(colsum_kernel<TO>, dim3((unsigned)ceil_div(g.Pa, kColBlock), g.chunks), dim3(kColBlock), 0, st,
                       O, ER, EI, W, Pc, cs, g.chunks, wk.colsum);
    hipLaunchKernelGGL(colmean_kernel, dim3((unsigned)g.Pa), dim3(256), 0, st, wk.colsum, g.chunks, g.Pa, W, mc,
                       wk.outmap, P, mean);
    if (mode == 0) {
        const int64_t total = g.Wp * g.Pp;
        int64_t blocks = ceil_div(total, 256);
        if (blocks > 16384) blocks = 16384;
        hipLaunchKernelGGL(pack64_kernel<TO>, dim3((unsigned)blocks), dim3(256), 0, st, O, ER, EI, W, Pc, cs, mc,
                           g.Wp, g.Pp, static_cast<double*>(wk.xt));
        hipLaunchKernelGGL(gemm64_kernel, dim3(g.ntiles * g.groups), dim3(64), 0, st, static_cast<const double*>(wk.xt),
                           g.ksteps, g.nb, g.groups, wk.partial);
    } else {
        const int64_t total = (int64_t)(g.Pp / 32) * (g.Wp / 16) * 64;
        int64_t blocks = ceil_div(total, 256);
        if (blocks > 16384) blocks = 16384;
        hipLaunchKernelGGL(pack_bf16_kernel<TO>, dim3((unsigned)blocks), dim3(256), 0, st, O, ER, EI, W, Pc, cs, mc,
                           g.Wp, g.Pp, static_cast<__bf16*>(wk.xt));
        hipLaunchKernelGGL(gemm_bf16x6_kernel, dim3(g.ntiles * g.groups), dim3(64), 0, st,
                           static_cast<const __bf16*>(wk.xt), g.ksteps, g.nb, g.groups, wk.partial);
    }
    hipLaunchKernelGGL(reduce_tiles_kernel, dim3(g.ntiles, g.tile * g.tile / 256), dim3(256), 0, st, wk.partial, g.ntiles, g.nb, g.tile,
                       g.groups, Pc, W, wk.outmap, P, S, F);
    return hipGetLastError();
}

template hipError_t launch_moments<float>(const float*, const double*, const double*, int64_t, int, int,
                                          const MomentsWork&, double*, double*, double*, hipStream_t);
template hipError_t launch_moments<double>(const double*, const double*, const double*, int64_t, int, int,
                                           const MomentsWork&, double*, double*, double*, hipStream_t);

}  // namespace tdvmc
