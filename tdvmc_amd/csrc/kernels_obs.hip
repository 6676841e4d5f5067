// Additional observables of every walker: the pair distribution g(r) and the
// structure factor S(k) of BosonsBulk::CalculateAdditionalSystemProperties
// (src/PhysicalSystems/BosonsBulk.cpp:474-520).
//
// One 256-thread workgroup per walker, coordinates staged in LDS as FP64
// (padded to 4 components; 32-bit box fractions as well in the mixed form).
//   g(r): every unordered pair once (row i meets partners i + 1 .. i + M
//   mod N, M = (N-1)/2, rows i < N/2 also i + N/2 for even N; a row is split
//   into segments over threads); the pair's bin is counted in an LDS u32 histogram, and the counts
//   reach a u64 total per bin with one global atomic each (exact and
//   order-free).  The value of a bin is count x (D/(N-1)) / scaling[bin]
//   (ObservableVsOnGridWithScaling::AddToHistogram, :45-50).
//   S(k): the shells' wave vectors are integer n with non-negative
//   components, k = 2 pi n / L, so exp(i k.r) = prod_a e_a^{n_a} with
//   e_a = exp(2 pi i x_a / L).  Per chunk of particles the powers e_a^m,
//   m = 0..nmax, are tabulated in LDS (particle index fastest, so a thread
//   walks three fixed rows with immediate offsets); a thread then forms the products for
//   its wave vectors (D-1 complex multiplies per particle and vector) and
//   adds them up (the vectors past the last multiple of 256 are split over
//   the threads by particle residue).  One thread per shell sums its
//   vectors' totals in order:
//   S = (C^2 + S^2) / (N n_k).
// FP64 form: distances by the reference's minimum image (src/Utils.cpp:266-281)
// and the bin of the reference's FP64 division, powers by complex recurrence
// from one sincospi; in 2-D and 3-D obs_mfma_kernel below takes S(k) as a matrix
// product and the bins from thresholds of r^2.  Mixed form: FP32 distances from
// the wrapping difference of 32-bit box fractions (exact minimum image), FP32
// powers each from its own reduced phase, FP32 sums per chunk added in FP64.

#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"

namespace tdvmc {

namespace {

constexpr int kObsThreads = 256;

template <typename T>
struct Cx {
    T re, im;
};

template <typename T>
__device__ __forceinline__ Cx<T> cmul(Cx<T> a, Cx<T> b)
{
    return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}

// entries of obs_mfma_kernel's table region: the powers of a chunk, or the product
__host__ __device__ inline size_t obs_mfma_table(int D, int nm, int CS, int npair)
{
    const size_t powers = (size_t)D * nm * CS;
    const size_t mt = (2 * npair + 15) / 16, nt = (2 * nm + 15) / 16;
    const size_t prod = (16 * mt * (16 * nt + 1) + 1) / 2;
    return powers > prod ? powers : prod;
}

// src/Utils.cpp:266-281: round half away from zero, an exact +-L/2 nudged inwards
__device__ __forceinline__ double nic_coord_ref(double x, double L, double Lr)
{
    const int k = (int)(x * Lr + ((x >= 0.0) ? 0.5 : -0.5));
    double res = x - k * L;
    if (res == L / 2.0)
        res -= 1e-10;
    else if (res == -L / 2.0)
        res += 1e-10;
    return res;
}

// The workgroup's counts into the totals.  One workgroup goes through several
// small walkers (obs_grid) and adds once: with a walker each, the atomics on
// the few totals were nearly all of the time (16384 walkers, N = 20: 360 us,
// 82 with 16 walkers each; N = 64: 420 and 205).
__device__ __forceinline__ void add_counts(const ObsArgs& a, const unsigned* cnt, int tid)
{
    for (int b = tid; b < a.count; b += kObsThreads) {
        const unsigned c = cnt[b];
        if (c) atomicAdd(a.gr_tot + b, (unsigned long long)c);
    }
}

// the workgroup's pair counts [count], behind the walker's LDS
template <typename T, int D>
__device__ __forceinline__ unsigned* obs_counts(const ObsArgs& a, unsigned char* smem)
{
    const int R = a.V >> 8, Vr = a.V & 255, G = Vr ? kObsThreads / Vr : 1;
    return reinterpret_cast<unsigned*>(smem + ((size_t)4 * a.N + 2 * (size_t)(256 * R + Vr * G)) * sizeof(double) +
                                       (sizeof(T) == 4 ? (size_t)a.N * sizeof(uint4) : 0) +
                                       (size_t)D * (a.nmax + 1) * (a.chunk + 1) * sizeof(Cx<T>));
}

// One walker w.  SHARED: the workgroup goes through several (obs_grid)
template <typename T, int D, bool SHARED>
__device__ __forceinline__ void obs_walker(const ObsArgs& a, int64_t w, unsigned char* smem)
{
    const int tid = threadIdx.x;
    const int N = a.N;
    const int nm = a.nmax + 1;
    double* pos = reinterpret_cast<double*>(smem);                           // [N][4] (x, y, z, 0)
    uint4* fix = reinterpret_cast<uint4*>(pos + 4 * (size_t)N);               // [N] box fractions (mixed form)
    // S(k) work split (below): R rounds of 256 vectors, Vr = V mod 256 vectors
    // left over, split into G items each
    const int R = a.V >> 8, Vr = a.V & 255;
    const int G = Vr ? kObsThreads / Vr : 1;
    double* part = reinterpret_cast<double*>(fix + (sizeof(T) == 4 ? N : 0));   // [256 R + Vr G][2] totals
    // phase tables [D][nm][chunk + 1]: the particle index runs fastest, and the
    // padded row keeps the rows of different powers in different banks
    int CS = a.chunk + 1;
    Cx<T>* tab = reinterpret_cast<Cx<T>*>(part + 2 * (size_t)(256 * R + Vr * G));
    unsigned* cnt = reinterpret_cast<unsigned*>(tab + (size_t)D * nm * CS);   // [count]
    const int* kvec = a.kvec;
    // a thread's vectors and table rows stay the walker's own: kept in registers over
    // all walkers they took 30 to 60 more
    if constexpr (SHARED) asm volatile("" : "+s"(CS), "+s"(kvec));
    if constexpr (!SHARED)
        for (int b = tid; b < a.count; b += kObsThreads) cnt[b] = 0u;
    const double* Rw = a.R + w * (int64_t)N * D;
    for (int e = tid; e < N * 4; e += kObsThreads) {
        const int i = e >> 2, c = e & 3;
        pos[e] = c < D ? Rw[i * D + c] : 0.0;
    }
    if constexpr (sizeof(T) == 4) {
        // 32-bit fractions of the box: the wrapping difference is the minimum image
        for (int i = tid; i < N; i += kObsThreads) {
            unsigned u[3] = {0u, 0u, 0u};
#pragma unroll
            for (int c = 0; c < D; c++) {
                double f = Rw[i * D + c] * a.Lr;
                f -= __builtin_floor(f);
                u[c] = (unsigned)(unsigned long long)(f * 4294967296.0);
            }
            fix[i] = make_uint4(u[0], u[1], u[2], 0u);
        }
    }
    __syncthreads();

    // ------------------------------------------------------------ g(r)
    // Work item (row i, segment): particle i stays in registers and meets the
    // partners j = i + 1 + o (mod N) for the segment's offsets o.  Every row
    // has M = (N-1)/2 offsets, rows i < N/2 one more (o = N/2 - 1, j = i + N/2)
    // when N is even, so every unordered pair occurs once.  Consecutive
    // threads hold consecutive segments of a row: with the same segment of
    // consecutive rows the lanes of a wavefront meet their neighbours at one
    // distance where the particles are in order, and their additions to one bin
    // wait for each other (1-D, N = 208, 702 walkers 85 us, this way 57; 2-D, N = 343,
    // 4000 walkers 369 and 259).  In the mixed 3-D form, where order matters less, the
    // reads decide: consecutive rows read consecutive partners, segments of a row
    // can all start in the same banks (4000 walkers, N = 214 215 us, segments first
    // 255; N = 343 381 and 389; N = 400 461 and 580).
    {
        const int M = (N - 1) / 2;
        const int even = (N % 2 == 0) ? 1 : 0;
        const int S = a.gr_segs;
        const int seg = (M + even + S - 1) / S;
        const float sc = (float)(a.L * (1.0 / 4294967296.0));
        for (int t = tid; t < N * S; t += kObsThreads) {
            constexpr bool ROWS = sizeof(T) == 4 && D == 3;
            const int hi = t / (ROWS ? N : S), lo = t - hi * (ROWS ? N : S);
            const int i = ROWS ? lo : hi, sg = ROWS ? hi : lo;
            const int Mi = M + ((even && i < N / 2) ? 1 : 0);
            const int o0 = sg * seg, o1 = min(Mi, o0 + seg);
            int j = i + 1 + o0;
            if (j >= N) j -= N;
            if constexpr (sizeof(T) == 8) {
                // the reference's minimum image and sum of squares, without fused multiply-adds
#pragma clang fp contract(off)
                const double4 ri = *reinterpret_cast<const double4*>(pos + 4 * i);
                for (int o = o0; o < o1; o++) {
                    const double4 rj = *reinterpret_cast<const double4*>(pos + 4 * j);
                    double d = nic_coord_ref(ri.x - rj.x, a.L, a.Lr);
                    double s = d * d;
                    if constexpr (D > 1) {
                        d = nic_coord_ref(ri.y - rj.y, a.L, a.Lr);
                        s += d * d;
                    }
                    if constexpr (D > 2) {
                        d = nic_coord_ref(ri.z - rj.z, a.L, a.Lr);
                        s += d * d;
                    }
                    const double r = __builtin_sqrt(s);
                    if (r < a.gmax) {
                        const int bin = (int)__builtin_floor(r / a.spacing);
                        if (bin < a.count) atomicAdd(cnt + bin, 1u);
                    }
                    if (++j == N) j = 0;
                }
            } else {
                const uint4 ui = fix[i];
                const float gmax = (float)a.gmax, isp = (float)(1.0 / a.spacing);
                for (int o = o0; o < o1; o++) {
                    const uint4 uj = fix[j];
                    float d = (float)(int)(ui.x - uj.x);
                    float s = d * d;
                    if constexpr (D > 1) {
                        d = (float)(int)(ui.y - uj.y);
                        s += d * d;
                    }
                    if constexpr (D > 2) {
                        d = (float)(int)(ui.z - uj.z);
                        s += d * d;
                    }
                    const float r = __builtin_amdgcn_sqrtf(s) * sc;
                    if (r < gmax) {
                        const int bin = (int)(r * isp);
                        if (bin < a.count) atomicAdd(cnt + bin, 1u);
                    }
                    if (++j == N) j = 0;
                }
            }
        }
    }

    // ------------------------------------------------------------ S(k)
    // Vectors v < 256 R (R = V / 256) go one per thread and round over all
    // particles.  The Vr = V mod 256 left over are split by particle residue:
    // item (r, g), g < G = 256 / Vr, sums vector 256 R + r over the particles
    // i = g mod G, so every thread has at most one such item.  Per-vector and
    // per-item totals meet in LDS and are added per shell in a fixed order.
    constexpr int kRounds = 4;
    const bool has_item = tid < Vr * G;
    const int ir = has_item ? tid % Vr : 0, ig = has_item ? tid / Vr : 0;
    int nv[kRounds + 1][3];
    double accR[kRounds + 1], accI[kRounds + 1];
#pragma unroll
    for (int q = 0; q <= kRounds; q++) {
        const int v = q < kRounds ? tid + q * kObsThreads : 256 * R + ir;
        const bool ok = q < kRounds ? q < R : has_item;
#pragma unroll
        for (int c = 0; c < 3; c++) nv[q][c] = (ok && c < D) ? kvec[v * 4 + c] : 0;
        accR[q] = accI[q] = 0.0;
    }
    // this thread's table rows: power n[c] of axis c, all particles of the chunk
    auto rows = [&](const int* n, const Cx<T>** r) {
#pragma unroll
        for (int c = 0; c < D; c++) r[c] = tab + ((size_t)c * nm + n[c]) * CS;
    };
    auto term = [&](const Cx<T>* const* r, int il) {
        Cx<T> z = r[0][il];
        if constexpr (D > 1) z = cmul(z, r[1][il]);
        if constexpr (D > 2) z = cmul(z, r[2][il]);
        return z;
    };
    for (int c0 = 0; c0 < N; c0 += a.chunk) {
        const int nc = min(a.chunk, N - c0);
        __syncthreads();   // previous chunk's table reads are done
        for (int e = tid; e < nc * D; e += kObsThreads) {
            const int il = e / D, c = e - il * D;
            double t = pos[(c0 + il) * 4 + c] * a.Lr;
            t -= __builtin_floor(t);
            Cx<T>* col = tab + (size_t)c * nm * CS + il;   // power m at col[m * CS]
            if constexpr (sizeof(T) == 8) {
                double sn, cs;
                sincospi(2.0 * t, &sn, &cs);
                const Cx<T> e1{cs, sn};
                Cx<T> pw{1.0, 0.0};
                for (int m = 0; m < nm; m++) {
                    col[(size_t)m * CS] = pw;
                    pw = cmul(pw, e1);
                }
            } else {
                for (int m = 0; m < nm; m++) {
                    double u = (double)m * t;
                    u -= __builtin_floor(u);
                    float sn, cs;
                    Prec<float>::sincos_small((float)u, &sn, &cs);
                    col[(size_t)m * CS] = Cx<T>{cs, sn};
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < kRounds; q++) {
            if (q >= R) break;
            const Cx<T>* r[D];
            rows(nv[q], r);
            T sr = (T)0, si = (T)0;
#pragma unroll 4
            for (int il = 0; il < nc; il++) {
                const Cx<T> z = term(r, il);
                sr += z.re;
                si += z.im;
            }
            accR[q] += (double)sr;
            accI[q] += (double)si;
        }
        if (has_item) {
            const Cx<T>* r[D];
            rows(nv[kRounds], r);
            T sr = (T)0, si = (T)0;
            for (int il = (ig - c0 % G + G) % G; il < nc; il += G) {
                const Cx<T> z = term(r, il);
                sr += z.re;
                si += z.im;
            }
            accR[kRounds] += (double)sr;
            accI[kRounds] += (double)si;
        }
    }
#pragma unroll
    for (int q = 0; q < kRounds; q++) {
        if (q < R) {
            const int v = tid + q * kObsThreads;
            part[2 * v] = accR[q];
            part[2 * v + 1] = accI[q];
        }
    }
    double* rest = part + 2 * 256 * R;   // [Vr][G][2]
    if (has_item) {
        rest[2 * (ir * G + ig)] = accR[kRounds];
        rest[2 * (ir * G + ig) + 1] = accI[kRounds];
    }
    __syncthreads();
    for (int s = tid; s < a.nshell; s += kObsThreads) {
        double cs = 0.0, sn = 0.0;
        const int v0 = a.shell_off[s], v1 = a.shell_off[s + 1];
        for (int v = v0; v < v1; v++) {
            if (v < 256 * R) {
                cs += part[2 * v];
                sn += part[2 * v + 1];
            } else {
                const double* p = rest + 2 * (v - 256 * R) * G;
                double pc = 0.0, ps = 0.0;
                for (int g = 0; g < G; g++) {
                    pc += p[2 * g];
                    ps += p[2 * g + 1];
                }
                cs += pc;
                sn += ps;
            }
        }
        a.sk_w[w * a.nshell + s] = (cs * cs + sn * sn) / ((double)N * (double)(v1 - v0));
    }
    if (a.gr_w)
        for (int b = tid; b < a.count; b += kObsThreads) a.gr_w[w * a.count + b] = (double)cnt[b] * a.scale[b];
    if constexpr (!SHARED) add_counts(a, cnt, tid);
}

template <typename T, int D, bool SHARED>
__global__ __launch_bounds__(kObsThreads) void obs_kernel(ObsArgs a)
{
    extern __shared__ __align__(16) unsigned char smem[];
    if constexpr (SHARED) {
        unsigned* cnt = obs_counts<T, D>(a, smem);
        for (int b = threadIdx.x; b < a.count; b += kObsThreads) cnt[b] = 0u;
        for (int64_t w = blockIdx.x; w < a.W; w += gridDim.x) {
            obs_walker<T, D, true>(a, w, smem);
            __syncthreads();   // the walker's LDS is free for the next one
        }
        add_counts(a, cnt, threadIdx.x);
    } else {
        obs_walker<T, D, false>(a, blockIdx.x, smem);
    }
}

// FP64 form in 2-D and 3-D.
//   S(k): rho(n) = sum_i P_i(n') Q_i(n_last), P the product of the leading
//   axes' factors and Q the last axis's power: for all vectors at once a matrix
//   product over the particles, rows (leading components, re / im), columns
//   (power, re / im), on v_mfma_f64_16x16x4 (7 x 1 tiles of 16 in 3-D, 2 x 2 in
//   2-D, for the 50 shells).  A lane forms its row's element of P from two
//   table reads and two multiply-adds, and the four products of real and
//   imaginary parts combine at the end.  The thread-per-vector form read three
//   16-byte table entries for 10 instructions' work and was bound by the LDS.
//   g(r): the bin is a monotone function of the squared distance s, so its
//   boundaries in s (the exact ones, found on the host by the same square root
//   and division) decide it; an FP32 guess of the bin is it or the one below.  The
//   bins of the same s are those of floor(sqrt(s) / spacing), without the 30-odd
//   instructions of the FP64 square root and division per pair.
// N = 343 3-D, 16384 walkers, 200 bins: 3.81 -> 1.77 ms; N = 400 2-D, 8192
// walkers: 1.71 -> 0.83 ms.
typedef double double4v __attribute__((ext_vector_type(4)));
constexpr int kObsTiles = 2;   // tiles per wavefront

// nic_coord_ref where the displacement is not within 1e-6 of half the box of
// its image (there the rounding of x / L + 1/2 and the nudge decide: near is
// set, and the caller takes nic_coord_ref).  One multiply-add, as the compiler
// makes of nic_coord_ref's x - k L: past one box it rounds once, and a pair whose
// r / spacing is then an integer to the last bit can fall to either side of it.
__device__ __forceinline__ double nic_coord_fast(double x, double L, double Lr, double near_half, bool* near)
{
    const double res = __builtin_fma(-__builtin_rint(x * Lr), L, x);
    *near = *near || !(__builtin_fabs(res) < near_half);
    return res;
}

template <int D>
__global__ __launch_bounds__(kObsThreads) void obs_mfma_kernel(ObsArgs a)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int N = a.N, nm = a.nmax + 1, CS = a.chunk + 1;
    // [D][NP]: the first N / 2 particles again after the last, so that a row's
    // partners follow each other
    const int NP = N + N / 2;
    double* pos = reinterpret_cast<double*>(smem);
    // [D][nm][CS], then the product
    Cx<double>* tab = reinterpret_cast<Cx<double>*>(pos + (((size_t)D * NP + 1) & ~(size_t)1));
    const size_t ntab = obs_mfma_table(D, nm, CS, a.npair);
    double* thr = reinterpret_cast<double*>(tab + ntab);             // [count + 1]
    unsigned* cnt = reinterpret_cast<unsigned*>(thr + a.count + 1);  // [count]

    for (int b = tid; b <= a.count; b += kObsThreads) thr[b] = a.thr[b];
    for (int b = tid; b < a.count; b += kObsThreads) cnt[b] = 0u;
    for (int64_t w = blockIdx.x; w < a.W; w += gridDim.x) {
        const double* Rw = a.R + w * (int64_t)N * D;
        for (int e = tid; e < N * D; e += kObsThreads) {
            const int i = e / D, c = e - i * D;
            const double v = Rw[e];
            pos[c * NP + i] = v;
            if (i < N / 2) pos[c * NP + N + i] = v;
        }
        __syncthreads();

        // ------------------------------------------------------------ g(r), rows and segments as in
        // obs_kernel, consecutive threads in consecutive rows
        {
            const int M = (N - 1) / 2;
            const int even = (N % 2 == 0) ? 1 : 0;
            const int S = a.gr_segs;
            const int seg = (M + even + S - 1) / S;
            const double smax = thr[a.count], near_half = a.L * 0.499999;
            // a little low: above the FP32 rounding of the guess (under 2^-21), and
            // below one bin in 8192 by far
            const float isp = (float)((1.0 - 0x1p-20) / a.spacing);
            for (int t = tid; t < N * S; t += kObsThreads) {
                const int sg = t / N, i = t - sg * N;
                const int Mi = M + ((even && i < N / 2) ? 1 : 0);
                const int o0 = sg * seg, o1 = min(Mi, o0 + seg);
                double ri[D];
#pragma unroll
                for (int c = 0; c < D; c++) ri[c] = pos[c * NP + i];
                auto pair = [&](int j) {
                    double s;
                    {
                        // the reference's minimum image and sum of squares, without fused multiply-adds
#pragma clang fp contract(off)
                        double x[D], d[D];
                        bool near = false;
#pragma unroll
                        for (int c = 0; c < D; c++) {
                            x[c] = ri[c] - pos[c * NP + j];
                            d[c] = nic_coord_fast(x[c], a.L, a.Lr, near_half, &near);
                        }
                        if (__builtin_amdgcn_ballot_w64(near)) {
                            asm volatile("" ::: "memory");
#pragma unroll
                            for (int c = 0; c < D; c++) d[c] = nic_coord_ref(x[c], a.L, a.Lr);
                        }
                        s = d[0] * d[0];
                        if constexpr (D > 1) s += d[1] * d[1];
                        if constexpr (D > 2) s += d[2] * d[2];
                    }
                    if (s < smax) {
                        const int guess = (int)(__builtin_amdgcn_sqrtf((float)s) * isp);   // the bin or the one below it
                        atomicAdd(cnt + guess + (s >= thr[guess + 1] ? 1 : 0), 1u);
                    }
                };
                for (int j = i + 1 + o0; j < i + 1 + o1; j++) pair(j);
            }
        }

        // ------------------------------------------------------------ S(k)
        // tile q of this wave: rows 16 (q / nt) .. of the leading components, columns
        // 16 (q mod nt) .. of the powers; row 2 p + part, column 2 m + part
        const int mt = (2 * a.npair + 15) / 16, nt = (2 * nm + 15) / 16, ntile = mt * nt;
        const int r16 = lane & 15, kk = lane >> 4;
        // (row: re  x.re y.re - x.im y.im, im  x.re y.im + x.im y.re: the two parts of y
        // are read in the row's order, the sign goes to the second)
        const Cx<double>* rowx[kObsTiles];
        const double* rowf[kObsTiles];
        const double* rowg[kObsTiles];
        const double* col[kObsTiles];
        double4v acc[kObsTiles];
#pragma unroll
        for (int u = 0; u < kObsTiles; u++) {
            const int q = min(wave + 4 * u, ntile - 1);
            const int p = min((16 * (q / nt) + r16) >> 1, a.npair - 1);   // rows past the last repeat it, unused
            const int m = min((16 * (q % nt) + r16) >> 1, nm - 1);
            rowx[u] = tab + (size_t)a.pairs[2 * p] * CS + kk;
            const Cx<double>* y = D == 2 ? rowx[u] : tab + (size_t)(nm + a.pairs[2 * p + 1]) * CS + kk;
            rowf[u] = &y->re + (r16 & 1);
            rowg[u] = &y->re + 1 - (r16 & 1);
            col[u] = &tab[((size_t)(D - 1) * nm + m) * CS + kk].re + (r16 & 1);
            acc[u] = double4v{0.0, 0.0, 0.0, 0.0};
        }
        const unsigned sign = (r16 & 1) ? 0u : 0x80000000u;
        for (int c0 = 0; c0 < N; c0 += a.chunk) {
            const int nc = min(a.chunk, N - c0), nz = (nc + 15) & ~15;
            __syncthreads();   // previous chunk's table reads are done
            for (int e = tid; e < nz * D; e += kObsThreads) {
                const int il = e / D, c = e - il * D;
                Cx<double>* t = tab + (size_t)c * nm * CS + il;   // power m at t[m * CS]
                Cx<double> pw{0.0, 0.0}, e1{0.0, 0.0};            // particles past the last add nothing
                if (il < nc) {
                    double x = pos[c * NP + c0 + il] * a.Lr;
                    x -= __builtin_floor(x);
                    Prec<double>::sincos_rev(x, &e1.im, &e1.re);
                    pw.re = 1.0;
                }
                for (int m = 0; m < nm; m++) {
                    t[(size_t)m * CS] = pw;
                    pw = cmul(pw, e1);
                }
            }
            __syncthreads();
#pragma unroll
            for (int u = 0; u < kObsTiles; u++) {
                if (wave + 4 * u >= ntile) break;
                auto steps = [&](int s, auto count) {
#pragma unroll
                    for (int h = 0; h < 4 * decltype(count)::value; h += 4) {
                        double v = rowf[u][2 * (s + h)];
                        if constexpr (D == 3) {
                            const Cx<double> x = rowx[u][s + h];
                            const double g = rowg[u][2 * (s + h)];
                            const double gs = __hiloint2double(__double2hiint(g) ^ sign, __double2loint(g));
                            v = __builtin_fma(x.re, v, x.im * gs);
                        }
                        acc[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(v, col[u][2 * (s + h)], acc[u], 0, 0, 0);
                    }
                };
                int s = 0;
                for (; s + 64 <= nz; s += 64) steps(s, std::integral_constant<int, 16>());
                for (; s < nz; s += 16) steps(s, std::integral_constant<int, 4>());
            }
        }
        __syncthreads();
        double* prod = reinterpret_cast<double*>(tab);   // [16 mt][16 nt + 1]
        const int ld = 16 * nt + 1;
#pragma unroll
        for (int u = 0; u < kObsTiles; u++) {
            const int q = wave + 4 * u;
            if (q >= ntile) break;
#pragma unroll
            for (int v = 0; v < 4; v++) prod[(16 * (q / nt) + 4 * v + kk) * ld + 16 * (q % nt) + r16] = acc[u][v];
        }
        __syncthreads();
        for (int s = tid; s < a.nshell; s += kObsThreads) {
            double cs = 0.0, sn = 0.0;
            const int v0 = a.shell_off[s], v1 = a.shell_off[s + 1];
            for (int v = v0; v < v1; v++) {
                const int p = a.kvec[4 * v + 3], m = a.kvec[4 * v + D - 1];
                const double* re = prod + (2 * p) * ld + 2 * m;
                const double* ip = re + ld;
                cs += re[0] - ip[1];
                sn += re[1] + ip[0];
            }
            a.sk_w[w * a.nshell + s] = (cs * cs + sn * sn) / ((double)N * (double)(v1 - v0));
        }
        if (a.gr_w)
            for (int b = tid; b < a.count; b += kObsThreads) a.gr_w[w * a.count + b] = (double)cnt[b] * a.scale[b];
        __syncthreads();   // the walker's LDS is free for the next one
    }
    add_counts(a, cnt, tid);
}

// acc[s] += sum over walkers of sk_w[w][s], in a fixed order: one workgroup
// per shell, a strided sum per thread, then a tree.
__global__ __launch_bounds__(kObsThreads) void obs_reduce_kernel(const double* __restrict__ sk_w, int64_t W,
                                                                  int nshell, double* __restrict__ acc)
{
    __shared__ double red[kObsThreads];
    const int s = blockIdx.x, tid = threadIdx.x;
    double v = 0.0;
    for (int64_t w = tid; w < W; w += kObsThreads) v += sk_w[w * nshell + s];
    red[tid] = v;
    __syncthreads();
    for (int o = kObsThreads / 2; o > 0; o >>= 1) {
        if (tid < o) red[tid] += red[tid + o];
        __syncthreads();
    }
    if (tid == 0) acc[s] += red[0];
}

}  // namespace

size_t obs_lds_bytes(int N, int D, int V, int chunk, int nmax, int count, bool fp32)
{
    const size_t cx = fp32 ? 2 * sizeof(float) : 2 * sizeof(double);
    const int R = V >> 8, Vr = V & 255, G = Vr ? 256 / Vr : 0;
    return (size_t)N * 4 * sizeof(double) + (fp32 ? (size_t)N * 16 : 0) + 2 * (size_t)(256 * R + Vr * G) * sizeof(double) +
           (size_t)(chunk + 1) * D * (nmax + 1) * cx + (size_t)count * sizeof(unsigned);
}

// Workgroups.  One walker each from N = alone on (or where each walker's g(r) is
// asked for): the pair loop hides the additions to the totals, and the last
// workgroups leave no CU waiting (N = 343, 16384 walkers: 1774 us, 1960 with 16
// walkers each; the 1-D FP64 form from N = 100: N = 166, 10615 walkers 452 us, 537
// shared), and of few walkers, which would wait for the workgroups that have
// two: up to 1024 in FP64 and, for the more registers of its shared kernel, up to
// 1152 and 1280 in the 2-D and 3-D mixed form.  Shared and single, us: FP64 3-D, N = 8,
// 1060 walkers 22.8 / 26.4; mixed 1-D, N = 50, 1060 walkers 24.3 / 29.7; 2-D, N = 50,
// 1060 walkers 28.0 / 27.1, 1200 walkers 27.6 / 29.4; 3-D, N = 24, 1060 walkers 34.0 /
// 29.0, 1280 walkers 32.8 / 32.1, 1400 walkers 31.2 / 34.1.  Otherwise 1024
// workgroups, at most 1024 walkers each (their counts have 32 bits).
static unsigned obs_grid(int N, int64_t W, bool per_walker, int alone, int few)
{
    if (per_walker || N >= alone || W <= few) return (unsigned)W;
    return (unsigned)std::max<int64_t>(1024, (W + 1023) / 1024);
}
constexpr int kMfmaAlone = 200, kMfmaFew = 1024;

// A workgroup of one walker with few pairs spends more on staging the bins'
// thresholds than its pairs save: N = 12, 1000 bins, 192 walkers 11.7 us without,
// 13.8 with them; N = 5, 808 walkers 17.4 and 20.4; N = 19 (1000 bins) and N = 5 (50
// bins) are even.
bool obs_mfma_pays(int N, int count, int64_t W, bool per_walker)
{
    return (int64_t)obs_grid(N, W, per_walker, kMfmaAlone, kMfmaFew) < W || 3LL * N * (N - 1) >= count;
}

size_t obs_mfma_lds_bytes(int N, int D, int chunk, int nmax, int count, int npair)
{
    const int nm = nmax + 1;
    if (D < 2 || ((2 * npair + 15) / 16) * ((2 * nm + 15) / 16) > 4 * kObsTiles || chunk % 16) return 0;
    return (((size_t)D * (N + N / 2) + 1) & ~(size_t)1) * sizeof(double) +
           obs_mfma_table(D, nm, chunk + 1, npair) * sizeof(Cx<double>) +
           (size_t)(count + 1) * sizeof(double) + (size_t)count * sizeof(unsigned);
}

hipError_t launch_obs_mfma(const ObsArgs& a, int D, size_t lds, hipStream_t st)
{
    if (a.W <= 0) return hipSuccess;
    const dim3 grid(obs_grid(a.N, a.W, a.gr_w, kMfmaAlone, kMfmaFew)), block(kObsThreads);
    if (D == 2)
        hipLaunchKernelGGL(obs_mfma_kernel<2>, grid, block, lds, st, a);
    else
        hipLaunchKernelGGL(obs_mfma_kernel<3>, grid, block, lds, st, a);
    return hipGetLastError();
}

template <typename T, int D>
static void launch_obs_d(const ObsArgs& a, size_t lds, hipStream_t st)
{
    constexpr bool f32 = sizeof(T) == 4;
    const unsigned grid = obs_grid(a.N, a.W, a.gr_w, f32 ? 200 : 100, f32 ? 1024 + 128 * (D - 1) : 1024);
    if (grid < a.W)
        hipLaunchKernelGGL((obs_kernel<T, D, true>), dim3(grid), dim3(kObsThreads), lds, st, a);
    else
        hipLaunchKernelGGL((obs_kernel<T, D, false>), dim3(grid), dim3(kObsThreads), lds, st, a);
}
template <typename T>
hipError_t launch_obs(const ObsArgs& a, int D, size_t lds, hipStream_t st)
{
    if (a.W <= 0) return hipSuccess;
    switch (D) {
    case 1: launch_obs_d<T, 1>(a, lds, st); break;
    case 2: launch_obs_d<T, 2>(a, lds, st); break;
    default: launch_obs_d<T, 3>(a, lds, st); break;
    }
    return hipGetLastError();
}

hipError_t launch_obs_reduce(const double* sk_w, int64_t W, int nshell, double* acc, hipStream_t st)
{
    if (W <= 0 || nshell <= 0) return hipSuccess;
    hipLaunchKernelGGL(obs_reduce_kernel, dim3(nshell), dim3(kObsThreads), 0, st, sk_w, W, nshell, acc);
    return hipGetLastError();
}

template hipError_t launch_obs<float>(const ObsArgs&, int, size_t, hipStream_t);
template hipError_t launch_obs<double>(const ObsArgs&, int, size_t, hipStream_t);

}  // namespace tdvmc
