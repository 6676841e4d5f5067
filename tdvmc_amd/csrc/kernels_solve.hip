// FP64 TDVP solve in one workgroup: S alpha-dot = b for the real and the
// imaginary right-hand side, phi-dot.
//
// Restates src/TDVMC.cpp:1506-1537 (right-hand sides from the moments, with
// the real/imaginary-time conventions), :1684-1701 (optional diagonal
// scaling), :1703-1711 (S += eps I), :1560-1592 (lower Cholesky; a
// non-positive pivot is counted and leaves the diagonal entry at its
// unreduced value), :1594-1622 (forward / back substitution), :1658-1682
// (phi-dot, computed on the scaled solution before the scaling is undone, as
// in :1749-1758).  Solver type 1 is the full-pivot QR kernel further down.
//
// Blocked right-looking Cholesky: one wavefront factors the NB x NB diagonal
// block in registers, one thread per row solves the rows below it against that
// block in LDS (row-major at a padded stride), and the trailing lower triangle
// is updated in 16 x 16 tiles on FP64 MFMA.  The factor lives in the work
// buffer, with 1 / L[c][c] on its diagonal so that the solves only multiply.
// solve_ahead_body (NB = 16, the systems up to P = 340) holds two panels and
// the right-hand sides in LDS and lets steps of neighbouring panels run side by
// side; solve_body (NB = 32, or 16 for the largest) needs one panel only.

#include <algorithm>
#include <type_traits>
#include <utility>

#include "common.hpp"
#include "kernels.hpp"

namespace tdvmc {

namespace {

constexpr int kThreads = 1024;
// solve_ahead_body: block width, LDS stride of a panel row, 64-entry pieces of a
// row that the back substitution loads ahead, the largest system it is used for
constexpr int kNB = 16, kLDP = kNB + 1, kRowPieces = 6, kAheadMaxP = 340;
static_assert(kAheadMaxP <= 64 * kRowPieces + kNB, "the back substitution holds a whole row");

typedef double double4v __attribute__((ext_vector_type(4)));

// (r, c) of the elements e = e0, e0 + kThreads, e0 + 2 kThreads, ... of a
// column-major range with `rows` rows, stepped without a division per element
struct Walk2 {
    int r, c, dr, dc, rows;
    __device__ Walk2(int e0, int rows_) : rows(rows_)
    {
        c = e0 / rows;
        r = e0 - c * rows;
        dc = kThreads / rows;
        dr = kThreads - dc * rows;
    }
    __device__ void next()
    {
        r += dr;
        c += dc;
        if (r >= rows) {
            r -= rows;
            c++;
        }
    }
};

__device__ double block_reduce(double v, double* red)
{
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) red[wv] = v;
    __syncthreads();
    double s = 0.0;
    for (int w = 0; w < kThreads / 64; w++) s += red[w];
    return s;
}

template <int NB>
__device__ __forceinline__ void solve_body(const SolveArgs& a)
{
    const int P = a.P, tid = threadIdx.x;
    const int lane = tid & 63, wv = tid >> 6;
    double* Lm = a.work;                 // column-major P x P: Lm[j * P + i] = L[i][j]
    double* bR = a.work + (size_t)P * P;
    double* bI = bR + P;
    double* sc = bI + P;
    double* dorig = sc + P;              // diagonal after scaling and the eps shift
    extern __shared__ __align__(16) unsigned char smem[];
    double* pan = reinterpret_cast<double*>(smem);   // [rows below][NB + 1] panel; [NB][NB] blocks in the solves
    __shared__ double red[kThreads / 64];
    __shared__ double ipiv[NB];          // 1 / L[c][c]
    __shared__ double ldc[NB * NB];      // diagonal block, column-major: ldc[c * NB + k] = L[k][c]
    __shared__ int nbad;
    const double* mO = a.mean;
    const double eR = a.mean[P], eI = a.mean[P + 1];
    const double* FR = a.F;
    const double* FI = a.F + P;

    if (tid == 0) nbad = 0;
    for (int i = tid; i < P; i += kThreads) {
        if (a.imag_time == 0) {
            bR[i] = FI[i];
            bI[i] = -FR[i];
        } else {
            bR[i] = -FR[i];
            bI[i] = -(FI[i] + mO[i] * eI);
        }
        sc[i] = a.precondition ? sqrt(a.S[(size_t)i * P + i]) : 1.0;
    }
    __syncthreads();
    // S is symmetric: read it column by column (coalesced), four entries in flight per thread
    const size_t PP = (size_t)P * P;
    Walk2 wk(tid, P);   // (row, column) of e0, stepped along with it
    for (size_t e0 = tid; e0 < PP; e0 += 4 * kThreads) {
        double v[4];
        int ri[4], ci[4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const size_t e = e0 + (size_t)q * kThreads;
            v[q] = e < PP ? a.S[e] : 0.0;
            ri[q] = wk.r;
            ci[q] = wk.c;
            wk.next();
        }
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const size_t e = e0 + (size_t)q * kThreads;
            if (e >= PP) continue;
            const int i = ri[q], j = ci[q];
            double x = v[q];
            if (a.precondition) x /= (sc[i] * sc[j]);
            if (i == j) {
                x += a.eps;
                dorig[i] = x;
            }
            Lm[e] = x;
        }
    }
    for (int i = tid; i < P; i += kThreads) {
        if (a.precondition) {
            bR[i] /= sc[i];
            bI[i] /= sc[i];
        }
    }
    __syncthreads();

    // ---------------------------------------------------------------- Cholesky
    // The rows below the diagonal block sit in LDS row-major with a padded
    // stride (pan[rb * LDP + c], LDP = NB + 1): a thread's row is read with
    // immediate offsets, and only threads rb and rb + 32 share a bank.  The
    // diagonal block is staged on its own, column-major and padded with the
    // identity to NB x NB (ldc[c * NB + l] = A[l][c]): padded columns have
    // pivot 1 and zero off-diagonal entries and leave the real rows unchanged,
    // so no step below has a run-time bound on the block.  Only the last
    // block can be partial, and it has no rows below it.
    constexpr int LDP = NB + 1;
    for (int p0 = 0; p0 < P; p0 += NB) {
        const int nb = min(NB, P - p0);
        const int below = P - p0 - nb;
        if (below > 0) {
            Walk2 wk2(tid, below);
            for (int e = tid; e < nb * below; e += kThreads) {
                pan[wk2.r * LDP + wk2.c] = Lm[(size_t)(p0 + wk2.c) * P + p0 + nb + wk2.r];
                wk2.next();
            }
        }
        for (int e = tid; e < NB * NB; e += kThreads) {
            const int c = e / NB, l = e % NB;
            ldc[e] = (c < nb && l < nb) ? Lm[(size_t)(p0 + c) * P + p0 + l] : (c == l ? 1.0 : 0.0);
        }
        __syncthreads();
        // diagonal block by one wavefront in registers: lane l holds row
        // l mod NB, column entries reach the other lanes by v_readlane.  Every
        // lane updates its whole row (the entries above the diagonal are
        // never read), and the diagonal gets 1 / L[c][c] from ipiv at the end.
        if (wv == 0) {
            const int l = lane & (NB - 1);
            double av[NB];
#pragma unroll
            for (int k = 0; k < NB; k++) av[k] = ldc[k * NB + l];
#pragma unroll
            for (int c = 0; c < NB; c++) {
                const double d = readlane_f(av[c], c);
                double ipj;
                if (d > 0.0) {
                    // 1 / sqrt(d) from the hardware estimate and two Newton
                    // steps (each squares the relative error): a shorter
                    // dependent chain than a correctly rounded sqrt and a
                    // divide, within an ulp or two of their quotient
                    double y = __builtin_amdgcn_rsq(d);
                    const double hd = 0.5 * d;
                    y = y * (1.5 - hd * y * y);
                    y = y * (1.5 - hd * y * y);
                    ipj = y;
                } else {
                    // the unreduced diagonal entry stands in as the pivot
                    ipj = 1.0 / dorig[p0 + c];
                    if (lane == 0) nbad++;
                }
                av[c] *= ipj;
                if (lane == 0) ipiv[c] = ipj;
#pragma unroll
                for (int k = c + 1; k < NB; k++) av[k] -= av[c] * readlane_f(av[c], k);
                // one column's lane reads at a time (scalar registers)
                __builtin_amdgcn_sched_barrier(0);
            }
            if (lane < NB) {
#pragma unroll
                for (int k = 0; k < NB; k++) ldc[k * NB + lane] = av[k];
                // the factor keeps 1 / L[c][c] on its diagonal: the triangular
                // solves multiply by it (same wavefront, after the writes above
                // and lane 0's ipiv writes)
                ldc[lane * NB + lane] = ipiv[lane];
            }
        }
        __syncthreads();
        // rows below the block, one thread per row, right-looking within the
        // row: L[r][c] = v_c / L[c][c], then v_k -= L[r][c] L[k][c] for k > c
        for (int rb = tid; rb < below; rb += kThreads) {
            double* pr = pan + rb * LDP;
            double v[NB];
#pragma unroll
            for (int k = 0; k < NB; k++) v[k] = pr[k];
#pragma unroll
            for (int c = 0; c < NB; c++) {
                const double xc = v[c] * ipiv[c];
                pr[c] = xc;
                const double* lcol = ldc + c * NB;   // L[k][c]
#pragma unroll
                for (int k = c + 1; k < NB; k++) v[k] -= xc * lcol[k];
                // keeps the 32 columns' table reads from being hoisted together (register spills)
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        __syncthreads();
        {
            Walk2 wk3(tid, nb + below);
            for (int e = tid; e < nb * (nb + below); e += kThreads) {
                const int c = wk3.c, r = wk3.r;
                if (r >= c)
                    Lm[(size_t)(p0 + c) * P + p0 + r] = r < nb ? ldc[c * NB + r] : pan[(r - nb) * LDP + c];
                wk3.next();
            }
        }
        // trailing update of the lower triangle, A[i][k] -= sum_c L[i][c] L[k][c],
        // on FP64 MFMA in 16 x 16 tiles spread over the wavefronts: lane 16 kk + pp
        // holds L[16 K + pp][4 s + kk] as the A operand and L[16 I + pp][4 s + kk]
        // as the B operand, so acc[v] sums row i = 16 I + pp, column
        // k = 16 K + 4 v + kk, and consecutive lanes update consecutive rows of the
        // column-major factor.  The old entries are loaded before the MFMA chain.
        // Rows past the end of the panel are read (inside the LDS allocation) but
        // their sums are not stored.
        if (below > 0) {
            const int n16 = (below + 15) / 16;
            const int ntiles = n16 * (n16 + 1) / 2;
            const size_t q0 = (size_t)(p0 + nb);   // first trailing row / column
            const int pp = lane & 15, kk = lane >> 4;
            for (int t = wv; t < ntiles; t += kThreads / 64) {
                int ti = (int)((sqrt(8.0 * t + 1.0) - 1.0) * 0.5);
                while (ti * (ti + 1) / 2 > t) ti--;
                while ((ti + 1) * (ti + 2) / 2 <= t) ti++;
                const int tk = t - ti * (ti + 1) / 2;   // tile (ti, tk), tk <= ti
                const int i = 16 * ti + pp;
                double old[4];
                bool ok[4];
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int k = 16 * tk + 4 * v + kk;
                    ok[v] = i < below && k <= i;
                    old[v] = ok[v] ? Lm[(q0 + k) * P + q0 + i] : 0.0;
                }
                const double* pa = pan + (16 * tk + pp) * LDP + kk;   // rows k
                const double* pb = pan + (16 * ti + pp) * LDP + kk;   // rows i
                double4v acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int s4 = 0; s4 < NB / 4; s4++)
                    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(pa[4 * s4], pb[4 * s4], acc, 0, 0, 0);
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int k = 16 * tk + 4 * v + kk;
                    if (ok[v]) Lm[(q0 + k) * P + q0 + i] = old[v] - acc[v];
                }
            }
        }
        __syncthreads();
    }

    // ---------------------------------------------------------------- L t = b
    for (int p0 = 0; p0 < P; p0 += NB) {
        const int nb = min(NB, P - p0);
        // diagonal block into LDS: pan[j * NB + l] = L[p0 + l][p0 + j]
        for (int e = tid; e < nb * nb; e += kThreads) {
            const int j = e / nb, l = e % nb;
            pan[j * NB + l] = Lm[(size_t)(p0 + j) * P + p0 + l];
        }
        __syncthreads();
        if (wv == 0) {
            // lane l owns row p0 + l; the diagonal holds 1 / L[j][j]
            double tR = lane < nb ? bR[p0 + lane] : 0.0, tI = lane < nb ? bI[p0 + lane] : 0.0;
            for (int j = 0; j < nb; j++) {
                const double rjj = pan[j * NB + j];
                const double xR = readlane_f(tR, j) * rjj, xI = readlane_f(tI, j) * rjj;
                if (lane == j) {
                    tR = xR;
                    tI = xI;
                } else if (lane > j && lane < nb) {
                    const double l = pan[j * NB + lane];
                    tR -= l * xR;
                    tI -= l * xI;
                }
            }
            if (lane < nb) {
                bR[p0 + lane] = tR;
                bI[p0 + lane] = tI;
            }
        }
        __syncthreads();
        for (int i = p0 + nb + tid; i < P; i += kThreads) {
            double sR = 0.0, sI = 0.0;
#pragma unroll 8
            for (int j = 0; j < nb; j++) {
                const double l = Lm[(size_t)(p0 + j) * P + i];
                sR += l * bR[p0 + j];
                sI += l * bI[p0 + j];
            }
            bR[i] -= sR;
            bI[i] -= sI;
        }
        __syncthreads();
    }

    // ---------------------------------------------------------------- L^T x = t
    const int npan = (P + NB - 1) / NB;
    for (int pb = npan - 1; pb >= 0; pb--) {
        const int p0 = pb * NB, nb = min(NB, P - p0), pe = p0 + nb;
        // t_i -= sum_{j >= pe} L[j][i] x_j for the panel's rows (one wave per row group)
        for (int i = p0 + wv; i < pe; i += kThreads / 64) {
            double sR = 0.0, sI = 0.0;
            for (int j = pe + lane; j < P; j += 64) {
                const double l = Lm[(size_t)i * P + j];
                sR += l * bR[j];
                sI += l * bI[j];
            }
            for (int o = 32; o > 0; o >>= 1) {
                sR += __shfl_xor(sR, o, 64);
                sI += __shfl_xor(sI, o, 64);
            }
            if (lane == 0) {
                bR[i] -= sR;
                bI[i] -= sI;
            }
        }
        // diagonal block into LDS: pan[j * NB + l] = L[p0 + l][p0 + j]
        for (int e = tid; e < nb * nb; e += kThreads) {
            const int j = e / nb, l = e % nb;
            pan[j * NB + l] = Lm[(size_t)(p0 + j) * P + p0 + l];
        }
        __syncthreads();
        if (wv == 0) {
            double tR = lane < nb ? bR[p0 + lane] : 0.0, tI = lane < nb ? bI[p0 + lane] : 0.0;
            for (int j = nb - 1; j >= 0; j--) {
                const double rjj = pan[j * NB + j];
                const double xR = readlane_f(tR, j) * rjj, xI = readlane_f(tI, j) * rjj;
                if (lane == j) {
                    tR = xR;
                    tI = xI;
                } else if (lane < j) {
                    const double l = pan[lane * NB + j];   // L[j][lane]
                    tR -= l * xR;
                    tI -= l * xI;
                }
            }
            if (lane < nb) {
                bR[p0 + lane] = tR;
                bI[p0 + lane] = tI;
            }
        }
        __syncthreads();
    }

    // phi-dot on the (scaled) solution, then undo the scaling
    double pr = 0.0, pi = 0.0;
    for (int i = tid; i < P; i += kThreads) {
        pr -= mO[i] * bR[i];
        pi -= mO[i] * bI[i];
    }
    pr = block_reduce(pr, red);
    pi = block_reduce(pi, red);
    for (int i = tid; i < P; i += kThreads) {
        a.xdot[i] = bR[i] / sc[i];
        a.xdot[P + i] = bI[i] / sc[i];
    }
    if (tid == 0) {
        if (a.imag_time == 0)
            pi -= eR;
        else
            pr -= eR;
        a.xdot[2 * P] = pr;
        a.xdot[2 * P + 1] = pi;
        if (a.status) a.status[0] += nbad;
    }
}

// ---------------------------------------------------------------------------
// The same solve where two panels and the right-hand sides fit the LDS.  One
// workgroup's solve is a chain of short dependent steps, not of work (8.6
// MFLOP at P = 296), so the steps that need not follow each other run side by
// side:
//   - the trailing update's first tile column goes straight into the LDS of
//     the next panel (no store, reload and staging), then one wavefront
//     factors the next diagonal block while the others update the rest;
//   - the right-hand sides are two more rows under the matrix: L t = b is done
//     with the factorisation;
//   - in L^T x = t a wavefront has its row's entries of the factor loaded
//     before the blocks that they meet are solved;
//   - S is not copied: the first panel's update reads it in place.
// The operations on each number and their order are those of solve_body with 16
// columns, so both give the same bits.
// At P = 32, 13 us against 27 without these; at P = 296, 152 against 373 us, of
// which the matrix unit's work on one CU is about 35 us and the rest the
// chains of the 19 diagonal blocks, row solves and back substitutions (about 5
// us a block) and the trailing tiles' loads (two tiles' or four tiles' entries
// under way instead of one: no faster).
// rows of the first panel buffer: the rows below the first block, in whole
// tiles (the second buffer holds a tile less); never less than the back
// substitution's diagonal blocks need
__host__ __device__ inline int ahead_rows(int P) { return P > 3 * kNB ? (P - kNB + 15) / 16 * 16 : 32; }

template <int CTRL>
__device__ __forceinline__ double row_dpp(double x)
{
    const int2 v = __builtin_bit_cast(int2, x);
    int2 r;
    r.x = __builtin_amdgcn_update_dpp(0, v.x, CTRL, 0xf, 0xf, true);
    r.y = __builtin_amdgcn_update_dpp(0, v.y, CTRL, 0xf, 0xf, true);
    return __builtin_bit_cast(double, r);
}
// x of lane C of every 16 lanes (DPP row broadcast): the value stays in vector
// registers, so there is no wait between the read and its use
template <int C>
__device__ __forceinline__ double row_bcast(double x) { return row_dpp<0x150 + C>(x); }
// the sum over the wavefront, as a butterfly over 32, 16, .. 1 gives it (from 8
// down the halves are alike, and rotating a row is the exchange)
__device__ __forceinline__ double wave_sum(double x)
{
    x += __shfl_xor(x, 32, 64);
    x += __shfl_xor(x, 16, 64);
    x += row_dpp<0x128>(x);
    x += row_dpp<0x124>(x);
    x += row_dpp<0x122>(x);
    return x + row_dpp<0x121>(x);
}
template <typename F, int... I>
__device__ __forceinline__ void each_of(F f, std::integer_sequence<int, I...>)
{
    (f(std::integral_constant<int, I>{}), ...);
}
// f(0), f(1), .. f(N - 1) with constant arguments
template <int N, typename F>
__device__ __forceinline__ void static_for(F f) { each_of(f, std::make_integer_sequence<int, N>{}); }

// Diagonal block d[c * 16 + l] = A[l][c] (l >= c; identity past the matrix)
// factored in place by one wavefront (every 16 lanes alike), 1 / L[c][c] on the
// diagonal; rd is the reciprocal of the lane's unreduced diagonal entry.  The
// next column's pivot is worked out beside the rest of a column's updates.
// Returns the number of non-positive pivots.
__device__ __forceinline__ int factor_block(double* d, double rd, int lane)
{
    const int l = lane & (kNB - 1);
    double av[kNB], own = 0.0;
#pragma unroll
    for (int k = 0; k < kNB; k++) av[k] = d[k * kNB + l];
    int bad = 0;
    auto pivot = [&](auto c) {
        // 1 / sqrt(x) as in solve_body; where x is not positive the unreduced
        // diagonal entry stands in as the pivot
        const double x = row_bcast<c>(av[c]), hx = 0.5 * x, alt = row_bcast<c>(rd);
        double y = __builtin_amdgcn_rsq(x);
        y = y * (1.5 - hx * y * y);
        y = y * (1.5 - hx * y * y);
        bad += x > 0.0 ? 0 : 1;
        return x > 0.0 ? y : alt;
    };
    double r = pivot(std::integral_constant<int, 0>{});
    static_for<kNB>([&](auto c) {
        av[c] *= r;
        own = l == c ? r : own;
        if constexpr (c + 1 < kNB) {
            av[c + 1] -= av[c] * row_bcast<c + 1>(av[c]);
            r = pivot(std::integral_constant<int, c + 1>{});
        }
        static_for<kNB>([&](auto k) {
            if constexpr (k > c + 1) av[k] -= av[c] * row_bcast<k>(av[c]);
        });
        __builtin_amdgcn_sched_barrier(0);
    });
    if (lane < kNB) {
#pragma unroll
        for (int k = 0; k < kNB; k++) d[k * kNB + lane] = av[k];
        d[lane * kNB + lane] = own;
    }
    return bad;
}

__device__ __forceinline__ void solve_ahead_body(const SolveArgs& a)
{
    const int P = a.P, tid = threadIdx.x;
    const int lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr int NW = kThreads / 64;
    static_assert(NW == kNB, "a wavefront per column of the first panel");
    // Column-major with LD = P rounded up to whole tiles: Lm[j * LD + i] is
    // A[i][j], later L[i][j].  No step of the update has an edge to look at;
    // rows and columns past the matrix reach no other ones.
    const int LD = (P + kNB - 1) / kNB * kNB;
    double* Lm = a.work;
    double* sc = a.work + (size_t)LD * LD;
    double* rdiag = sc + LD;             // reciprocal of the diagonal after scaling and the eps shift
    extern __shared__ __align__(16) unsigned char smem[];
    const int cap = ahead_rows(P);
    double* pan0 = reinterpret_cast<double*>(smem);   // [cap][kLDP], [cap - 16][kLDP]
    double* bl = pan0 + (size_t)(2 * cap - kNB) * kLDP;   // [2][LD] right-hand sides, then t, then x
    __shared__ double ldc[2][kNB * kNB];              // diagonal blocks, column-major
    __shared__ double red[NW];
    __shared__ int nbad;
    const double* mO = a.mean;
    const double eR = a.mean[P], eI = a.mean[P + 1];

    if (tid == 0) nbad = 0;
    for (int i = tid; i < LD; i += kThreads) {
        double r = 0.0, m = 0.0;
        if (i < P) {
            const double sii = a.S[(size_t)i * P + i];
            const double s = a.precondition ? sqrt(sii) : 1.0;
            if (a.imag_time == 0) {
                r = a.F[P + i];
                m = -a.F[i];
            } else {
                r = -a.F[i];
                m = -(a.F[P + i] + mO[i] * eI);
            }
            sc[i] = s;
            if (a.precondition) {
                r /= s;
                m /= s;
            }
            rdiag[i] = 1.0 / ((a.precondition ? sii / (s * s) : sii) + a.eps);
        }
        bl[i] = r;
        bl[LD + i] = m;
    }
    __syncthreads();
    // entry of the scaled and shifted matrix, row r of column c <= r (S is
    // symmetric: read along its row c)
    auto entry = [&](double x, int r, int c) {
        if (a.precondition) x /= (sc[r] * sc[c]);
        return r == c ? x + a.eps : x;
    };
    {
        const int c = min(wv, P - 1);
        for (int r0 = lane; r0 < LD; r0 += 4 * 64) {
            double v[4];
#pragma unroll
            for (int q = 0; q < 4; q++) v[q] = a.S[(size_t)c * P + min(r0 + 64 * q, P - 1)];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int r = r0 + 64 * q;
                if (r >= LD) continue;
                const double x = entry(v[q], min(r, P - 1), c);
                if (r < kNB)
                    ldc[0][wv * kNB + r] = max(r, wv) < P ? x : r == wv ? 1.0 : 0.0;
                else
                    pan0[(r - kNB) * kLDP + wv] = x;
            }
        }
    }
    __syncthreads();
    if (wv == 0) {
        const int bad = factor_block(ldc[0], lane < P ? rdiag[lane & (kNB - 1)] : 1.0, lane);
        if (lane == 0) nbad += bad;
    }
    __syncthreads();

    // ---------------------------------------------------------------- Cholesky and L t = b
    const int pp = lane & 15, kk = lane >> 4;
    const unsigned loff = kk * LD + pp;
    auto panel = [&](int p0, auto first) {
        const int cur = (p0 / kNB) & 1, nxt = cur ^ 1;
        double* pan = pan0 + (size_t)cur * cap * kLDP;
        double* pann = pan0 + (size_t)nxt * cap * kLDP;
        const double* blk = ldc[cur];
        const int q0 = p0 + kNB;                 // first trailing row / column
        const int below = max(P - q0, 0), n16 = (below + 15) / 16;
        // rows below the block, and the right-hand sides, one thread each; a
        // column of the block is read while the one before it is used
        for (int rb = tid; rb < below + 2; rb += kThreads) {
            double* pr = rb < below ? pan + rb * kLDP : bl + (rb - below) * LD + p0;
            double v[kNB], lc[2][kNB];
#pragma unroll
            for (int k = 0; k < kNB; k++) v[k] = pr[k];
#pragma unroll
            for (int k = 0; k < kNB; k++) lc[0][k] = blk[k];
#pragma unroll
            for (int c = 0; c < kNB; c++) {
#pragma unroll
                for (int k = c + 1; k < kNB; k++) lc[(c + 1) & 1][k] = blk[(c + 1) * kNB + k];
                const double xc = v[c] * lc[c & 1][c];
                pr[c] = xc;
#pragma unroll
                for (int k = c + 1; k < kNB; k++) v[k] -= xc * lc[c & 1][k];
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        __syncthreads();
        // Trailing update A[i][k] -= sum_c L[i][c] L[k][c] of tile (ti, tk):
        // lane 16 kk + pp holds rows 16 tk + pp and 16 ti + pp, entry 4 s + kk;
        // acc[v] sums row 16 ti + pp, column 16 tk + 4 v + kk (solve_body)
        auto rows = [&](int tile, double* x) {
            const double* q = pan + (16 * tile + pp) * kLDP + kk;
#pragma unroll
            for (int s4 = 0; s4 < 4; s4++) x[s4] = q[4 * s4];
        };
        auto load_old = [&](int ti, int tk, double* o) {
            if (first) {
                const int i = min(q0 + 16 * ti + pp, P - 1);
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int k = min(q0 + 16 * tk + 4 * v + kk, P - 1);
                    o[v] = entry(a.S[(size_t)k * P + i], i, k);
                }
            } else {
                const double* src = Lm + (size_t)(q0 + 16 * tk) * LD + q0 + 16 * ti;
#pragma unroll
                for (int v = 0; v < 4; v++) o[v] = (src + 4 * v * LD)[loff];
            }
        };
        auto update = [&](const double* ra, const double* rb, double* o) {
            double4v acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int s4 = 0; s4 < 4; s4++) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(ra[s4], rb[s4], acc, 0, 0, 0);
#pragma unroll
            for (int v = 0; v < 4; v++) o[v] -= acc[v];
        };
        if (wv == 0) {
            // the next diagonal block (identity past the matrix) and its factor
            if (below > 0) {
                double ra[4], o[4];
                const double rd = q0 + pp < P ? rdiag[q0 + pp] : 1.0;
                load_old(0, 0, o);
                rows(0, ra);
                update(ra, ra, o);
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int k = 4 * v + kk;
                    ldc[nxt][k * kNB + pp] = max(k, pp) < below ? o[v] : k == pp ? 1.0 : 0.0;
                }
                // the other wavefronts of its SIMD have the rest of the step to wait in
                __builtin_amdgcn_s_setprio(3);
                const int bad = factor_block(ldc[nxt], rd, lane);
                __builtin_amdgcn_s_setprio(0);
                if (lane == 0) nbad += bad;
            }
        } else {
            // the other tiles of the triangle, row by row in equal shares
            const int m = n16 * (n16 + 1) / 2 - 1;
            int t = 1 + (wv - 1) * m / (NW - 1);
            const int te = 1 + wv * m / (NW - 1);
            if (t < te) {
                int ti = (int)((sqrtf(8.0f * t + 1.0f) - 1.0f) * 0.5f);
                while (ti * (ti + 1) / 2 > t) ti--;
                while ((ti + 1) * (ti + 2) / 2 <= t) ti++;
                ti = __builtin_amdgcn_readfirstlane(ti);
                int tk = t - ti * (ti + 1) / 2;
                double o[4], on[4], ra[4], rb[4];
                load_old(ti, tk, o);
                rows(ti, rb);
                for (;;) {
                    const int ni = tk == ti ? ti + 1 : ti, nk = tk == ti ? 0 : tk + 1;
                    const bool more = t + 1 < te;
                    if (more) load_old(ni, nk, on);
                    rows(tk, ra);
                    update(ra, rb, o);
                    if (tk == 0) {
                        double* dst = pann + (16 * (ti - 1) + pp) * kLDP + kk;
#pragma unroll
                        for (int v = 0; v < 4; v++) dst[4 * v] = o[v];
                    } else {
                        double* dst = Lm + (size_t)(q0 + 16 * tk) * LD + q0 + 16 * ti;
#pragma unroll
                        for (int v = 0; v < 4; v++) (dst + 4 * v * LD)[loff] = o[v];
                    }
                    if (!more) break;
                    if (ni != ti) rows(ni, rb);
                    ti = ni;
                    tk = nk;
                    t++;
#pragma unroll
                    for (int v = 0; v < 4; v++) o[v] = on[v];
                }
            }
            // b -= L t of the rows below; the panel of the factor
            for (int e = tid - 64; e < 2 * below; e += kThreads - 64) {
                const int h = e >= below, i = h ? e - below : e;
                const double* tb = bl + h * LD + p0;
                double s = 0.0;
#pragma unroll
                for (int c = 0; c < kNB; c++) s += tb[c] * pan[i * kLDP + c];
                bl[h * LD + q0 + i] -= s;
            }
            for (int i = tid - 64; i < kNB + below; i += kThreads - 64) {
#pragma unroll
                for (int c = 0; c < kNB; c++)
                    (Lm + (size_t)(p0 + c) * LD + p0)[(unsigned)i] = i < kNB ? blk[c * kNB + i] : pan[(i - kNB) * kLDP + c];
            }
        }
        __syncthreads();
    };
    panel(0, std::true_type{});
    for (int p0 = kNB; p0 < P; p0 += kNB) panel(p0, std::false_type{});

    // ---------------------------------------------------------------- L^T x = t
    // Block by block from the last: each wavefront takes the solved part off
    // one row, then the first one solves the block (lane l holds column l below
    // the diagonal in f and 1 / L[l][l] in di; identity past the matrix), with
    // the diagonal blocks in LDS (over the panels).
    double* diag = pan0;   // [LD][kLDP]: L[p0 + j][c] of column c's block at c * kLDP + j
    for (int e = tid; e < kNB * LD; e += kThreads) {
        const int c = e / kNB, j = e % kNB;
        diag[c * kLDP + j] = Lm[(size_t)c * LD + c / kNB * kNB + j];
    }
    constexpr int NQ = kRowPieces;
    double lr[NQ];
    auto load_row = [&](int p0) {
        const double* row = Lm + (size_t)(p0 + wv) * LD + p0 + kNB;
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            if (p0 + kNB + 64 * q < P) lr[q] = row[(unsigned)min(64 * q + lane, P - 1 - kNB - p0)];
        }
    };
    __syncthreads();
    for (int p0 = LD - kNB; p0 >= 0; p0 -= kNB) {
        const int pe = p0 + kNB;
        if (pe < P) {
            double sR = 0.0, sI = 0.0;
#pragma unroll
            for (int q = 0; q < NQ; q++) {
                if (pe + 64 * q < P) {
                    const int j = pe + 64 * q + lane;
                    if (j < P) {
                        sR += lr[q] * bl[j];
                        sI += lr[q] * bl[LD + j];
                    }
                }
            }
            sR = wave_sum(sR);
            sI = wave_sum(sI);
            if (lane == 0) {
                bl[p0 + wv] -= sR;
                bl[LD + p0 + wv] -= sI;
            }
            __syncthreads();
        }
        if (p0 > 0) load_row(p0 - kNB);
        if (wv == 0) {
            const int i = p0 + pp;
            double f[kNB];
#pragma unroll
            for (int j = 0; j < kNB; j++) f[j] = diag[i * kLDP + j];
            const double di = diag[i * kLDP + pp];
            double tR = bl[i], tI = bl[LD + i], xR = 0.0, xI = 0.0;
            static_for<kNB>([&](auto jj) {
                constexpr int j = kNB - 1 - jj;
                const double uR = tR * di, uI = tI * di, fj = pp < j ? f[j] : 0.0;
                xR = pp == j ? uR : xR;
                xI = pp == j ? uI : xI;
                tR -= fj * row_bcast<j>(uR);
                tI -= fj * row_bcast<j>(uI);
            });
            if (lane < kNB) {
                bl[i] = xR;
                bl[LD + i] = xI;
            }
        }
        __syncthreads();
    }

    // phi-dot on the (scaled) solution, then undo the scaling
    double pr = 0.0, pi = 0.0;
    for (int i = tid; i < P; i += kThreads) {
        pr -= mO[i] * bl[i];
        pi -= mO[i] * bl[LD + i];
    }
    pr = block_reduce(pr, red);
    pi = block_reduce(pi, red);
    for (int i = tid; i < P; i += kThreads) {
        a.xdot[i] = bl[i] / sc[i];
        a.xdot[P + i] = bl[LD + i] / sc[i];
    }
    if (tid == 0) {
        if (a.imag_time == 0)
            pi -= eR;
        else
            pr -= eR;
        a.xdot[2 * P] = pr;
        a.xdot[2 * P + 1] = pi;
        if (a.status) a.status[0] += nbad;
    }
}

// ---------------------------------------------------------------------------
// Solver type 1 (src/TDVMC.cpp:1763-1822): Householder QR with full pivoting,
// the decomposition of Eigen::FullPivHouseholderQR, with its conventions
// (pivot = largest magnitude of the trailing block, first in column-major
// order on ties; stop when it falls to n eps of the first pivot; trailing-row
// and whole-column swaps; v = (1, tail / (c0 - beta)), tau = (beta - c0) /
// beta, beta = -sign(c0) |x|; rank from n eps max |R_kk|), then the mean of
// each solution vector is subtracted.  For an S made singular by the exactly
// equal O of k and -k this picks the same solution as the reference's
// decomposition; Cholesky would not.  The matrix is held column-major in the
// work buffer, one thread per column for the reflector updates.

__device__ void argmax_reduce(double& v, int& e, double* rv, int* re)
{
    // larger value wins, equal values: smaller column-major index
    for (int o = 32; o > 0; o >>= 1) {
        const double v2 = __shfl_xor(v, o, 64);
        const int e2 = __shfl_xor(e, o, 64);
        if (v2 > v || (v2 == v && e2 < e)) {
            v = v2;
            e = e2;
        }
    }
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) {
        rv[wv] = v;
        re[wv] = e;
    }
    __syncthreads();
    v = rv[0];
    e = re[0];
    for (int w = 1; w < kThreads / 64; w++)
        if (rv[w] > v || (rv[w] == v && re[w] < e)) {
            v = rv[w];
            e = re[w];
        }
}

__device__ __forceinline__ void solve_qr_body(const SolveArgs& a)
{
    const int P = a.P, tid = threadIdx.x;
    double* Q = a.work;                  // column-major: Q[j * P + i] = A[i][j]
    double* bR = a.work + (size_t)P * P;
    double* bI = bR + P;
    double* sc = bI + P;
    double* tau = sc + P;
    extern __shared__ __align__(16) unsigned char smem[];
    int* rt = reinterpret_cast<int*>(smem);   // row transpositions [P]
    int* ct = rt + P;                          // column transpositions [P]
    __shared__ double red[kThreads / 64];
    __shared__ double rv[kThreads / 64];
    __shared__ int re[kThreads / 64];
    const double* mO = a.mean;
    const double eR = a.mean[P], eI = a.mean[P + 1];
    const double* FR = a.F;
    const double* FI = a.F + P;
    const double prec = P * 2.220446049250313e-16;

    for (int i = tid; i < P; i += kThreads) {
        if (a.imag_time == 0) {
            bR[i] = FI[i];
            bI[i] = -FR[i];
        } else {
            bR[i] = -FR[i];
            bI[i] = -(FI[i] + mO[i] * eI);
        }
        sc[i] = a.precondition ? sqrt(a.S[(size_t)i * P + i]) : 1.0;
    }
    __syncthreads();
    Walk2 wk(tid, P);
    for (size_t e = tid; e < (size_t)P * P; e += kThreads) {
        const int i = wk.r, j = wk.c;
        wk.next();
        double v = a.S[(size_t)i * P + j];
        if (a.precondition) v /= (sc[i] * sc[j]);
        if (i == j) v += a.eps;
        Q[e] = v;
    }
    for (int i = tid; i < P; i += kThreads) {
        if (a.precondition) {
            bR[i] /= sc[i];
            bI[i] /= sc[i];
        }
    }
    __syncthreads();

    double biggest = 0.0, maxpivot = 0.0;
    int nz = P;
    for (int k = 0; k < P; k++) {
        const int m = P - k;
        double bv = -1.0;
        int be = 0x7fffffff;
        for (int e = tid; e < m * m; e += kThreads) {
            const int jj = e / m, ii = e - jj * m;   // e increases in column-major order
            const double v = fabs(Q[(size_t)(k + jj) * P + k + ii]);
            if (v > bv) {
                bv = v;
                be = e;
            }
        }
        argmax_reduce(bv, be, rv, re);
        if (k == 0) biggest = bv;
        if (bv <= biggest * prec) {
            nz = k;
            break;
        }
        const int bj = k + be / m, bi = k + be % m;
        if (tid == 0) {
            rt[k] = bi;
            ct[k] = bj;
        }
        if (bi != k)
            for (int j = k + tid; j < P; j += kThreads) {
                const double t = Q[(size_t)j * P + k];
                Q[(size_t)j * P + k] = Q[(size_t)j * P + bi];
                Q[(size_t)j * P + bi] = t;
            }
        __syncthreads();
        if (bj != k)
            for (int i = tid; i < P; i += kThreads) {
                const double t = Q[(size_t)k * P + i];
                Q[(size_t)k * P + i] = Q[(size_t)bj * P + i];
                Q[(size_t)bj * P + i] = t;
            }
        __syncthreads();
        double* col = Q + (size_t)k * P;
        double tl = 0.0;
        for (int i = k + 1 + tid; i < P; i += kThreads) tl += col[i] * col[i];
        tl = block_reduce(tl, red);
        const double c0 = col[k];
        double beta, tk;
        if (tl <= 2.2250738585072014e-308) {
            tk = 0.0;
            beta = c0;
            for (int i = k + 1 + tid; i < P; i += kThreads) col[i] = 0.0;
        } else {
            beta = sqrt(c0 * c0 + tl);
            if (c0 >= 0.0) beta = -beta;
            const double den = c0 - beta;
            for (int i = k + 1 + tid; i < P; i += kThreads) col[i] /= den;
            tk = (beta - c0) / beta;
        }
        maxpivot = fmax(maxpivot, fabs(beta));
        __syncthreads();
        if (tid == 0) {
            col[k] = beta;
            tau[k] = tk;
        }
        // H applied to the trailing columns, one thread per column
        for (int j = k + 1 + tid; j < P; j += kThreads) {
            double* cj = Q + (size_t)j * P;
            double w = cj[k];
            for (int i = k + 1; i < P; i++) w += col[i] * cj[i];
            cj[k] -= tk * w;
            for (int i = k + 1; i < P; i++) cj[i] -= (tk * col[i]) * w;
        }
        __syncthreads();
    }
    for (int k = nz + tid; k < P; k += kThreads) {
        rt[k] = k;
        ct[k] = k;
    }
    __syncthreads();
    int rank = 0;
    for (int i = 0; i < nz; i++) rank += fabs(Q[(size_t)i * P + i]) > maxpivot * prec;

    // c = Q^T (row-swapped) b for the first rank reflectors
    for (int k = 0; k < rank; k++) {
        if (tid == 0 && rt[k] != k) {
            double t = bR[k]; bR[k] = bR[rt[k]]; bR[rt[k]] = t;
            t = bI[k]; bI[k] = bI[rt[k]]; bI[rt[k]] = t;
        }
        __syncthreads();
        const double* col = Q + (size_t)k * P;
        const double ck_r = bR[k], ck_i = bI[k];   // read before the barriers of the reductions
        double wr = 0.0, wi = 0.0;
        for (int i = k + 1 + tid; i < P; i += kThreads) {
            wr += col[i] * bR[i];
            wi += col[i] * bI[i];
        }
        wr = ck_r + block_reduce(wr, red);
        wi = ck_i + block_reduce(wi, red);
        const double tk = tau[k];
        for (int i = k + 1 + tid; i < P; i += kThreads) {
            bR[i] -= (tk * col[i]) * wr;
            bI[i] -= (tk * col[i]) * wi;
        }
        if (tid == 0) {
            bR[k] -= tk * wr;
            bI[k] -= tk * wi;
        }
        __syncthreads();
    }
    // R z = c on the leading rank x rank block (column-oriented), zero beyond
    for (int i = rank - 1; i >= 0; i--) {
        const double rii = Q[(size_t)i * P + i];
        const double zr = bR[i] / rii, zi = bI[i] / rii;
        __syncthreads();
        for (int l = tid; l < i; l += kThreads) {
            const double r = Q[(size_t)i * P + l];
            bR[l] -= r * zr;
            bI[l] -= r * zi;
        }
        if (tid == 0) {
            bR[i] = zr;
            bI[i] = zi;
        }
        __syncthreads();
    }
    for (int i = rank + tid; i < P; i += kThreads) {
        bR[i] = 0.0;
        bI[i] = 0.0;
    }
    __syncthreads();
    if (tid == 0)
        for (int k = P - 1; k >= 0; k--) {
            const int c = ct[k];
            if (c != k) {
                double t = bR[k]; bR[k] = bR[c]; bR[c] = t;
                t = bI[k]; bI[k] = bI[c]; bI[c] = t;
            }
        }
    __syncthreads();

    // mean subtraction, phi-dot on the scaled solution, unscaling
    double sr = 0.0, si = 0.0;
    for (int i = tid; i < P; i += kThreads) {
        sr += bR[i];
        si += bI[i];
    }
    const double mr = block_reduce(sr, red) / P;
    const double mi = block_reduce(si, red) / P;
    double pr = 0.0, pi = 0.0;
    for (int i = tid; i < P; i += kThreads) {
        const double xr = bR[i] - mr, xi = bI[i] - mi;
        pr -= mO[i] * xr;
        pi -= mO[i] * xi;
        a.xdot[i] = xr / sc[i];
        a.xdot[P + i] = xi / sc[i];
    }
    pr = block_reduce(pr, red);
    pi = block_reduce(pi, red);
    if (tid == 0) {
        if (a.imag_time == 0)
            pi -= eR;
        else
            pr -= eR;
        a.xdot[2 * P] = pr;
        a.xdot[2 * P + 1] = pi;
    }
}

template <int NB>
__global__ __launch_bounds__(kThreads) void solve_kernel(SolveArgs a)
{
    solve_body<NB>(a);
}
__global__ __launch_bounds__(kThreads) void solve_ahead_kernel(SolveArgs a) { solve_ahead_body(a); }
__global__ __launch_bounds__(kThreads) void solve_qr_kernel(SolveArgs a)
{
    solve_qr_body(a);
}
// one workgroup per system of a batch; NB = 0: solve_ahead_body
template <int NB>
__global__ __launch_bounds__(kThreads) void solve_batch_kernel(const SolveArgs* __restrict__ args)
{
    const SolveArgs a = args[blockIdx.x];
    if (a.mean_sub)
        solve_qr_body(a);
    else if constexpr (NB == 0)
        solve_ahead_body(a);
    else
        solve_body<NB>(a);
}

constexpr size_t kMaxPanelLds = 150 * 1024;   // beside the static LDS (NB x NB block, reductions)
// Block width of the Cholesky; 0: solve_ahead_body, for the systems up to P =
// 340 (at P = 296 the whole call with its copies takes 229 us, with solve_body
// 447).  Above, 32 columns (fewer panels and barriers: at P = 420, 705 against
// 738 us with 16), and 16 again where the panel of 32 no longer fits in LDS.
// With more pieces of a row held ahead (kRowPieces; as it stands it takes up to P
// = 400) solve_ahead_body was the faster one up to P = 608, where its panels no
// longer fit the LDS (P = 560: 743 against 1315 us).  Up to 581 its 16 columns group
// the sums otherwise than 32 do: a nearly singular S of a few hundred parameters
// turns such a last-bit change into 1e-9 of the stepped parameters, so those
// sizes keep their 32 columns; 582 to 608 are left with solve_body's 16.
size_t solve_lds_bytes(int NB, int P)
{
    if (NB == 0) return ((size_t)(2 * ahead_rows(P) - kNB) * kLDP + 2 * (size_t)((P + kNB - 1) / kNB * kNB)) * sizeof(double);
    // the rows below a block at stride NB + 1 (also holds the blocks of the triangular solves)
    return (size_t)(NB + 1) * std::max(P, NB) * sizeof(double);
}
int solve_width(int P) { return P <= kAheadMaxP ? 0 : solve_lds_bytes(32, P) <= kMaxPanelLds ? 32 : 16; }

template <typename K, typename A>
hipError_t launch_cholesky(K kern, int n, size_t lds, const A& args, hipStream_t st)
{
    if (lds > 65536) {
        hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(kern, dim3(n), dim3(kThreads), lds, st, args);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_solve_batch(const SolveArgs* args_dev, int n, int P_max, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    const size_t qr = 2 * (size_t)P_max * sizeof(int);   // the QR's transpositions
    const int nb = solve_width(P_max);
    const size_t lds = std::max(qr, solve_lds_bytes(nb, P_max));
    if (nb == 0) return launch_cholesky(solve_batch_kernel<0>, n, lds, args_dev, st);
    if (nb == 32) return launch_cholesky(solve_batch_kernel<32>, n, lds, args_dev, st);
    if (lds <= kMaxPanelLds) return launch_cholesky(solve_batch_kernel<16>, n, lds, args_dev, st);
    return hipErrorInvalidValue;
}

int solve_max_params(int solver_type)
{
    if (solver_type == 1) return (int)(kMaxPanelLds / (2 * sizeof(int)));
    return (int)(kMaxPanelLds / (17 * sizeof(double)));
}

hipError_t launch_solve(const SolveArgs& a, hipStream_t st)
{
    if (a.P <= 0) return hipErrorInvalidValue;
    if (a.mean_sub) {
        hipLaunchKernelGGL(solve_qr_kernel, dim3(1), dim3(kThreads), 2 * (size_t)a.P * sizeof(int), st, a);
        return hipGetLastError();
    }
    const int nb = solve_width(a.P);
    const size_t lds = solve_lds_bytes(nb, a.P);
    if (nb == 0) return launch_cholesky(solve_ahead_kernel, 1, lds, a, st);
    if (nb == 32) return launch_cholesky(solve_kernel<32>, 1, lds, a, st);
    if (lds <= kMaxPanelLds) return launch_cholesky(solve_kernel<16>, 1, lds, a, st);
    return hipErrorInvalidValue;
}

}  // namespace tdvmc
