// Sizes and choices of the sweep's launches: LDS of a workgroup, which tables it
// holds, lanes per walker.
#pragma once

#include "common.hpp"
#include "kernels.hpp"

namespace tdvmc {

constexpr int kSweepThreads = 256;

// Rows of the spline table in LDS (uniform knots: intervals, extended in a
// periodic box to the largest minimum-image distance; non-uniform knots: P_s
// interval rows, then the lookup cells).
__host__ __device__ inline int sweep_table_len(const KSys& sy)
{
    if (sy.nu) return sy.P_s + sy.ncell;
    if (!sy.periodic) return sy.P_s - 1;
    // largest minimum-image distance sqrt(D)/2 L, in knot intervals, + margin
    const double xmax = 0.5 * sqrt((double)sy.D) * sy.L * sy.hinv;
    const int j = (int)xmax + 2;
    return j > sy.P_s - 1 ? j : sy.P_s - 1;
}

// Phase factors of the FP64 form: e^{ik.r} = prod_a e^{2 pi i n_a x_a}, so the
// group tabulates e^{2 pi i m x_a}, |m| <= kmax, of two positions (a trial's
// old and new one, or two particles while rho_k is built) in LDS, one sine and
// cosine per lane for the 2 D kmax factors, and a k-space term takes them from
// there with D - 1 complex products.  Two sincos per term, lane and trial took
// 237 of about 720 vector instructions of a trial (N = 343, 128 terms, 64
// lanes) and set the time in 2-D.  16384 walkers, 64 lanes: 7.48 -> 6.33 ms
// (3-D, N = 343, 128 terms), 18.0 -> 8.50 ms (2-D, N = 400, 258 terms).  In 1-D
// kmax is the number of terms and nothing is shared: each term keeps its own
// sincos there, as where the tables would not fit the LDS or the group.  Nor do
// they pay where a lane has one term only, which needs two sines and cosines
// either way (N = 12, 10 terms, 3256 walkers, 16 lanes: 15.4 us, with tables 19.0;
// N = 61, 10 terms, 7636 walkers: 124 and 144).
constexpr size_t kLdsMax = 160 * 1024;
// LDS of one workgroup without the phase tables: spline rows and coordinates
template <typename T>
__host__ __device__ inline size_t sweep_base_lds(const KSys& sy, int lpw)
{
    // coordinates: uint32 fractions (FP32, periodic) or T
    const size_t cs = (sizeof(T) == 4 && sy.periodic) ? sizeof(uint32_t) : sizeof(T);
    return sizeof(T) * 4 * (size_t)sweep_table_len(sy) + ((cs * (kSweepThreads / lpw) * sy.N * sy.D + 15) & ~(size_t)15);
}
// entries of a walker's table: [axis][m + kmax][position], (cos, sin) each
__host__ __device__ inline int sweep_phase_len(const KSys& sy) { return sy.D * (2 * sy.kmax + 1) * 2; }
template <typename T>
__host__ __device__ inline bool sweep_phase_table(const KSys& sy, int lpw)
{
    if (sizeof(T) == 4 || sy.D < 2 || sy.Kh <= lpw || 2 * sy.D * sy.kmax > 64) return false;   // 64: factors per group
    return sweep_base_lds<T>(sy, lpw) + (kSweepThreads / lpw) * (size_t)sweep_phase_len(sy) * 2 * sizeof(T) <= kLdsMax;
}

// Spline rows of the mixed form 256 bytes apart, in 16 copies: the conversion of
// r / h to an integer writes it into byte 1 of the row's LDS address, whose
// other bytes stay (the lane's copy in byte 0, zeros above).  One instruction
// instead of a conversion and a shift-add, for both distances of a pair's 37
// vector instructions and 4 LDS reads, and no two of the 16 lanes that the LDS
// serves together share a bank.  Same values, same bits.
// Taken where five workgroups fit the LDS of a CU (the registers allow no
// more); below that the wavefronts it costs take the gain back.  Sweep of
// 16384 walkers in us, plain and wide: 2-D N = 400, 258 terms, 64 lanes (27 KB)
// 3829 / 3680; 3-D, 32 lanes, N = 64 (24 KB) 112 / 109, N = 125 (30 KB) 370 / 362,
// N = 160 (33 KB) 529 / 534, N = 260 (43 KB) 1240 / 1341, N = 343 (51 KB) 2478 /
// 2485 (one workgroup of 1024 threads and one table for it: 2587).
constexpr int kWide = 16;
template <typename T>
inline size_t sweep_wide_lds(const KSys& sy, int lpw)
{
    return sweep_base_lds<T>(sy, lpw) + (kWide - 1) * sizeof(T) * 4 * (size_t)sweep_table_len(sy);
}
template <typename T>
inline bool sweep_wide(const KSys& sy, int lpw)
{
    // (32 KB hold at most 128 rows: a byte counts them)
    return sizeof(T) == 4 && sy.periodic && !sy.nu && sweep_wide_lds<T>(sy, lpw) <= kLdsMax / 5;
}
// Default lanes per walker without tuning: 32 from N = 24 on (two walkers
// per wavefront share the per-trial overhead and waste fewer partner slots
// than one walker per wavefront), 16 below; more when the k-space terms would
// need more than 8 per lane.
inline int pick_lpw(int N, int K)
{
    int l = N >= 24 ? 32 : 16;
    while (l < 64 && K > 8 * l) l *= 2;
    return l;
}

template <typename T>
size_t sweep_lds_bytes(const KSys& sy, int lpw)
{
    if (lpw <= 0) lpw = pick_lpw(sy.N, sy.Kh);
    const size_t base = sweep_base_lds<T>(sy, lpw);
    return sweep_phase_table<T>(sy, lpw) ? base + (kSweepThreads / lpw) * (size_t)sweep_phase_len(sy) * 2 * sizeof(T) : base;
}

// Default lanes per walker of a single system.  Mixed form: pick_lpw (its FP32
// sums, and with them rare decisions, depend on the lane count).  FP64: the
// fewest lanes, which share a trial's overhead among the most walkers, that
// leave at most four k-space terms a lane, the LDS room for three workgroups per
// CU, and either three wavefronts for two SIMDs or a lane for every particle and
// term (more lanes would have nothing to do).  Sweep in us with 16 / 32 / 64
// lanes: N = 64, 16384 / 2048 / 512 walkers 209 / 233 / 264, 82 / 55 / 49, 77 / 51 /
// 35; N = 125, 60 k, 8192 walkers (2, 5 and 8 workgroups by LDS) 561 / 510 / 614;
// N = 12, 10 terms, 3256 walkers 15 / 20 / 30; N = 14, 16 terms, 3370 walkers 17 / 23 /
// 34; N = 15 (2-D), 258 terms, 3203 walkers 56 with 64; 101 terms, N = 10, 17471
// walkers 135 / 92 / 124; N = 343, 256 k, 512 walkers 3147 / 1294 / 769.  Without the
// tables and with 16 (N < 24) or 32 lanes everywhere, none of 800 systems drawn
// over D, N = 4 .. 343, 0 .. 512 k and 256 .. 32768 walkers was faster.
template <typename T>
inline int default_lanes(const KSys& sy, int64_t W)
{
    if (sizeof(T) == 4) return pick_lpw(sy.N, sy.Kh);
    for (int l = 16; l < 64; l *= 2)
        if (sy.Kh <= 4 * l && sweep_lds_bytes<T>(sy, l) <= kLdsMax / 3 && (W * l >= 64 * 1536 || (l >= sy.N && l >= sy.Kh)))
            return l;
    return 64;
}

}  // namespace tdvmc
