// Launchers of the single-system evaluation kernel (one translation unit per
// precision instantiates them).
#pragma once

#include "eval_impl.hpp"

namespace tdvmc {

template <typename T, int D, bool PP, bool PER, typename TO, int WPW>
static hipError_t launch_eval_w(const KSys& sy, const KTables<T>& tb, const double* R, int64_t W,
                                const EvalOut<TO>& o, const T* rho_in, hipStream_t st)
{
    const size_t slot = eval_lds_bytes<T>(sy, PP, WPW);
    const size_t lds = (4 / WPW) * slot;
    auto kern = eval_kernel<T, D, PP, PER, TO, WPW>;
    if (lds > 65536) {
        hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    const int64_t blocks = (W + 4 / WPW - 1) / (4 / WPW);
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(kThreads), lds, st, sy, tb, R, W, o, rho_in, slot);
    return hipGetLastError();
}

// Wavefronts per walker.  Four share the set-up, the histogram's clearing and
// reduction and the assembly of one walker, which is most of a small walker's
// time; with one or two, four or two walkers do theirs side by side (one
// pair tile leaves four wavefronts N / 8 steps each).  Fewer are taken where that
// leaves the chip full:
//   - two wavefronts for every one of the 1024 SIMDs: N = 20, 1024 walkers 18.7 /
//     16.4 / 16.6 us with 1 / 2 / 4; N = 19, 101 terms, 588 walkers 48 / 32 / 25;
//   - the LDS of three workgroups (one each) or four (two each) in a CU: N = 27
//     (2-D), 48 knots, 64 terms, 2610 walkers 61 / 48 / 56 (two, four and four
//     workgroups); N = 15 (2-D), 48 knots, 258 terms, 3164 walkers 267 / 157 / 127;
//   - at most 64 and 200 k-space terms, which a walker's wavefronts go through one
//     after the other: N = 14, 206 terms, 48 knots, 1328 walkers 158 / 70 / 63; N = 27,
//     101 terms, 2291 walkers 77 / 67 / 61, N = 16, 101 terms, 11568 walkers 173 /
//     173 / 208, N = 20, 206 terms, 2063 walkers 176 / 106 / 87.
// Where all hold, up to N = 32 one, to 80 two (64 in open space, where most pairs
// fall into a few of the histogram's intervals; with per-particle output, whose
// sums per particle the wavefronts share: 16 and 36).  1 / 2 / 4, us: N = 8 (16384
// walkers) 55 / 85 / 141; N = 25 (2-D, 16 terms, 4099) 67 / 66 / 136; N = 30 (2-D trap,
// 8 knots, complex, 2100) 32 / 30 / 32; N = 38 (2-D, 64 terms, 7876) 107 / 114 / 137;
// N = 48 (2-D trap, 48 knots, 3200) 60 / 48 / 47; N = 64 (16384) 154 / 147 / 181;
// N = 90 (2-D trap, 24 knots, 2100) 105 / 74 / 58; N = 96 (8192) 196 / 154 / 160; N = 128
// (8192) 267 / 191 / 180; with per-particle output N = 33 (8192) 74 / 81 / 92, N = 40
// (2-D trap, 48 knots, 2100) 46 / 40 / 34, N = 48 (same) 53 / 44 / 37.  The mixed form
// keeps four: its FP32 sums are added up per wavefront.
template <typename T>
static int eval_waves(const KSys& sy, bool pp, int64_t W)
{
    const int one = pp ? 16 : 32, two = pp ? 36 : (sy.periodic ? 80 : 64);   // particles
    if (sizeof(T) == 4 || sy.N > two) return 4;
    auto workgroups = [&](int wpw) { return 160 * 1024 / ((4 / wpw) * eval_lds_bytes<T>(sy, pp, wpw)); };
    if (sy.N <= one && W >= 2048 && sy.Kh <= 64 && workgroups(1) >= 3) return 1;
    if (W >= 1024 && sy.Kh <= 200 && workgroups(2) >= 4) return 2;
    return 4;
}

template <typename T, int D, bool PP, bool PER, typename TO>
static hipError_t launch_eval_k(const KSys& sy, const KTables<T>& tb, const double* R, int64_t W,
                                const EvalOut<TO>& o, const T* rho_in, hipStream_t st)
{
    if constexpr (sizeof(T) == 8) {
        const int wpw = eval_waves<T>(sy, PP, W);
        if (wpw == 1) return launch_eval_w<T, D, PP, PER, TO, 1>(sy, tb, R, W, o, rho_in, st);
        if (wpw == 2) return launch_eval_w<T, D, PP, PER, TO, 2>(sy, tb, R, W, o, rho_in, st);
    }
    return launch_eval_w<T, D, PP, PER, TO, 4>(sy, tb, R, W, o, rho_in, st);
}

template <typename T, int D, typename TO>
static hipError_t launch_eval_d(const KSys& sy, const KTables<T>& tb, const double* R, int64_t W,
                                const EvalOut<TO>& o, const T* rho_in, bool pp, hipStream_t st)
{
    if (sy.periodic)
        return pp ? launch_eval_k<T, D, true, true, TO>(sy, tb, R, W, o, rho_in, st)
                  : launch_eval_k<T, D, false, true, TO>(sy, tb, R, W, o, rho_in, st);
    return pp ? launch_eval_k<T, D, true, false, TO>(sy, tb, R, W, o, rho_in, st)
              : launch_eval_k<T, D, false, false, TO>(sy, tb, R, W, o, rho_in, st);
}

template <typename T, typename TO>
hipError_t launch_eval(const KSys& sy, const KTables<T>& tb, const double* R, int64_t W, double* expo, double* ER,
                       double* EI, TO* O, double* other, double* grad, double* lap, double* outer,
                       const T* rho_in, hipStream_t st, double* bsum, uint32_t* tick)
{
    if (W <= 0) return hipSuccess;
    EvalOut<TO> o{expo, ER, EI, O, other, grad, lap, outer, bsum, tick};
    const bool pp = grad != nullptr;
    switch (sy.D) {
    case 1: return launch_eval_d<T, 1, TO>(sy, tb, R, W, o, rho_in, pp, st);
    case 2: return launch_eval_d<T, 2, TO>(sy, tb, R, W, o, rho_in, pp, st);
    case 3: return launch_eval_d<T, 3, TO>(sy, tb, R, W, o, rho_in, pp, st);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace tdvmc
