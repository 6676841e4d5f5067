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
// pair tile leaves four wavefronts N / 8 steps each).  FP64, us with 1 / 2 / 4:
//   N = 8 (3-D, 16384 walkers) 55 / 85 / 141; N = 25 (2-D, 16 terms, 4099) 67 / 66 / 136;
//   N = 33 (8192) 67 / 74 / 99; N = 64 (16384) 154 / 147 / 181; N = 96 (8192) 196 / 154 / 160;
//   N = 128 (8192) 267 / 191 / 180; with per-particle output N = 33 74 / 81 / 92, N = 64 193 / 180 / 174.
// Few walkers need more wavefronts each to reach every SIMD: N = 20, 1024
// walkers 18.7 / 16.4 / 16.6; N = 64 24 / 23 / 21 with 1024, 32 / 30 / 34 with
// 2048.  The mixed form keeps four: its FP32 sums are added up per wavefront.
template <typename T>
static int eval_waves(const KSys& sy, bool pp, int64_t W)
{
    if (sizeof(T) == 4 || sy.N > (pp ? 48 : 100)) return 4;
    int wpw = sy.N <= 48 ? 1 : 2;
    const int64_t least = sy.N <= 48 ? 1025 : 4096;   // wavefronts
    while (wpw < 4 && (W * wpw < least || (4 / wpw) * eval_lds_bytes<T>(sy, pp, wpw) > 160 * 1024)) wpw *= 2;
    return wpw;
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
