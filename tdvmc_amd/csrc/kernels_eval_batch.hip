// Measurement of a batch of systems in one launch.
#include "eval_impl.hpp"

namespace tdvmc {

namespace {

// Batch of independent systems in one launch.  Each system has its own
// walker shape: 1, 2 or 4 wavefronts per walker (4, 2 or 1 walkers per
// workgroup); a workgroup belongs to one system.  Small walkers are bound by
// latency more than by issue, so the FP32 form is compiled for 6 waves per
// SIMD (80 registers) instead of 4; the FP64 form keeps 4 (it would spill).
template <typename T, int D, bool PER>
__global__ __launch_bounds__(kThreads, sizeof(T) == 4 ? 6 : 4) void eval_batch_kernel(EvalBatch<T> bt)
{
    int lo = 0, hi = bt.n;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (bt.block_start[mid] <= (int64_t)blockIdx.x)
            lo = mid;
        else
            hi = mid;
    }
    const EvalBatchItem<T>& it = bt.item[lo];
    EvalOut<double> o{it.expo, it.ER, it.EI, it.O, it.other, nullptr, nullptr, it.outer};
    const int64_t b = (int64_t)blockIdx.x - bt.block_start[lo];
    const size_t sb = (size_t)it.slot_bytes;
    switch (it.wpw) {
    case 1: {
        const int slot = threadIdx.x >> 6;
        eval_body<T, D, false, PER, double, 1>(bt.sys[lo], bt.tab[lo], it.R, it.W, o, it.rho, b * 4 + slot, slot, sb);
        break;
    }
    case 2: {
        const int slot = threadIdx.x >> 7;
        eval_body<T, D, false, PER, double, 2>(bt.sys[lo], bt.tab[lo], it.R, it.W, o, it.rho, b * 2 + slot, slot, sb);
        break;
    }
    default:
        eval_body<T, D, false, PER, double, 4>(bt.sys[lo], bt.tab[lo], it.R, it.W, o, it.rho, b, 0, sb);
        break;
    }
}

}  // namespace

// One wavefront per walker up to N = 32 (a single 64-row pair tile), two up
// to 64, four above.
int eval_default_wpw(int N) { return N <= 32 ? 1 : (N <= 64 ? 2 : 4); }

template <typename T, int D, bool PER>
static hipError_t launch_eval_batch_k(const EvalBatch<T>& bt, int64_t blocks, size_t lds, hipStream_t st)
{
    auto kern = eval_batch_kernel<T, D, PER>;
    if (lds > 65536) {
        hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(kThreads), lds, st, bt);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_eval_batch(const EvalBatch<T>& bt, int D, bool periodic, int64_t blocks, size_t lds, hipStream_t st)
{
    if (blocks <= 0) return hipSuccess;
    switch (D) {
    case 1: return periodic ? launch_eval_batch_k<T, 1, true>(bt, blocks, lds, st)
                            : launch_eval_batch_k<T, 1, false>(bt, blocks, lds, st);
    case 2: return periodic ? launch_eval_batch_k<T, 2, true>(bt, blocks, lds, st)
                            : launch_eval_batch_k<T, 2, false>(bt, blocks, lds, st);
    case 3: return periodic ? launch_eval_batch_k<T, 3, true>(bt, blocks, lds, st)
                            : launch_eval_batch_k<T, 3, false>(bt, blocks, lds, st);
    default: return hipErrorInvalidValue;
    }
}

template hipError_t launch_eval_batch<float>(const EvalBatch<float>&, int, bool, int64_t, size_t, hipStream_t);
template hipError_t launch_eval_batch<double>(const EvalBatch<double>&, int, bool, int64_t, size_t, hipStream_t);

}  // namespace tdvmc
