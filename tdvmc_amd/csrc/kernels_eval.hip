// Measurement and evaluation of one system, FP32 pair arithmetic (mixed form).
#include "eval_launch.hpp"

namespace tdvmc {

template size_t eval_lds_bytes<float>(const KSys&, bool, int);
template hipError_t launch_eval<float, float>(const KSys&, const KTables<float>&, const double*, int64_t, double*,
                                              double*, double*, float*, double*, double*, double*, double*,
                                              const float*, hipStream_t, double*, uint32_t*);
template hipError_t launch_eval<float, double>(const KSys&, const KTables<float>&, const double*, int64_t, double*,
                                               double*, double*, double*, double*, double*, double*, double*,
                                               const float*, hipStream_t, double*, uint32_t*);

}  // namespace tdvmc
