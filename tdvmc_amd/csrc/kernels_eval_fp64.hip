// Measurement and evaluation of one system, FP64.
#include "eval_launch.hpp"

namespace tdvmc {

template size_t eval_lds_bytes<double>(const KSys&, bool, int);
template hipError_t launch_eval<double, double>(const KSys&, const KTables<double>&, const double*, int64_t, double*,
                                                double*, double*, double*, double*, double*, double*, double*,
                                                const double*, hipStream_t, double*, uint32_t*);

}  // namespace tdvmc
