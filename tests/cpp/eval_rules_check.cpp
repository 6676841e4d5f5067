// The measurement's launch rules (tdvmc_amd/csrc/eval_launch.hpp, eval_impl.hpp) on
// the host: for each line "D N P_s Kh W per_particle nrun kmax" of the input, the
// FP64 form's wavefronts per walker, the LDS of a workgroup of walkers of 1, 2 and
// 4 of them, and for 1, 2 and 4 whether the k-space gradient goes by runs and how
// many particles a pass of the rho_k table holds, with real and complex parameters.
#include <cstdio>

#include "../../tdvmc_amd/csrc/eval_launch.hpp"

int main()
{
    int D, N, Ps, Kh, pp, nrun, kmax;
    long long W;
    while (std::scanf("%d %d %d %d %lld %d %d %d", &D, &N, &Ps, &Kh, &W, &pp, &nrun, &kmax) == 8) {
        tdvmc::KSys sy{};
        sy.D = D;
        sy.N = N;
        sy.P_s = Ps;
        sy.Kh = Kh;
        sy.nrun = nrun;
        sy.kmax = kmax;
        sy.periodic = 1;
        std::printf("%d", tdvmc::eval_waves<double>(sy, pp != 0, W));
        for (int w = 1; w <= 4; w *= 2) std::printf(" %zu", (4 / w) * tdvmc::eval_lds_bytes<double>(sy, pp != 0, w));
        for (int w = 1; w <= 4; w *= 2) {
            std::printf(" %d", (int)tdvmc::eval_use_runs(sy, w));
            for (int cplx = 0; cplx < 2; cplx++) {
                const size_t nd = (size_t)Ps * 4 * tdvmc::hist_cols(cplx, w) + (size_t)N * (cplx ? 2 : 1) * D;
                std::printf(" %d", tdvmc::rho_table_particles(sy, nd * sizeof(double), 64 * w).particles);
            }
        }
        std::printf("\n");
    }
}
