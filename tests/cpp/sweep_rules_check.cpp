// The sweep's launch rules (tdvmc_amd/csrc/sweep_rules.hpp) on the host: for each
// line "D N P_s Kh kmax W" of the input, the FP64 form's lanes per walker, whether
// it tabulates the phase factors, and the LDS of a workgroup.
#include <cstdio>

#include "../../tdvmc_amd/csrc/sweep_rules.hpp"

int main()
{
    int D, N, Ps, Kh, kmax;
    long long W;
    while (std::scanf("%d %d %d %d %d %lld", &D, &N, &Ps, &Kh, &kmax, &W) == 6) {
        tdvmc::KSys sy{};
        sy.D = D;
        sy.N = N;
        sy.P_s = Ps;
        sy.Kh = Kh;
        sy.kmax = kmax;
        sy.periodic = 1;
        sy.L = 1.0;
        sy.Linv = 1.0;
        sy.rc = 0.5;
        sy.hinv = 2.0 * (Ps - 1);
        const int lanes = tdvmc::default_lanes<double>(sy, W);
        std::printf("%d %d %zu\n", lanes, (int)tdvmc::sweep_phase_table<double>(sy, lanes),
                    tdvmc::sweep_lds_bytes<double>(sy, lanes));
    }
}
