// The measurement's launch rules (tdvmc_amd/csrc/eval_launch.hpp) on the host: for
// each line "D N P_s Kh W per_particle" of the input, the FP64 form's wavefronts
// per walker and the LDS of a workgroup of one walker per 1, 2 and 4 of them.
#include <cstdio>

#include "../../tdvmc_amd/csrc/eval_launch.hpp"

int main()
{
    int D, N, Ps, Kh, pp;
    long long W;
    while (std::scanf("%d %d %d %d %lld %d", &D, &N, &Ps, &Kh, &W, &pp) == 6) {
        tdvmc::KSys sy{};
        sy.D = D;
        sy.N = N;
        sy.P_s = Ps;
        sy.Kh = Kh;
        sy.periodic = 1;
        std::printf("%d", tdvmc::eval_waves<double>(sy, pp != 0, W));
        for (int w = 1; w <= 4; w *= 2) std::printf(" %zu", (4 / w) * tdvmc::eval_lds_bytes<double>(sy, pp != 0, w));
        std::printf("\n");
    }
}
