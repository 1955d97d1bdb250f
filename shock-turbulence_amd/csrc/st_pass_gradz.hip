// z pass of the first-derivative right-hand side (with two mixed terms).
#include "st_pass_grad.hpp"

namespace st {

hipError_t launch_grad_z(const DirTab &t, int nt, int My, int Mz, int Mx, const PassArgs &a, hipStream_t s)
{
    // 8 points per lane on 256 threads: two workgroups per CU
    if (nt == 256 && t.M == 8 && t.P == 32) return launch_at<PassGrad<2, 2, true>, 8, 32, 256>(t, 2, My, Mz, Mx, a, s);
    return launch<PassGrad<2, 1>, false>(t, nt, 2, My, Mz, Mx, a, s);
}

hipError_t launch_grad_z_ragged(const RaggedSpec &sp, hipStream_t s) { return launch_ragged<PassGrad<2, 1>>(sp, s); }

}  // namespace st
