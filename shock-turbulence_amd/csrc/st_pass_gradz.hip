// z pass of the first-derivative right-hand side (with two mixed terms).
#include "st_pass_grad.hpp"

namespace st {

// Lines of 32 lanes: two rounds of staging (TWO) need five slots instead of
// seven.  At 8 points per lane that lets two workgroups of 256 threads share a
// CU; below, a tile of 512 threads (16 lines: whole 128-byte rows, which stream)
// does better than the plain form on 256 (stage at 192^3 2337 -> 2315 us, 128^3
// 710 -> 699; at 256^3 the 512-thread tile loses, 5210 -> 5255).
hipError_t launch_grad_z(const DirTab &t, int nt, int My, int Mz, int Mx, const PassArgs &a, hipStream_t s)
{
    if (nt == 512 && t.P == 32) {
        switch (t.M) {
        case 4: return launch_at<PassGrad<2, 2, true>, 4, 32, 512>(t, 2, My, Mz, Mx, a, s);
        case 5: return launch_at<PassGrad<2, 2, true>, 5, 32, 512>(t, 2, My, Mz, Mx, a, s);
        case 6: return launch_at<PassGrad<2, 2, true>, 6, 32, 512>(t, 2, My, Mz, Mx, a, s);
        case 7: return launch_at<PassGrad<2, 2, true>, 7, 32, 512>(t, 2, My, Mz, Mx, a, s);
        }
    }
    if (nt == 256 && t.M == 8 && t.P == 32) return launch_at<PassGrad<2, 2, true>, 8, 32, 256>(t, 2, My, Mz, Mx, a, s);
    return launch<PassGrad<2, 1>, false>(t, nt, 2, My, Mz, Mx, a, s);
}

hipError_t launch_grad_z_ragged(const RaggedSpec &sp, hipStream_t s) { return launch_ragged<PassGrad<2, 1>>(sp, s); }

}  // namespace st
