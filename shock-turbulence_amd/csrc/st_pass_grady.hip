// y pass of the first-derivative right-hand side (with four mixed terms and
// the pointwise assembly).
#include "st_pass_grad.hpp"

namespace st {

hipError_t launch_grad_y(const DirTab &t, int nt, int My, int Mz, int Mx, const PassArgs &a, hipStream_t s)
{
    return launch<PassGrad<1, 2>, false>(t, nt, 1, My, Mz, Mx, a, s);
}

hipError_t launch_grad_y_ragged(const RaggedSpec &sp, hipStream_t s) { return launch_ragged<PassGrad<1, 2>>(sp, s); }

}  // namespace st
