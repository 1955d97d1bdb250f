// x pass of the first-derivative right-hand side.
#include "st_pass_grad.hpp"

namespace st {

hipError_t launch_grad_x(const DirTab &t, int nt, int My, int Mz, int Mx, const PassArgs &a, hipStream_t s)
{
    return launch<PassGrad<0, 1>>(t, nt, 0, My, Mz, Mx, a, s);
}

hipError_t launch_grad_x_ragged(const RaggedSpec &sp, hipStream_t s) { return launch_ragged<PassGrad<0, 1>>(sp, s); }

}  // namespace st
