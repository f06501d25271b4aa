// Instantiates the null-space build by elimination: PHS5 in 3-D, degree 3.
#include "build_nse_kernel.h"

namespace rbfx {

hipError_t launch_nse_3d_phs5(const BuildDev& P, int64_t n_work, hipStream_t s)
{
    if (P.n_mono == 20) return launch_nse_rc<RBFX_PHS5, 3, 20>(P, n_work, s);
    return hipErrorInvalidValue;
}

}  // namespace rbfx
