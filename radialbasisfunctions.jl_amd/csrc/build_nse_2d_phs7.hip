// Instantiates the null-space build by elimination: PHS7 in 2-D, degrees 3 and 4.
#include "build_nse_kernel.h"

namespace rbfx {

hipError_t launch_nse_2d_phs7(const BuildDev& P, int64_t n_work, hipStream_t s)
{
    if (P.n_mono == 10) return launch_nse_rc<RBFX_PHS7, 2, 10>(P, n_work, s);
    if (P.n_mono == 15) return launch_nse_rc<RBFX_PHS7, 2, 15>(P, n_work, s);
    return hipErrorInvalidValue;
}

}  // namespace rbfx
