// Instantiates the null-space build by elimination: PHS3 in 2-D, degrees 1 to 4.
#include "build_nse_kernel.h"

namespace rbfx {

hipError_t launch_nse_2d_phs3(const BuildDev& P, int64_t n_work, hipStream_t s)
{
    if (P.n_mono == 3) return launch_nse_rc<RBFX_PHS3, 2, 3>(P, n_work, s);
    if (P.n_mono == 6) return launch_nse_rc<RBFX_PHS3, 2, 6>(P, n_work, s);
    if (P.n_mono == 10) return launch_nse_rc<RBFX_PHS3, 2, 10>(P, n_work, s);
    if (P.n_mono == 15) return launch_nse_rc<RBFX_PHS3, 2, 15>(P, n_work, s);
    return hipErrorInvalidValue;
}

}  // namespace rbfx
