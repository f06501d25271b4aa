// Instantiates the null-space build by elimination: PHS3 (degrees 1 and 2) and PHS5 (degree 2) in 3-D.
#include "build_nse_kernel.h"

namespace rbfx {

hipError_t launch_nse_3d_low(const BuildDev& P, int64_t n_work, hipStream_t s)
{
    if (P.n_mono == 4 && P.basis_kind == RBFX_PHS3) return launch_nse_rc<RBFX_PHS3, 3, 4>(P, n_work, s);
    if (P.n_mono == 10 && P.basis_kind == RBFX_PHS3) return launch_nse_rc<RBFX_PHS3, 3, 10>(P, n_work, s);
    if (P.n_mono == 10 && P.basis_kind == RBFX_PHS5) return launch_nse_rc<RBFX_PHS5, 3, 10>(P, n_work, s);
    return hipErrorInvalidValue;
}

}  // namespace rbfx
