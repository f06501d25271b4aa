// Instantiates the null-space build by elimination for uneven builds in 3-D.
#include "build_nse_kernel.h"

namespace rbfx {

hipError_t launch_nse_rag_3d(const BuildDev& P, int m, int hi, int64_t n_work, hipStream_t s)
{
    if (m == 10 && P.basis_kind == RBFX_PHS3) return launch_nse_class_rc<RBFX_PHS3, 3, 10>(P, hi, n_work, s);
    if (m == 20 && P.basis_kind == RBFX_PHS5) return launch_nse_class_rc<RBFX_PHS5, 3, 20>(P, hi, n_work, s);
    return hipErrorInvalidValue;
}

}  // namespace rbfx
