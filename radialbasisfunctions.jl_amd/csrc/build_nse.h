// Null-space build by elimination: interface between the C ABI layer and the kernels of
// build_nse*.hip.
#pragma once
#include "build.h"

namespace rbfx {

// Whether a kernel is built for uniform stencils of k points with m monomials and n_cols
// operator columns of a basis in dim dimensions.
bool nse_fits(int basis_kind, int dim, int k, int m, int n_cols);

// FP64 null-space build (by elimination) of the work (P.list / P.order / all stencils) of a
// uniform interior build within nse_fits, without multipliers (no out_lambda). Stencils
// whose factorisation breaks down and Hermite stencils are appended to P.fail_list for
// the rook-pivoted kernels; every other stencil gets status P.ok_status.
hipError_t launch_build_nse(const BuildDev& P, int dim, int64_t n_work, hipStream_t s);

}  // namespace rbfx
