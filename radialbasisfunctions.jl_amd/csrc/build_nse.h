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

// Shape classes of an uneven build (ragged stencils, per-stencil degrees): stencils of m
// monomials and lo < k - m <= hi points beyond them run together in one launch. At most
// kNseClasses of them, for the degrees up to poly_deg that a kernel is built for.
struct NseClass {
    int m, lo, hi;
};
constexpr int kNseClasses = 8;
int nse_classes(int basis_kind, int dim, int poly_deg, int n_cols, NseClass* out);

// The stencils of P.list, all of class c. What they hand back goes to the list of its size
// bucket (k + m <= 32, <= 64, above): P.fail_list + b * P.fail_stride, P.fail_count + b.
hipError_t launch_build_nse_class(const BuildDev& P, int dim, const NseClass& c, int64_t n_work, hipStream_t s);

}  // namespace rbfx
