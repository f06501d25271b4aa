// Dispatch of the null-space build by elimination over basis, dimension and stencil
// shape (kernel template in build_nse_kernel.h, instantiations in build_nse_*.hip).
#include "build_nse.h"
#include "build_nsc.h"

namespace rbfx {

hipError_t launch_nse_2d_phs3(const BuildDev& P, int64_t n_work, hipStream_t s);
hipError_t launch_nse_2d_phs5(const BuildDev& P, int64_t n_work, hipStream_t s);
hipError_t launch_nse_2d_phs7(const BuildDev& P, int64_t n_work, hipStream_t s);
hipError_t launch_nse_3d_low(const BuildDev& P, int64_t n_work, hipStream_t s);
hipError_t launch_nse_3d_phs3(const BuildDev& P, int64_t n_work, hipStream_t s);
hipError_t launch_nse_3d_phs5(const BuildDev& P, int64_t n_work, hipStream_t s);
hipError_t launch_nse_3d_phs7(const BuildDev& P, int64_t n_work, hipStream_t s);

hipError_t launch_nse_rag_2d(const BuildDev& P, int m, int hi, int64_t n_work, hipStream_t s);
hipError_t launch_nse_rag_3d(const BuildDev& P, int m, int hi, int64_t n_work, hipStream_t s);

// Shapes of uniform builds. The null points (k - m) and the operator columns share the lanes of
// one or two slots of 16: at most 26 null points with the most columns, and none beyond that
// here (the classes of uneven builds below go to 32 less the columns in 2-D). The monomial
// tables of degree 1 to 4 (2-D) and 1 to 3 (3-D) that the basis is definite with. Other
// shapes (1-D, other bases, wider stencils, more columns) stay with the other kernels.
bool nse_fits(int kind, int dim, int k, int m, int n_cols)
{
    const int nn = k - m;
    if (nn < 1 || n_cols < 1) return false;
    if (kind != RBFX_PHS3 && kind != RBFX_PHS5 && kind != RBFX_PHS7) return false;
    if (dim == 2) {
        if (n_cols > 3) return false;
        if (m == 3) return kind == RBFX_PHS3 && nn <= 13 - n_cols;
        if (m == 6) return kind != RBFX_PHS7 && nn <= 26;
        return (m == 10 || m == 15) && nn <= 26;
    }
    if (dim == 3) {
        if (n_cols > 6) return false;
        const int rc = n_cols == 2 ? 3 : (n_cols == 5 ? 6 : n_cols);
        if (m == 4) return kind == RBFX_PHS3 && nn <= 16 - rc;
        if (m == 10) return kind != RBFX_PHS7 && nn <= 26;
        return m == 20 && nn <= 26;
    }
    return false;
}

hipError_t launch_build_nse(const BuildDev& P, int dim, int64_t n_work, hipStream_t s)
{
    if (!nse_fits(P.basis_kind, dim, P.k, P.n_mono, P.n_cols)) return hipErrorInvalidValue;
    // uniform builds only: the kernel takes every stencil's k and m from P.k and P.n_mono
    if (P.adj_ptr || P.deg_map || P.out_lambda) return hipErrorInvalidValue;
    if (dim == 2) {
        if (P.basis_kind == RBFX_PHS3) return launch_nse_2d_phs3(P, n_work, s);
        if (P.basis_kind == RBFX_PHS5) return launch_nse_2d_phs5(P, n_work, s);
        return launch_nse_2d_phs7(P, n_work, s);
    }
    if (P.n_mono <= 10) return launch_nse_3d_low(P, n_work, s);
    if (P.basis_kind == RBFX_PHS3) return launch_nse_3d_phs3(P, n_work, s);
    if (P.basis_kind == RBFX_PHS5) return launch_nse_3d_phs5(P, n_work, s);
    return launch_nse_3d_phs7(P, n_work, s);
}

// operator columns of the kernel that serves n_cols of them (0: none)
static int nse_rc(int dim, int n_cols)
{
    if (dim == 2) return n_cols <= 3 ? n_cols : 0;
    if (dim == 3) return n_cols == 2 ? 3 : (n_cols == 5 ? 6 : (n_cols <= 6 ? n_cols : 0));
    return 0;
}

// Built: PHS3 with 6 and 10 monomials and PHS5 with 10 in 2-D, PHS3 with 10 and PHS5 with 20
// in 3-D (the basis must be definite with each stencil's own degree). The second class stops
// at 26 null points, where its columns cost less than those of the full two slots; in 2-D a
// third takes the rest of them (the 3-D kernels have no registers left for it). Update of
// 1.29M stencils in a disk, 120,000 of them of 33 to 37 points: 15.7 ms without the third
// class, 12.4 with it.
int nse_classes(int kind, int dim, int poly_deg, int n_cols, NseClass* out)
{
    const int rc = n_cols >= 1 ? nse_rc(dim, n_cols) : 0;
    int n = 0;
    if (rc == 0) return 0;
    for (int deg = 0; deg <= poly_deg; ++deg) {
        const int m = n_mono_of(dim, deg);
        const bool built = dim == 2 ? (kind == RBFX_PHS3 && (m == 6 || m == 10)) || (kind == RBFX_PHS5 && m == 10)
                                    : (kind == RBFX_PHS3 && m == 10) || (kind == RBFX_PHS5 && m == 20);
        if (!built || nsc_sign(kind, deg) == 0 || n + (dim == 2 ? 3 : 2) > kNseClasses) continue;
        const int one = m == 20 ? 20 : 16 - rc;
        out[n++] = NseClass{m, 0, one};
        out[n++] = NseClass{m, one, 26};
        if (dim == 2) out[n++] = NseClass{m, 26, 32 - rc};
    }
    return n;
}

hipError_t launch_build_nse_class(const BuildDev& P, int dim, const NseClass& c, int64_t n_work, hipStream_t s)
{
    if (P.out_lambda) return hipErrorInvalidValue;
    return dim == 2 ? launch_nse_rag_2d(P, c.m, c.hi, n_work, s) : launch_nse_rag_3d(P, c.m, c.hi, n_work, s);
}

}  // namespace rbfx
