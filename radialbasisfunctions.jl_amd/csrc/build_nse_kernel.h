// Null-space stencil build by elimination, register-resident, for gfx950 (kernel template).
//
// Same system and same reference code as build_kernel.h (src/solve/execution.jl:186-265,
// assembly.jl:95-222):
//     [ Phi  P ] [ w      ]   [ L phi (x_e, .) ]
//     [ P^T  0 ] [ lambda ] = [ L P (x_e)      ]
// for interior stencils of uniform builds whose Phi is definite on the null space of P^T
// (nsc_sign). P is factorised first, P = L U with row pivoting over the stencil's points:
// the M pivot points are the basic ones (B), the others the null ones (N). With
// C = L_N L_B^-1 (P_N = C P_B), w_B = w0 - C^T w_N and w0 = P_B^-T L P, what remains is
//     S w_N = t,   S = Phi_NN - T C^T - C T^T,   T = Phi_NB - C Phi_BB / 2,
// definite, so it needs no pivot search. The right-hand side t is the same bilinear
// form: with the rows C_g = w0^T and T_g = b_B^T - w0^T Phi_BB / 2 of an operator column
// appended, t = b_N - T C_g^T - C T_g^T. So each operator column is carried as one more
// row of P, C and T and one more column of S.
//
// Mapping: 16 lanes (one DPP row) per stencil, four stencils per wavefront; lane li owns
// rows li, li + 16, ... of the points (LU), of the null points (C, T, S) and of the basic
// points (L_B, Phi_BB). Basic and null points get fixed positions after the LU (through
// LDS), so all later indices are compile-time constants. A value of one lane enters the
// FMAs of the other fifteen through the DPP broadcast of the instruction itself
// (v_fmac_f64 with row_newbcast), which runs at the FMA's own rate (5.1 against 4.7
// cycles measured, four waves per SIMD): no LDS read and no move per broadcast operand.
// S is eliminated by Gauss-Jordan steps, so no triangular solve follows and the columns of
// the right-hand sides are updated by the same instructions. Last, w_B is corrected once by the
// residual of the polynomial conditions (Gauss-Jordan on P_B^T, in the lanes as well). LDS
// carries the pivot rows of the LU, the two changes of layout, and what the correction reads
// again.
//
// Bound by FP64 VALU issue; VGPRs (the instantiation's W waves per SIMD) and LDS
// (NseLds) set how many wavefronts hide the LU's serial chain of pivots. Measured against
// the kernels that served these builds before: 4M-point 2-D Laplacian (PHS3, degree 2,
// k = 20) 12.03 -> 3.51 ms per build (null-space Cholesky, 8 lanes of three rows; 448
// VALU instructions per stencil against 897), 2M-point 3-D gradient and Laplacian (PHS5,
// degree 3, k = 40) 149.1 -> 13.9 ms (rook LDL^T in LDS; 2,850 against 21,800).
//
// Breakdown: an LU pivot below kNseLuTol (scaled coordinates, monomials of order one), or
// a pivot of S below kNsePivTol of the stencil's scale, hands the stencil to the rook-pivoted
// kernels. The scale is the largest pivot so far and no less than the largest entry of T: the
// entries of S are differences of products of T, so each carries an error of some u times it,
// whatever they cancel to (a repeated point's pivot is that error alone, and a scale of the
// pivots only would not see it in the first one). The weights accepted carry up to some
// u / kNsePivTol = 1e-7 of error from the elimination.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>
#include <utility>

#include "build_nse.h"
#include "build_nsc_kernel.h"

namespace rbfx {

constexpr double kNseLuTol = 1e-6;
constexpr double kNsePivTol = 1e-9;

// ---------------------------------------------------------------- unrolled loops
template <class F, int... I>
__device__ __forceinline__ void nse_for_seq(F&& f, std::integer_sequence<int, I...>)
{
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void nse_for(F&& f)
{
    nse_for_seq(f, std::make_integer_sequence<int, N>{});
}
#define RBFX_INL __attribute__((always_inline))

// ---------------------------------------------------------------- broadcast FMAs
// Every block starts with two wait states: a DPP read of a register written by the
// previous VALU instructions needs them, and the compiler does not see into the block.
// All lanes are active wherever these run (the control flow around them is uniform).
#define RBFX_BC "row_newbcast:"
#define RBFX_BCM " row_mask:0xf bank_mask:0xf"

// v of lane LANE of the row, in all of its lanes
template <int LANE>
__device__ __forceinline__ double nse_bc(double v)
{
    double r;
    asm("s_nop 1\n\tv_mov_b64_dpp %0, %1 " RBFX_BC "%2" RBFX_BCM : "=v"(r) : "v"(v), "n"(LANE));
    return r;
}

#define RBFX_F_SAME(D, S) "v_fmac_f64_dpp " D ", " S ", %[m] " RBFX_BC "%[l]" RBFX_BCM "\n\t"

// d[i] += s[i](lane LANE) * m, i < CNT
template <int LANE, int CNT>
__device__ __forceinline__ void nse_fmac_row(double* d, const double* s, double m)
{
    if constexpr (CNT >= 8) {
        asm("s_nop 1\n\t" RBFX_F_SAME("%0", "%8") RBFX_F_SAME("%1", "%9") RBFX_F_SAME("%2", "%10")
                RBFX_F_SAME("%3", "%11") RBFX_F_SAME("%4", "%12") RBFX_F_SAME("%5", "%13") RBFX_F_SAME("%6", "%14")
                    RBFX_F_SAME("%7", "%15")
            : "+v"(d[0]), "+v"(d[1]), "+v"(d[2]), "+v"(d[3]), "+v"(d[4]), "+v"(d[5]), "+v"(d[6]), "+v"(d[7])
            : "v"(s[0]), "v"(s[1]), "v"(s[2]), "v"(s[3]), "v"(s[4]), "v"(s[5]), "v"(s[6]), "v"(s[7]), [m] "v"(m),
              [l] "n"(LANE));
        if constexpr (CNT > 8) nse_fmac_row<LANE, CNT - 8>(d + 8, s + 8, m);
    } else if constexpr (CNT >= 4) {
        asm("s_nop 1\n\t" RBFX_F_SAME("%0", "%4") RBFX_F_SAME("%1", "%5") RBFX_F_SAME("%2", "%6")
                RBFX_F_SAME("%3", "%7")
            : "+v"(d[0]), "+v"(d[1]), "+v"(d[2]), "+v"(d[3])
            : "v"(s[0]), "v"(s[1]), "v"(s[2]), "v"(s[3]), [m] "v"(m), [l] "n"(LANE));
        if constexpr (CNT > 4) nse_fmac_row<LANE, CNT - 4>(d + 4, s + 4, m);
    } else if constexpr (CNT >= 2) {
        asm("s_nop 1\n\t" RBFX_F_SAME("%0", "%2") RBFX_F_SAME("%1", "%3")
            : "+v"(d[0]), "+v"(d[1])
            : "v"(s[0]), "v"(s[1]), [m] "v"(m), [l] "n"(LANE));
        if constexpr (CNT > 2) nse_fmac_row<LANE, CNT - 2>(d + 2, s + 2, m);
    } else if constexpr (CNT == 1) {
        asm("s_nop 1\n\t" RBFX_F_SAME("%0", "%1") : "+v"(d[0]) : "v"(s[0]), [m] "v"(m), [l] "n"(LANE));
    }
}

// the same in place: d[i] += d[i](lane LANE) * m (lane LANE itself holds m = 0)
template <int LANE, int CNT>
__device__ __forceinline__ void nse_fmac_self(double* d, double m)
{
    if constexpr (CNT >= 8) {
        asm("s_nop 1\n\t" RBFX_F_SAME("%0", "%0") RBFX_F_SAME("%1", "%1") RBFX_F_SAME("%2", "%2")
                RBFX_F_SAME("%3", "%3") RBFX_F_SAME("%4", "%4") RBFX_F_SAME("%5", "%5") RBFX_F_SAME("%6", "%6")
                    RBFX_F_SAME("%7", "%7")
            : "+v"(d[0]), "+v"(d[1]), "+v"(d[2]), "+v"(d[3]), "+v"(d[4]), "+v"(d[5]), "+v"(d[6]), "+v"(d[7])
            : [m] "v"(m), [l] "n"(LANE));
        if constexpr (CNT > 8) nse_fmac_self<LANE, CNT - 8>(d + 8, m);
    } else if constexpr (CNT >= 4) {
        asm("s_nop 1\n\t" RBFX_F_SAME("%0", "%0") RBFX_F_SAME("%1", "%1") RBFX_F_SAME("%2", "%2")
                RBFX_F_SAME("%3", "%3")
            : "+v"(d[0]), "+v"(d[1]), "+v"(d[2]), "+v"(d[3])
            : [m] "v"(m), [l] "n"(LANE));
        if constexpr (CNT > 4) nse_fmac_self<LANE, CNT - 4>(d + 4, m);
    } else if constexpr (CNT >= 2) {
        asm("s_nop 1\n\t" RBFX_F_SAME("%0", "%0") RBFX_F_SAME("%1", "%1")
            : "+v"(d[0]), "+v"(d[1])
            : [m] "v"(m), [l] "n"(LANE));
        if constexpr (CNT > 2) nse_fmac_self<LANE, CNT - 2>(d + 2, m);
    } else if constexpr (CNT == 1) {
        asm("s_nop 1\n\t" RBFX_F_SAME("%0", "%0") : "+v"(d[0]) : [m] "v"(m), [l] "n"(LANE));
    }
}

// d[i] += s(lane LANE + i) * m, i < CNT
#define RBFX_F_LANE(D, L) "v_fmac_f64_dpp " D ", %[s], %[m] " RBFX_BC L RBFX_BCM "\n\t"
template <int LANE, int CNT>
__device__ __forceinline__ void nse_fmac_lanes(double* d, double s, double m)
{
    static_assert(LANE + CNT <= 16, "lanes of one row");
    if constexpr (CNT >= 8) {
        asm("s_nop 1\n\t" RBFX_F_LANE("%0", "%10") RBFX_F_LANE("%1", "%11") RBFX_F_LANE("%2", "%12")
                RBFX_F_LANE("%3", "%13") RBFX_F_LANE("%4", "%14") RBFX_F_LANE("%5", "%15") RBFX_F_LANE("%6", "%16")
                    RBFX_F_LANE("%7", "%17")
            : "+v"(d[0]), "+v"(d[1]), "+v"(d[2]), "+v"(d[3]), "+v"(d[4]), "+v"(d[5]), "+v"(d[6]), "+v"(d[7])
            : [s] "v"(s), [m] "v"(m), "n"(LANE), "n"(LANE + 1), "n"(LANE + 2), "n"(LANE + 3), "n"(LANE + 4),
              "n"(LANE + 5), "n"(LANE + 6), "n"(LANE + 7));
        if constexpr (CNT > 8) nse_fmac_lanes<LANE + 8, CNT - 8>(d + 8, s, m);
    } else if constexpr (CNT >= 4) {
        asm("s_nop 1\n\t" RBFX_F_LANE("%0", "%6") RBFX_F_LANE("%1", "%7") RBFX_F_LANE("%2", "%8")
                RBFX_F_LANE("%3", "%9")
            : "+v"(d[0]), "+v"(d[1]), "+v"(d[2]), "+v"(d[3])
            : [s] "v"(s), [m] "v"(m), "n"(LANE), "n"(LANE + 1), "n"(LANE + 2), "n"(LANE + 3));
        if constexpr (CNT > 4) nse_fmac_lanes<LANE + 4, CNT - 4>(d + 4, s, m);
    } else if constexpr (CNT >= 2) {
        asm("s_nop 1\n\t" RBFX_F_LANE("%0", "%4") RBFX_F_LANE("%1", "%5")
            : "+v"(d[0]), "+v"(d[1])
            : [s] "v"(s), [m] "v"(m), "n"(LANE), "n"(LANE + 1));
        if constexpr (CNT > 2) nse_fmac_lanes<LANE + 2, CNT - 2>(d + 2, s, m);
    } else if constexpr (CNT == 1) {
        asm("s_nop 1\n\t" RBFX_F_LANE("%0", "%3") : "+v"(d[0]) : [s] "v"(s), [m] "v"(m), "n"(LANE));
    }
}

// ---------------------------------------------------------------- per-group LDS
template <int DIM, int M, int NN, int RC>
struct NseLds {
    static constexpr int MP = M | 1;                       // odd row stride: a column read by 16 lanes
    static constexpr int ROWS = NN + RC > M ? NN + RC : M;  //   and a row per lane are both conflict-free
    // scaled coordinates, then L_B rows, then C rows, then the lanes' shares of a residual
    double buf[(ROWS > 16 ? ROWS : 16) * MP];
    double aux[RC > 2 ? RC * M : 2 * M];       // L P rows, then pivot rows (two), then b_B
    double h;                                  // the scale 1 / h of the offsets
    int32_t src[M + NN];                       // stencil index of each position
};

// Stencil e (n rows) to the list of what the rook-pivoted kernels solve: the launch's own, or
// in a ragged launch its size bucket's.
template <bool RAG>
__device__ __forceinline__ void nse_hand_back(const BuildDev& P, bool yes, int64_t e, int n)
{
    if (!yes || !P.fail_list) return;
    const int b = !RAG ? 0 : (n <= 32 ? 0 : (n <= 64 ? 1 : 2));
    const int q = atomicAdd(P.fail_count + b, 1);
    P.fail_list[b * P.fail_stride + q] = (int32_t)e;
}

// position of the monomial x_i x_j in the graded order (fill_mono_table)
template <int DIM>
__device__ __forceinline__ int nse_pair(int i, int j)
{
    const int a = i < j ? i : j, b = i < j ? j : i;
    if constexpr (DIM == 2) return 3 + a + b;
    return 4 + (a == 0 ? b : (a == 1 ? 2 + b : 5));
}

// KIND PHS3, PHS5 or PHS7 (a compile-time constant: with a switch around the loops the
// compiler hoists the square roots common to its cases and holds all of them); DIM 2 or
// 3; M monomials; up to NN null points (k - M); up to RC operator columns; W
// waves per SIMD the register allocation targets; RAG: the stencils of a wavefront differ in
// k (loops run to the longest of the four; a step past a stencil's own points multiplies
// its rows by zero)
template <int KIND, int DIM, int M, int NN, int RC, int W, bool RAG>
__global__ __attribute__((amdgpu_flat_work_group_size(64, 64), amdgpu_waves_per_eu(W))) void
k_nse(const BuildDev P)
{
    constexpr int SLP = (M + NN + RC + 15) / 16;  // slots of the points and operator columns
    constexpr int SLN = (NN + RC + 15) / 16;      // slots of the null points and operator columns
    constexpr int SLB = (M + 15) / 16;            // slots of the basic points
    constexpr int GL = 16 - RC;                   // first lane (last slot) of the operator columns
    using Lds = NseLds<DIM, M, NN, RC>;
    constexpr int MP = Lds::MP;
    static_assert((M + NN) * DIM <= Lds::ROWS * MP, "coordinates fit the row buffer");
    __shared__ Lds s_st[4];

    const int L = lane_id();
    const int g = L >> 4, li = L & 15;
    Lds& S_ = s_st[g];
    const int64_t lb = xcd_contiguous_block(P.n_blocks);
    if (lb < 0) return;  // padding block: the whole workgroup leaves
    const int64_t n_work = P.list ? (int64_t)*P.list_len : P.n_eval;
    const int64_t wi = lb * 4 + g;
    int alive = wi < n_work;
    int64_t e = alive ? (P.list ? (int64_t)P.list[wi] : (P.order ? (int64_t)P.order[wi] : wi)) : 0;
    if (e < 0 || e >= P.n_eval) {
        alive = 0;
        e = 0;
    }
    // Uniform builds (the host checks k - M <= NN and the column count): kk and nn are
    // scalars. A group without work repeats stencil 0 and writes nothing. Ragged ones: kk
    // and nn are the group's; a stencil outside the class is handed back.
    int kk = P.k, nn = kk - M, nnw = nn;
    int64_t s0 = e * (int64_t)kk;
    int rag_ok = 1;
    if constexpr (RAG) {
        if (P.adj_ptr) {
            s0 = P.adj_ptr[e];
            kk = (int)(P.adj_ptr[e + 1] - s0);
        }
        rag_ok = stencil_n_mono(P, e, DIM) == M && kk > M && kk - M <= NN;
        nn = rag_ok ? kk - M : 1;
        nnw = max(max(__builtin_amdgcn_readlane(nn, 0), __builtin_amdgcn_readlane(nn, 16)),
                  max(__builtin_amdgcn_readlane(nn, 32), __builtin_amdgcn_readlane(nn, 48)));
    }
    const int kp = M + nn;  // points of the arithmetic
    const int n_cols = P.n_cols, n_terms = P.n_terms;
    int handoff = 0, fail = 0;
    if (RAG && alive && !rag_ok) {
        handoff = 1;
        alive = 0;
    }

    // ---- points li + 16 s: offsets from the evaluation point
    double x[SLP][DIM], hinv;
    int isp[SLP];
    {
        double xe[DIM];
#pragma unroll
        for (int d = 0; d < DIM; ++d) xe[d] = P.eval[e * DIM + d];
        double r2max = 0.0;
        bool ib = P.is_boundary && e < P.n_data && P.is_boundary[e];
#pragma unroll
        for (int s = 0; s < SLP; ++s) {
            const int q = li + 16 * s;
            isp[s] = q < kp;
            const int32_t idx = rag_ok ? P.adj_idx[s0 + (q < kp ? q : 0)] : 0;
            double r2 = 0.0;
#pragma unroll
            for (int d = 0; d < DIM; ++d) {
                x[s][d] = P.data[(int64_t)idx * DIM + d] - xe[d];
                r2 += x[s][d] * x[s][d];
            }
            r2max = fmax(r2max, r2);  // (lanes past the stencil repeat its first point)
            if (P.is_boundary) ib = ib || P.is_boundary[idx];
        }
        // Hermite stencils are the rook kernels' work (the ballot is over whole wavefronts,
        // each group reads its own 16 bits)
        if (P.is_boundary) {
            if (((__ballot(ib) >> (16 * g)) & 0xffffull) != 0ull) {
                handoff = handoff | alive;
                alive = 0;
            }
        }
        if (RAG && __ballot(alive) == 0ull) {  // (a wavefront of hand-backs or padding)
            nse_hand_back<RAG>(P, handoff && li == 0, e, kk + M);
            return;
        }
        // scaled by a power of two, so the scaling rounds nothing (|x| < 1; a PHS build's
        // weights do not depend on the scale)
        r2max = gmax<16>(r2max);
        int ex = 0;
        if (r2max > 0.0 && r2max < 1e300) ex = -((__builtin_amdgcn_frexp_exp(r2max) + 1) >> 1);
#pragma unroll
        for (int s = 0; s < SLP; ++s)
#pragma unroll
            for (int d = 0; d < DIM; ++d) x[s][d] = __builtin_amdgcn_ldexp(x[s][d], ex);
        hinv = __builtin_amdgcn_ldexp(1.0, ex);
    }

    // ---- rows of P: monomials of the points; on the last lanes of the last slot the operator
    // columns' polynomial right-hand sides
    const bool isg = li >= GL;
    const int gc = isg ? li - GL : 0;
    // the operator columns' polynomial right-hand sides L P(x_e), into aux by the lanes isg (x_e
    // is the origin, so a term reaches only the monomial of its own exponents)
    auto poly_rhs = [&](double hinv) RBFX_INL {
#pragma unroll
        for (int a = 0; a < M; ++a) S_.aux[gc * M + a] = 0.0;
        if (isg) {
            for (int t = 0; t < n_terms; ++t) {
                const TermDev tm = P.terms[t];
                const double sc1 = tm.coeff * hinv, sc2 = sc1 * hinv;
                int idx = 0;
                double v = tm.coeff;
                if (tm.kind == RBFX_OP_D1) {
                    idx = 1 + tm.d1;
                    v = sc1;
                } else if (tm.kind == RBFX_OP_D2 || (tm.kind == RBFX_OP_MIXED && tm.d1 == tm.d2)) {
                    idx = nse_pair<DIM>(tm.d1, tm.d1);
                    v = 2.0 * sc2;
                } else if (tm.kind == RBFX_OP_MIXED) {
                    idx = nse_pair<DIM>(tm.d1, tm.d2);
                    v = sc2;
                } else if (tm.kind == RBFX_OP_LAP) {
                    idx = nse_pair<DIM>(0, 0);
                    v = 2.0 * sc2;
                }
                if (tm.col == gc) {
                    if (idx < M) S_.aux[gc * M + idx] += v;
                    if (tm.kind == RBFX_OP_LAP) {
#pragma unroll
                        for (int d = 1; d < DIM; ++d) {
                            const int id = nse_pair<DIM>(d, d);
                            if (id < M) S_.aux[gc * M + id] += v;
                        }
                    }
                }
            }
        }
    };
    double p[SLP][M];
    {
        S_.h = hinv;
        poly_rhs(hinv);
        // (lanes past the stencil hold its first point again; they are never candidates, and
        // what the LU leaves in them is not used)
        nse_for<M>([&](auto a) RBFX_INL {
#pragma unroll
            for (int s = 0; s < SLP; ++s) p[s][a.value] = mono_graded<DIM>(a.value, x[s]);
        });
#pragma unroll
        for (int a = 0; a < M; ++a) {
            const double v = S_.aux[gc * M + a];
            p[SLP - 1][a] = isg ? v : p[SLP - 1][a];
        }
        __syncthreads();
    }

    // ---- LU of P with row pivoting over the points. Every row is eliminated at every step,
    // also the ones already chosen: p[s][a] is left holding -L for every row that was not
    // yet a pivot at step a, and what later steps leave in a pivot row is not used. A
    // candidate's key packs the magnitude's leading bits with the point index (ties and
    // near-ties, to 2^-14, go to the nearer point); 0 for rows that are no candidates.
    uint32_t kmask[SLP], kidx[SLP];
    int pos[SLP];
#pragma unroll
    for (int s = 0; s < SLP; ++s) {
        kmask[s] = isp[s] ? 0x7fffffc0u : 0u;
        kidx[s] = isp[s] ? (uint32_t)(63 - (li + 16 * s)) : 0u;
        pos[s] = -1;
    }
    nse_for<M>([&](auto ac) RBFX_INL {
        constexpr int a = ac.value;
        uint32_t key = 0;
#pragma unroll
        for (int s = 0; s < SLP; ++s) {
            const uint32_t hi = (uint32_t)((unsigned long long)__double_as_longlong(p[s][a]) >> 32);
            key = max(key, (hi & kmask[s]) | kidx[s]);
        }
        key = group_max_u32<16>(key);
        const int q = 63 - (int)(key & 63u);
        double* row = S_.aux + (a & 1) * M;
#pragma unroll
        for (int s = 0; s < SLP; ++s) {
            const bool own = q == li + 16 * s;
            if (own) {
#pragma unroll
                for (int c = a; c < M; ++c) row[c] = p[s][c];
            }
            pos[s] = own ? a : pos[s];
            kmask[s] = own ? 0u : kmask[s];
            kidx[s] = own ? 0u : kidx[s];
        }
        __syncthreads();
        double rc[M];
#pragma unroll
        for (int c = a; c < M; ++c) rc[c] = row[c];
        if (!(fabs(rc[a]) > kNseLuTol && fabs(rc[a]) < 1e300)) fail = 1;
        const double nrp = -nsc_rcp(rc[a]);
#pragma unroll
        for (int s = 0; s < SLP; ++s) {
            p[s][a] *= nrp;
#pragma unroll
            for (int c = a + 1; c < M; ++c) p[s][c] = fma(p[s][a], rc[c], p[s][c]);
        }
        // (results pinned to this step: sunk to their uses, they would hold the step's
        // multipliers and pivot row in registers)
#pragma unroll
        for (int s = 0; s < SLP; ++s)
#pragma unroll
            for (int c = a; c < M; ++c) asm volatile("" : "+v"(p[s][c]));
        asm volatile("" : "+v"(fail));
    });

    // positions: basic points 0..M-1 in pivot order, null points M.. in stencil order
    {
        int base = M;
#pragma unroll
        for (int s = 0; s < SLP; ++s) {
            const bool nl = isp[s] && pos[s] < 0;
            const uint32_t m = (uint32_t)(__ballot(nl) >> (16 * g)) & 0xffffu;
            if (nl) pos[s] = base + __popc(m & ((1u << li) - 1u));
            base += __popc(m);
        }
    }

    // ---- change of layout: coordinates and stencil indices, then the rows of C
    double xb[SLB][DIM], xn[SLN][DIM];
#pragma unroll
    for (int s = 0; s < SLP; ++s) {
        if (pos[s] >= 0) {
#pragma unroll
            for (int d = 0; d < DIM; ++d) S_.buf[pos[s] * DIM + d] = x[s][d];
            S_.src[pos[s]] = li + 16 * s;
        }
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < SLB; ++s) {
        const int b = li + 16 * s < M ? li + 16 * s : M - 1;
#pragma unroll
        for (int d = 0; d < DIM; ++d) xb[s][d] = S_.buf[b * DIM + d];
    }
#pragma unroll
    for (int t = 0; t < SLN; ++t) {
        const int i = M + (li + 16 * t < nn ? li + 16 * t : nn - 1);
#pragma unroll
        for (int d = 0; d < DIM; ++d) xn[t][d] = S_.buf[i * DIM + d];
    }
    __syncthreads();
    // C = L_N L_B^-1, rows of the null points and of the operator columns (-C is held): entry b
    // is final once the entries above it have been applied. Up to ten monomials L_B moves
    // to the basic points' lanes and is broadcast from there, after the rows of C have
    // moved; beyond, its rows are read from LDS before they move (the rows of P, L_B and C
    // would not fit the registers together).
    constexpr bool CREG = M <= 10;
    double nlb[SLB][CREG ? M : 1];  // -L_B
#pragma unroll
    for (int s = 0; s < SLP; ++s) {
        if (pos[s] >= 0 && pos[s] < M) {
#pragma unroll
            for (int a = 0; a < M - 1; ++a) S_.buf[pos[s] * MP + a] = p[s][a];
        }
    }
    __syncthreads();
    if constexpr (CREG) {
#pragma unroll
        for (int s = 0; s < SLB; ++s) {
            const int b = li + 16 * s < M ? li + 16 * s : M - 1;
#pragma unroll
            for (int a = 0; a < M - 1; ++a) nlb[s][a] = S_.buf[b * MP + a];
        }
    } else {
        nse_for<M - 1>([&](auto ib) RBFX_INL {
            constexpr int b = M - 1 - ib.value;
            asm volatile("" ::: "memory");  // (one row of L_B in flight, not all of them)
            double l[M];
#pragma unroll
            for (int a = 0; a < b; ++a) l[a] = S_.buf[b * MP + a];
#pragma unroll
            for (int s = 0; s < SLP; ++s)
#pragma unroll
                for (int a = 0; a < b; ++a) p[s][a] = fma(p[s][b], l[a], p[s][a]);
#pragma unroll
            for (int s = 0; s < SLP; ++s)
#pragma unroll
                for (int a = 0; a < b; ++a) asm volatile("" : "+v"(p[s][a]));
        });
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < SLP; ++s) {
        if (pos[s] >= M || (s == SLP - 1 && isg)) {
            const int r = pos[s] >= M ? pos[s] - M : NN + gc;
#pragma unroll
            for (int a = 0; a < M; ++a) S_.buf[r * MP + a] = p[s][a];
        }
    }
    __syncthreads();
    int crow[SLN];  // own row of C in the buffer
#pragma unroll
    for (int t = 0; t < SLN; ++t)
        crow[t] = ((t == SLN - 1 && isg) ? NN + gc : (li + 16 * t < nn ? li + 16 * t : nn - 1)) * MP;
    double cr[SLN][CREG ? M : 1];
    if constexpr (CREG) {
#pragma unroll
        for (int t = 0; t < SLN; ++t)
#pragma unroll
            for (int a = 0; a < M; ++a) cr[t][a] = S_.buf[crow[t] + a];
        nse_for<M - 1>([&](auto ib) RBFX_INL {
            constexpr int b = M - 1 - ib.value;
#pragma unroll
            for (int t = 0; t < SLN; ++t) nse_fmac_row<b % 16, b>(cr[t], nlb[b / 16], cr[t][b]);
        });
        __syncthreads();
        // back to LDS for the column reads at the end
#pragma unroll
        for (int t = 0; t < SLN; ++t)
            if ((t == SLN - 1 && isg) || li + 16 * t < nn) {
#pragma unroll
                for (int a = 0; a < M; ++a) S_.buf[crow[t] + a] = cr[t][a];
            }
    }
    auto cn_at = [&](const int t, const int a) RBFX_INL {
        if constexpr (CREG) return cr[t][a];
        else return S_.buf[crow[t] + a];
    };

    // ---- L phi at the own null and basic points, per operator column
    double sn[SLN][NN + RC];  // rows of [S | t]
    {
        double bb[SLB][RC];
        auto rhs = [&](const double (&xi)[DIM], double (&out)[RC]) RBFX_INL {
            double q2 = 0.0;
#pragma unroll
            for (int d = 0; d < DIM; ++d) q2 += xi[d] * xi[d];
            const double r = nsc_sqrt(q2);
            // r^(p-2) and r^(p-4) of phi = r^p (for p = 3 the latter as 1 / (r + 1e-16))
            constexpr double pw = KIND;
            double rp2 = r, rp4;
            if constexpr (KIND == RBFX_PHS3) {
                rp4 = nsc_rcp(r + kAvoidInf);
            } else if constexpr (KIND == RBFX_PHS5) {
                rp2 = r * q2;
                rp4 = r;
            } else {
                rp2 = r * (q2 * q2);
                rp4 = r * q2;
            }
#pragma unroll
            for (int c = 0; c < RC; ++c) out[c] = 0.0;
            for (int t = 0; t < n_terms; ++t) {
                const TermDev tm = P.terms[t];
                double d1 = 0.0, d2 = 0.0;  // (offset x_e - x_j = -xi)
#pragma unroll
                for (int d = 0; d < DIM; ++d) {
                    if (d == tm.d1) d1 = -xi[d];
                    if (d == tm.d2) d2 = -xi[d];
                }
                double v;
                if (tm.kind == RBFX_OP_VALUE) {
                    v = tm.coeff * (q2 * rp2);
                } else if (tm.kind == RBFX_OP_D1) {
                    v = (tm.coeff * hinv) * (pw * d1 * rp2);
                } else if (tm.kind == RBFX_OP_LAP) {
                    v = (tm.coeff * hinv * hinv) * ((pw * (pw + 1.0)) * rp2);
                } else if (tm.kind == RBFX_OP_D2 || tm.d1 == tm.d2) {
                    v = (tm.coeff * hinv * hinv) * (pw * fma((pw - 2.0) * (d1 * d1), rp4, rp2));
                } else {
                    v = (tm.coeff * hinv * hinv) * (pw * (pw - 2.0) * (d1 * d2) * rp4);
                }
#pragma unroll
                for (int c = 0; c < RC; ++c)
                    if (tm.col == c) out[c] += v;
            }
        };
#pragma unroll
        for (int s = 0; s < SLB; ++s) {
            rhs(xb[s], bb[s]);
            if (li + 16 * s < M) {
#pragma unroll
                for (int c = 0; c < RC; ++c) S_.aux[c * M + li + 16 * s] = bb[s][c];
            }
        }
#pragma unroll
        for (int t = 0; t < SLN; ++t) {
            double bn[RC];
            rhs(xn[t], bn);
#pragma unroll
            for (int c = 0; c < RC; ++c) sn[t][NN + c] = bn[c];
        }
        __syncthreads();
    }

    // coordinates of the point that lane LANE holds in slot XO (written by ordinary
    // instructions, so the compiler places the wait states of the moves)
#define RBFX_NSE_POINT(O, XO, LANE)                                                               \
    double O[DIM];                                                                                \
    _Pragma("unroll") for (int d = 0; d < DIM; ++d) O[d] = __longlong_as_double(                  \
        __builtin_amdgcn_mov_dpp(__double_as_longlong(XO[d]), 0x150 + (LANE), 0xF, 0xF, true));
    auto phi_at = [&](const double (&xa)[DIM], const double (&o)[DIM]) RBFX_INL {
        double q2 = 0.0;
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            const double t = xa[d] - o[d];
            q2 = fma(t, t, q2);
        }
        return phi_kind<KIND>(0.0, q2);
    };

    // ---- T = Phi_NB + (-C) Phi_BB / 2 (operator columns: b_B in place of Phi_NB). Phi_NB is
    // added last, and Phi_NN below between the two halves of its sum: sums that start from it
    // round at its size in every step. Error of the weights over that of the kernels that took
    // these builds before, 14 shapes of 10 monomials and more: 1.13 in the geometric mean with
    // sums that start from phi, 0.93 in this order (2M 3-D stencils of 60 rows: 11.8 and 12.4 ms).
    double T[SLN][M];
    {
        double bbm[SLB][M];
        nse_for<M>([&](auto b) RBFX_INL {
            RBFX_NSE_POINT(o, xb[b.value / 16], b.value % 16)
#pragma unroll
            for (int s = 0; s < SLB; ++s) bbm[s][b.value] = phi_at(xb[s], o);
            if constexpr (SLN + SLB > 2) {
                // (one point's values at a time)
#pragma unroll
                for (int s = 0; s < SLB; ++s) asm volatile("" : "+v"(bbm[s][b.value]));
            }
        });
#pragma unroll
        for (int t = 0; t < SLN; ++t)
#pragma unroll
            for (int a = 0; a < M; ++a) T[t][a] = 0.0;
        nse_for<M>([&](auto b) RBFX_INL {
            if constexpr (!CREG && b.value % 2 == 0) asm volatile("" ::: "memory");
#pragma unroll
            for (int t = 0; t < SLN; ++t)
                nse_fmac_row<b.value % 16, M>(T[t], bbm[b.value / 16], 0.5 * cn_at(t, b.value));
            if constexpr (!CREG) __builtin_amdgcn_sched_barrier(0);
        });
#pragma unroll
        for (int t = 0; t < SLN; ++t)
#pragma unroll
            for (int a = 0; a < M; ++a) asm volatile("" : "+v"(T[t][a]));
    }
    // (or the broadcasts of the loop above would be kept for this one)
#pragma unroll
    for (int s = 0; s < SLB; ++s)
#pragma unroll
        for (int d = 0; d < DIM; ++d) asm volatile("" : "+v"(xb[s][d]));
    if constexpr (SLN + SLB > 2) __builtin_amdgcn_sched_barrier(0);
    nse_for<M>([&](auto b) RBFX_INL {
        RBFX_NSE_POINT(o, xb[b.value / 16], b.value % 16)
        const double g_ = S_.aux[gc * M + b.value];
#pragma unroll
        for (int t = 0; t < SLN; ++t) {
            const double v = phi_at(xn[t], o);
            T[t][b.value] += t == SLN - 1 && isg ? g_ : v;
        }
        if constexpr (SLN + SLB > 2) {
#pragma unroll
            for (int t = 0; t < SLN; ++t) asm volatile("" : "+v"(T[t][b.value]));
            __builtin_amdgcn_sched_barrier(0);
        }
    });

    // the largest |T| of the null points (its leading bits; infinity, which no pivot passes, for a NaN)
    double tscale;
    {
        uint32_t hi = 0;
#pragma unroll
        for (int t = 0; t < SLN; ++t)
#pragma unroll
            for (int a = 0; a < M; ++a) {
                const uint32_t h = (uint32_t)((unsigned long long)__double_as_longlong(T[t][a]) >> 32) & 0x7fffffffu;
                hi = max(hi, t == SLN - 1 && isg ? 0u : h);
            }
        hi = min(group_max_u32<16>(hi), 0x7ff00000u);
        tscale = __longlong_as_double((long long)((unsigned long long)hi << 32));
    }

    // ---- S = Phi_NN + T (-C)^T + (-C) T^T, and the same for the operator columns
#pragma unroll
    for (int t = 0; t < SLN; ++t)
#pragma unroll
        for (int j = 0; j < NN; ++j) sn[t][j] = 0.0;
    // columns of S in chunks of eight: += (-C) T^T, then += T (-C)^T
    auto half = [&](auto second) RBFX_INL {
        nse_for<(NN + 7) / 8>([&](auto ch) RBFX_INL {
            constexpr int j0 = 8 * ch.value, cnt = NN - j0 < 8 ? NN - j0 : 8, jt = j0 / 16, jl = j0 % 16;
            if (j0 < nnw) {
                if constexpr (!CREG) asm volatile("" ::: "memory");  // (reread, not kept from the last chunk)
#pragma unroll
                for (int a = 0; a < M; ++a) {
                    const double cj = cn_at(jt, a);
#pragma unroll
                    for (int t = 0; t < SLN; ++t) {
                        if constexpr (decltype(second)::value) nse_fmac_lanes<jl, cnt>(&sn[t][j0], cj, T[t][a]);
                        else nse_fmac_lanes<jl, cnt>(&sn[t][j0], T[jt][a], cn_at(t, a));
                    }
                    if constexpr (!CREG) __builtin_amdgcn_sched_barrier(0);
                }
                // (pinned: sunk to their uses, the sums would hold their operands)
#pragma unroll
                for (int t = 0; t < SLN; ++t)
#pragma unroll
                    for (int q = 0; q < cnt; ++q) asm volatile("" : "+v"(sn[t][j0 + q]));
            }
        });
    };
    half(std::false_type{});
    if constexpr (SLN > 1) __builtin_amdgcn_sched_barrier(0);
    nse_for<NN>([&](auto j) RBFX_INL {
        RBFX_NSE_POINT(o, xn[j.value / 16], j.value % 16)
#pragma unroll
        for (int t = 0; t < SLN; ++t) {
            sn[t][j.value] += phi_at(xn[t], o);
            asm volatile("" : "+v"(sn[t][j.value]));
        }
        if constexpr (SLN > 1 && j.value % 2 == 1) __builtin_amdgcn_sched_barrier(0);
    });
#undef RBFX_NSE_POINT
    if constexpr (SLN > 1) __builtin_amdgcn_sched_barrier(0);
    half(std::true_type{});
    if constexpr (!CREG) asm volatile("" ::: "memory");
#pragma unroll
    for (int a = 0; a < M; ++a) {
        double ca[SLN];
#pragma unroll
        for (int t = 0; t < SLN; ++t) ca[t] = cn_at(t, a);
#pragma unroll
        for (int t = 0; t < SLN; ++t) {
            nse_fmac_lanes<GL, RC>(&sn[t][NN], ca[SLN - 1], T[t][a]);
            nse_fmac_lanes<GL, RC>(&sn[t][NN], T[SLN - 1][a], ca[t]);
        }
        if constexpr (!CREG) __builtin_amdgcn_sched_barrier(0);
    }

    // ---- Gauss-Jordan on [S | t]: every row but the pivot's, every later column
    double dinv[SLN];
#pragma unroll
    for (int t = 0; t < SLN; ++t) dinv[t] = 0.0;
    {
        constexpr double sg = KIND == RBFX_PHS5 ? -1.0 : 1.0;  // (nsc_sign)
        double dmax = tscale;
        nse_for<NN>([&](auto jc) RBFX_INL {
            constexpr int j = jc.value, jt = j / 16, jl = j % 16, rest = NN - 1 - j;
            if (j < nnw) {
                const double piv = nse_bc<jl>(sn[jt][j]);
                const double ap = sg * piv;
                const bool has = !RAG || j < nn;
                dmax = has ? fmax(dmax, ap) : dmax;
                if (has && !(ap > kNsePivTol * dmax)) fail = 1;
                asm volatile("" : "+v"(fail));
                double rd = nsc_rcp(piv);
                if constexpr (RAG) rd = has ? rd : 0.0;
                const bool own = li == jl;
                dinv[jt] = own ? rd : dinv[jt];
                double nl[SLN];
#pragma unroll
                for (int t = 0; t < SLN; ++t) {
                    nl[t] = -(sn[t][j] * rd);
                    if (t == jt) nl[t] = own ? 0.0 : nl[t];
                }
#pragma unroll
                for (int t = 0; t < SLN; ++t) {
                    if (t != jt) {
                        nse_fmac_row<jl, rest>(&sn[t][j + 1], &sn[jt][j + 1], nl[t]);
                        nse_fmac_row<jl, RC>(&sn[t][NN], &sn[jt][NN], nl[t]);
                    }
                }
                nse_fmac_self<jl, rest>(&sn[jt][j + 1], nl[jt]);
                nse_fmac_self<jl, RC>(&sn[jt][NN], nl[jt]);
            }
        });
    }

    // ---- w_N, and w_B = w0 - C^T w_N: lane b reads column b of -C from LDS
    double wb[SLB][RC];
    {
        double u[SLN][RC];
        int qb[SLB], qn[SLN];  // stencil index of the own points
#pragma unroll
        for (int t = 0; t < SLN; ++t)
#pragma unroll
            for (int c = 0; c < RC; ++c) u[t][c] = sn[t][NN + c] * dinv[t];
#pragma unroll
        for (int s = 0; s < SLB; ++s) {
            const int b = li + 16 * s < M ? li + 16 * s : M - 1;
#pragma unroll
            for (int c = 0; c < RC; ++c) wb[s][c] = -S_.buf[(NN + c) * MP + b];
        }
        nse_for<NN>([&](auto i) RBFX_INL {
            if (i.value < nnw) {
#pragma unroll
                for (int s = 0; s < SLB; ++s) {
                    const int b = li + 16 * s < M ? li + 16 * s : M - 1;
                    double cv = S_.buf[i.value * MP + b];
                    if constexpr (RAG) cv = i.value < nn ? cv : 0.0;
                    nse_fmac_row<i.value % 16, RC>(wb[s], u[i.value / 16], cv);
                }
            }
        });
        // ---- The polynomial conditions P^T w = L P, corrected once: C carries the rounding of its
        // elimination, so they hold to two or three times what the weights' own rounding
        // leaves, and that, not the weights' error, is what an applied operator shows on a
        // smooth field. Their residual r, summed over the stencil's points, and P_B^T dw = r by
        // Gauss-Jordan steps (lane b holds condition b; the reciprocals need few digits). The
        // points are fetched again: kept, they would cost registers in every phase.
        // Applied operators' error over that of the kernels that took the builds before, 130
        // shapes and clouds: 1.44 in the geometric mean without this step, 0.76 with it (4M 2-D
        // stencils of 26 rows 3.2 -> 3.5 ms, 2M 3-D ones of 60 rows 12.4 -> 13.9 ms).
        {
#pragma unroll
            for (int s = 0; s < SLB; ++s)
#pragma unroll
                for (int c = 0; c < RC; ++c) asm volatile("" : "+v"(wb[s][c]));
            __syncthreads();
            const double hs = S_.h;
            int lq = li;  // (its own addresses, or those of the phases above would be kept)
            asm volatile("" : "+v"(lq));
#pragma unroll
            for (int s = 0; s < SLB; ++s) qb[s] = S_.src[lq + 16 * s < M ? lq + 16 * s : M - 1];
#pragma unroll
            for (int t = 0; t < SLN; ++t) qn[t] = S_.src[M + (lq + 16 * t < nn ? lq + 16 * t : nn - 1)];
            double yb[SLB][DIM], yn[SLN][DIM];
            auto point = [&](int q, double (&y)[DIM]) RBFX_INL {
                const int64_t idx = rag_ok ? P.adj_idx[s0 + q] : 0;
#pragma unroll
                for (int d = 0; d < DIM; ++d) y[d] = (P.data[idx * DIM + d] - P.eval[e * DIM + d]) * hs;
            };
#pragma unroll
            for (int s = 0; s < SLB; ++s) point(qb[s], yb[s]);
#pragma unroll
            for (int t = 0; t < SLN; ++t) point(qn[t], yn[t]);
            // (beyond ten monomials their values are made again for each use, not held)
            auto renew = [&]() RBFX_INL {
                if constexpr (!CREG) {
#pragma unroll
                    for (int d = 0; d < DIM; ++d) {
#pragma unroll
                        for (int s = 0; s < SLB; ++s) asm volatile("" : "+v"(yb[s][d]));
#pragma unroll
                        for (int t = 0; t < SLN; ++t) asm volatile("" : "+v"(yn[t][d]));
                    }
                }
            };
            poly_rhs(hs);
            double rr[SLB][RC];
#pragma unroll
            for (int c = 0; c < RC; ++c) {
                double mb[SLB], mn[SLN];
#pragma unroll
                for (int s = 0; s < SLB; ++s) mb[s] = lq + 16 * s < M ? -wb[s][c] : 0.0;
#pragma unroll
                for (int t = 0; t < SLN; ++t) mn[t] = lq + 16 * t < nn ? -u[t][c] : 0.0;
                renew();
                nse_for<M>([&](auto a) RBFX_INL {
                    if constexpr (!CREG) __builtin_amdgcn_sched_barrier(0);
                    double v = 0.0;
#pragma unroll
                    for (int s = 0; s < SLB; ++s) v = fma(mono_graded<DIM>(a.value, yb[s]), mb[s], v);
#pragma unroll
                    for (int t = 0; t < SLN; ++t) v = fma(mono_graded<DIM>(a.value, yn[t]), mn[t], v);
                    S_.buf[lq * MP + a.value] = v;
                });
                __syncthreads();
#pragma unroll
                for (int s = 0; s < SLB; ++s) {
                    const int b = lq + 16 * s < M ? lq + 16 * s : M - 1;
                    double v = S_.aux[c * M + b];
#pragma unroll
                    for (int l = 0; l < 16; ++l) v += S_.buf[l * MP + b];
                    rr[s][c] = v;
                    asm volatile("" : "+v"(rr[s][c]));
                }
                __syncthreads();
            }
            renew();
#pragma unroll
            for (int s = 0; s < SLB; ++s)
                if (lq + 16 * s < M) {
                    nse_for<M>([&](auto a) RBFX_INL {
                        S_.buf[(lq + 16 * s) * MP + a.value] = mono_graded<DIM>(a.value, yb[s]);
                    });
                }
            __syncthreads();
            double q[SLB][M], dq[SLB];
#pragma unroll
            for (int s = 0; s < SLB; ++s) {
                const int b = lq + 16 * s < M ? lq + 16 * s : M - 1;
                dq[s] = 0.0;
#pragma unroll
                for (int a = 0; a < M; ++a) q[s][a] = S_.buf[a * MP + b];
            }
            nse_for<M>([&](auto jc) RBFX_INL {
                constexpr int j = jc.value, js = j / 16, jl = j % 16, rest = M - 1 - j;
                const double rd = __builtin_amdgcn_rcp(nse_bc<jl>(q[js][j]));
                const bool own = lq == jl;
                dq[js] = own ? rd : dq[js];
#pragma unroll
                for (int s = 0; s < SLB; ++s) {
                    if (s != js) {
                        const double nl = -(q[s][j] * rd);
                        nse_fmac_row<jl, rest>(&q[s][j + 1], &q[js][j + 1], nl);
                        nse_fmac_row<jl, RC>(rr[s], rr[js], nl);
                    }
                }
                const double nl = own ? 0.0 : -(q[js][j] * rd);
                nse_fmac_self<jl, rest>(&q[js][j + 1], nl);
                nse_fmac_self<jl, RC>(rr[js], nl);
            });
#pragma unroll
            for (int s = 0; s < SLB; ++s)
#pragma unroll
                for (int c = 0; c < RC; ++c) {
                    wb[s][c] = fma(rr[s][c], dq[s], wb[s][c]);
                    asm volatile("" : "+v"(wb[s][c]));  // (here, with all lanes active)
                }
        }
        if (alive && !fail) {
            const int64_t o0 = P.out_ptr ? P.out_ptr[e] : s0;
#pragma unroll
            for (int t = 0; t < SLN; ++t)
                if (li + 16 * t < nn) {
#pragma unroll
                    for (int c = 0; c < RC; ++c)
                        if (c < n_cols) P.out_val[(int64_t)c * P.out_nnz + o0 + qn[t]] = u[t][c];
                }
#pragma unroll
            for (int s = 0; s < SLB; ++s)
                if (li + 16 * s < M) {
#pragma unroll
                    for (int c = 0; c < RC; ++c)
                        if (c < n_cols) P.out_val[(int64_t)c * P.out_nnz + o0 + qb[s]] = wb[s][c];
                }
            if (P.out_col)
                for (int q = li; q < kp; q += 16) P.out_col[o0 + q] = P.adj_idx[s0 + q];
            if (li == 0 && P.status) P.status[e] = P.ok_status;
        }
    }
    nse_hand_back<RAG>(P, (handoff || (alive && fail)) && li == 0, e, kk + M);
}

template <int KIND, int DIM, int M, int NN, int RC, int W, bool RAG = false>
inline hipError_t launch_nse_one(const BuildDev& P, int64_t n_work, hipStream_t s)
{
    if (n_work <= 0) return hipSuccess;
    BuildDev Q = P;
    Q.n_blocks = (n_work + 3) / 4;
    hipLaunchKernelGGL((k_nse<KIND, DIM, M, NN, RC, W, RAG>), dim3((unsigned)pad_to_xcds(Q.n_blocks)), dim3(64), 0, s, Q);
    return hipGetLastError();
}

// The instantiation of fewest slots that holds the stencil: null points and operator columns
// within one slot of 16 lanes (also the basic points, up to six monomials: one slot less
// in the LU), or two. W follows the registers each needs without scratch memory.
template <int KIND, int DIM, int M, int RC>
inline hipError_t launch_nse_m(const BuildDev& P, int64_t n_work, hipStream_t s)
{
    const int nn = P.k - M;
    if (nn < 1) return hipErrorInvalidValue;
    if constexpr (M <= 6) {
        if (nn <= 16 - M - RC) return launch_nse_one<KIND, DIM, M, 16 - M - RC, RC, 5>(P, n_work, s);
    }
    if constexpr (M == 3) {
        return hipErrorInvalidValue;
    } else if constexpr (M == 20) {
        if (nn <= 20) return launch_nse_one<KIND, DIM, M, 20, RC, 2>(P, n_work, s);
        if (nn <= 26) return launch_nse_one<KIND, DIM, M, 26, RC, RC <= 1 ? 2 : 1>(P, n_work, s);
    } else {
        if (nn <= 16 - RC) return launch_nse_one<KIND, DIM, M, 16 - RC, RC, M <= 6 ? 4 : 3>(P, n_work, s);
        if constexpr (M > 4) {
            if (nn <= 26) return launch_nse_one<KIND, DIM, M, 26, RC, 2>(P, n_work, s);
        }
    }
    return hipErrorInvalidValue;
}

template <int KIND, int DIM, int M>
inline hipError_t launch_nse_rc(const BuildDev& P, int64_t n_work, hipStream_t s)
{
    if (P.n_cols == 1) return launch_nse_m<KIND, DIM, M, 1>(P, n_work, s);
    if constexpr (DIM == 2) {
        if (P.n_cols == 2) return launch_nse_m<KIND, DIM, M, 2>(P, n_work, s);
        if (P.n_cols == 3) return launch_nse_m<KIND, DIM, M, 3>(P, n_work, s);
    } else {
        if (P.n_cols <= 3) return launch_nse_m<KIND, DIM, M, 3>(P, n_work, s);
        if (P.n_cols == 4) return launch_nse_m<KIND, DIM, M, 4>(P, n_work, s);
        if (P.n_cols <= 6) return launch_nse_m<KIND, DIM, M, 6>(P, n_work, s);
    }
    return hipErrorInvalidValue;
}

// Ragged launches: the classes of one slot and of two (nse_classes).
template <int KIND, int DIM, int M, int RC>
inline hipError_t launch_nse_class_m(const BuildDev& P, int hi, int64_t n_work, hipStream_t s)
{
    if constexpr (M == 20) {
        if (hi <= 20) return launch_nse_one<KIND, DIM, M, 20, RC, 2, true>(P, n_work, s);
        return launch_nse_one<KIND, DIM, M, 26, RC, RC <= 1 ? 2 : 1, true>(P, n_work, s);
    } else {
        if (hi <= 16 - RC) return launch_nse_one<KIND, DIM, M, 16 - RC, RC, M <= 6 ? 4 : 3, true>(P, n_work, s);
        if constexpr (DIM == 2)
            if (hi > 26) return launch_nse_one<KIND, DIM, M, 32 - RC, RC, 2, true>(P, n_work, s);
        return launch_nse_one<KIND, DIM, M, 26, RC, 2, true>(P, n_work, s);
    }
}

template <int KIND, int DIM, int M>
inline hipError_t launch_nse_class_rc(const BuildDev& P, int hi, int64_t n_work, hipStream_t s)
{
    if (P.n_cols == 1) return launch_nse_class_m<KIND, DIM, M, 1>(P, hi, n_work, s);
    if constexpr (DIM == 2) {
        if (P.n_cols == 2) return launch_nse_class_m<KIND, DIM, M, 2>(P, hi, n_work, s);
        if (P.n_cols == 3) return launch_nse_class_m<KIND, DIM, M, 3>(P, hi, n_work, s);
    } else {
        if (P.n_cols <= 3) return launch_nse_class_m<KIND, DIM, M, 3>(P, hi, n_work, s);
        if (P.n_cols == 4) return launch_nse_class_m<KIND, DIM, M, 4>(P, hi, n_work, s);
        if (P.n_cols <= 6) return launch_nse_class_m<KIND, DIM, M, 6>(P, hi, n_work, s);
    }
    return hipErrorInvalidValue;
}

}  // namespace rbfx
