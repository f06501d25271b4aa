// Fused build for stencil systems of 65..RBFX_MAX_N rows (k up to 60 with a degree-3
// polynomial gives 70): one wavefront per stencil, the augmented system [A | b] in LDS
// (row-major: the n columns, padding to a multiple of eight, then the RC right-hand sides;
// odd leading dimension). Lane li owns row m0 + li, and for systems of more than 64 rows
// (m0 = n - 64 > 0) also row li < m0: the second rows are the first ones, the polynomial
// rows, which the pivot order freezes within the first few steps, so the second pass of
// the trailing update is skipped for the rest of the factorisation.
//
// The arithmetic is that of k_build (build_kernel.h): centred, radius-scaled
// saddle-point system assembled in FP64, rook-pivoted LDL^T (pivot tests of Ashcraft,
// Grimes & Lewis) with rows that never move, the trailing update applied to the
// still-active rows, and a back substitution over the rows frozen at their pivot step.
// Only the storage differs: the rows live in LDS instead of registers, so a pivot-row
// read is an LDS load and the pivot search reads the column entries of the lane's own
// rows. The active columns are kept in a prefix of every row, and the trailing update
// runs over that prefix eight columns per LDS round trip.
#include "build_kernel.h"

namespace rbfx {

static_assert(RBFX_MAX_N <= 128, "at most two rows per lane");

// maximum over the 64 lanes, as a scalar: rotations within each row of 16 lanes, then the
// four row maxima read from lanes 0, 16, 32 and 48 (no LDS permute)
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t k)
{
    k = max(k, (uint32_t)dpp_i<0x121>((int)k));
    k = max(k, (uint32_t)dpp_i<0x122>((int)k));
    k = max(k, (uint32_t)dpp_i<0x124>((int)k));
    k = max(k, (uint32_t)dpp_i<0x128>((int)k));
    const uint32_t a = (uint32_t)__builtin_amdgcn_readlane((int)k, 0), b = (uint32_t)__builtin_amdgcn_readlane((int)k, 16);
    const uint32_t c = (uint32_t)__builtin_amdgcn_readlane((int)k, 32), d = (uint32_t)__builtin_amdgcn_readlane((int)k, 48);
    return max(max(a, b), max(c, d));
}

__device__ __forceinline__ uint32_t row_key(double v, int row)
{
    const uint32_t hi = (uint32_t)((unsigned long long)__double_as_longlong(v) >> 32);
    return (hi & ~127u) | (uint32_t)(127 - row);
}

// TWO: rows per lane (1 for systems of up to 64 rows, 2 up to 128)
template <int DIM, int RC, int TWO>
__global__ __attribute__((amdgpu_flat_work_group_size(64, 64))) void k_build_wide(const BuildDev P, int rows_cap,
                                                                                  int lda)
{
    constexpr int ROWS = 64 * TWO;
    // the system (rows_cap x lda), then the point tables of the assembly, sized by rows_cap
    // so that small systems leave LDS for more wavefronts per CU: the scaled points, and
    // for builds with boundary data the normals, boundary coefficients and types
    extern __shared__ __attribute__((aligned(16))) double s_A[];
    double(*s_xi)[DIM] = reinterpret_cast<double(*)[DIM]>(s_A + (int64_t)rows_cap * lda);
    double(*s_bn)[DIM] = s_xi + rows_cap;
    double* s_ba = reinterpret_cast<double*>(s_bn + rows_cap);
    double* s_bb = s_ba + rows_cap;
    int* s_bt = reinterpret_cast<int*>(s_bb + rows_cap);
    const bool bnd_tables = P.is_boundary != nullptr;
    __shared__ int s_piv[ROWS], s_blk[ROWS];
    __shared__ int s_mono[kMaxMono][3];
    __shared__ TermDev s_terms[RBFX_MAX_TERMS];

    const int L = threadIdx.x;
    const int n_cols = P.n_cols, n_terms = P.n_terms;
    for (int i = L; i < kMaxMono * 3; i += 64) (&s_mono[0][0])[i] = (&P.mono_e[0][0])[i];
    if (L < RBFX_MAX_TERMS) s_terms[L] = P.terms[L];

    // one stencil per workgroup: every exit below is uniform over the workgroup
    const int64_t lb = xcd_contiguous_block(P.n_blocks);
    if (lb < 0) return;
    const int64_t n_work = P.list ? (int64_t)*P.list_len : P.n_eval;
    if (lb >= n_work) return;
    const int64_t e = P.list ? (int64_t)P.list[lb] : (P.order ? (int64_t)P.order[lb] : lb);
    if (e < 0 || e >= P.n_eval) return;
    const int64_t s0 = P.adj_ptr ? P.adj_ptr[e] : e * (int64_t)P.k;
    const int kk = P.adj_ptr ? (int)(P.adj_ptr[e + 1] - s0) : P.k;
    const int64_t o0 = P.out_ptr ? P.out_ptr[e] : e * (int64_t)P.k;
    const int M = stencil_n_mono(P, e, DIM);
    if (M < 0) {
        if (L == 0 && P.status) P.status[e] = RBFX_ST_INVALID;
        return;
    }
    if (kk < 1 || M + kk > rows_cap) {
        if (L == 0 && P.status) P.status[e] = RBFX_ST_TOO_LARGE;
        return;
    }
    const int n = M + kk;
    const int rhs0 = (n + 7) & ~7;  // position of the first right-hand side in a row
    // row ownership: slot 0 of lane L holds row m0 + L, slot 1 (TWO == 2) row L < m0
    const int m0 = TWO == 2 ? max(n - 64, 0) : 0;
    auto rowof = [&](int t) -> int { return (TWO == 2 && t == 1) ? L : L + m0; };
    auto owns = [&](int t) -> bool { return (TWO == 2 && t == 1) ? L < m0 : L + m0 < n; };
    // the owner of row r (uniform): its lane and slot
    auto lane_of = [&](int r) -> int { return r < m0 ? r : r - m0; };
    auto slot_t = [&](int r) -> int { return (TWO == 2 && r < m0) ? 1 : 0; };

    // ---- the stencil points this lane loads: q = L (and q = L + 64)
    double xe[DIM];
#pragma unroll
    for (int d = 0; d < DIM; ++d) xe[d] = P.eval[e * DIM + d];
    int gidx[TWO] = {};
    double D[TWO][DIM];
    double r2max = 0.0;
    bool ib[TWO] = {};
#pragma unroll
    for (int t = 0; t < TWO; ++t) {
        const int q = L + 64 * t;
#pragma unroll
        for (int d = 0; d < DIM; ++d) D[t][d] = 0.0;
        if (q < kk) {
            gidx[t] = P.adj_idx[s0 + q];
            double r2 = 0.0;
#pragma unroll
            for (int d = 0; d < DIM; ++d) {
                D[t][d] = P.data[(int64_t)gidx[t] * DIM + d] - xe[d];
                r2 += D[t][d] * D[t][d];
            }
            r2max = fmax(r2max, r2);
            ib[t] = P.is_boundary && P.is_boundary[gidx[t]];
        }
    }
    // stencil classification (types.jl:208-223)
    const bool hermite = P.is_boundary && (__ballot(ib[0] || ib[TWO - 1]) != 0ull);
    // a Dirichlet eval node is an identity row whatever its neighbours are (the row
    // length count_nonzeros gives it, execution.jl:39-69)
    if (P.is_boundary && e < P.n_data && P.is_boundary[e]) {
        const int bi = P.bnd_index[e];
        if (P.bc_alpha[bi] == 1.0 && P.bc_beta[bi] == 0.0) {
            // identity row (fill_dirichlet_entry!, execution.jl:297-303)
            if (L < n_cols) P.out_val[(int64_t)L * P.out_nnz + o0] = 1.0;
            if (L == 0) {
                if (P.out_col) P.out_col[o0] = (int32_t)e;
                if (P.status) P.status[e] = RBFX_ST_DIRICHLET;
            }
            return;
        }
    }
    double h = sqrt(group_max<64>(r2max));
    if (!(h > 0.0)) h = 1.0;
    const double hinv = 1.0 / h;
    unsigned long long at_eval[TWO];
#pragma unroll
    for (int t = 0; t < TWO; ++t) {
        const int q = L + 64 * t;
        bool eq = false;
        if (q < kk) {
            int bt = 0;
            double ba = 0.0, bb = 0.0;
            if (hermite && ib[t]) {
                const int bi = P.bnd_index[gidx[t]];
                ba = P.bc_alpha[bi];
                bb = P.bc_beta[bi];
#pragma unroll
                for (int d = 0; d < DIM; ++d) s_bn[q][d] = P.normals[(int64_t)bi * DIM + d];
                bt = (ba == 1.0 && bb == 0.0) ? 1 : 2;
            }
            eq = hermite;
#pragma unroll
            for (int d = 0; d < DIM; ++d) {
                s_xi[q][d] = D[t][d] / h;
                eq = eq && (D[t][d] == 0.0);
            }
            if (bnd_tables) {
                s_bt[q] = bt;
                s_ba[q] = ba;
                s_bb[q] = bb / h;  // beta acts through a first derivative
            }
        }
        at_eval[t] = __ballot(eq);
    }
    int eval_local = 0;
    if (hermite) {
        const unsigned long long ae1 = TWO == 2 ? at_eval[TWO - 1] : 0ull;
        if (!at_eval[0] && !ae1) {
            if (L == 0 && P.status) P.status[e] = RBFX_ST_EVAL_NOT_FOUND;
            return;
        }
        eval_local = at_eval[0] ? __builtin_ctzll(at_eval[0]) : 64 + __builtin_ctzll(ae1);
    }
    __syncthreads();

    BasisDev B;
    B.kind = P.basis_kind;
    B.eps = (B.kind == RBFX_IMQ || B.kind == RBFX_GAUSSIAN) ? P.eps * h : P.eps;

    // ---- assembly (FP64): the lane's rows; columns 0..n-1, then the RHS at rhs0..rhs0+RC-1
#pragma unroll
    for (int t = 0; t < TWO; ++t) {
        const int i = rowof(t);
        if (!owns(t)) continue;
        double* Ai = s_A + (int64_t)i * lda;
        const bool is_poly = i < M;
        const int pi = i - M;
        double xi[DIM], bn[DIM];
        int bt = 0;
        double ba = 0.0, bb = 0.0;
        if (!is_poly) {
#pragma unroll
            for (int d = 0; d < DIM; ++d) {
                xi[d] = s_xi[pi][d];
                bn[d] = hermite ? s_bn[pi][d] : 0.0;
            }
            if (hermite) {
                bt = s_bt[pi];
                ba = s_ba[pi];
                bb = s_bb[pi];
            }
        }
        // columns 0..M-1. A point row holds its monomials; the polynomial rows' entries at
        // the point columns are the same numbers (symmetry of the saddle-point matrix), so
        // each point lane also writes its value into column i of polynomial row a, and the
        // polynomial lanes only zero their corner block.
        for (int a = 0; a < M; ++a) {
            if (is_poly) {
                Ai[a] = 0.0;
            } else {
                double v = mono_op<DIM>(s_mono[a], RBFX_OP_VALUE, 0, 0, xi);
                if (hermite && bt == 2) v = ba * v + bb * mono_normal<DIM>(s_mono[a], bn, xi);
                Ai[a] = v;
                s_A[(int64_t)a * lda + i] = v;
            }
        }
        // columns M..n-1 of the point rows: phi between the points (instantiated once per
        // basis kind; without boundary data four independent entries per iteration)
        auto point_cols = [&](auto KC) __attribute__((always_inline)) {
            if (is_poly) return;
            if (!hermite) {
#pragma unroll 4
                for (int jj = 0; jj < kk; ++jj) {
                    double q2 = 0.0;
#pragma unroll
                    for (int d = 0; d < DIM; ++d) {
                        const double t_ = xi[d] - s_xi[jj][d];
                        q2 += t_ * t_;
                    }
                    Ai[M + jj] = phi_r2_k<decltype(KC)::value>(B.eps, q2);
                }
                return;
            }
            for (int jj = 0; jj < kk; ++jj) {
                double xj[DIM];
#pragma unroll
                for (int d = 0; d < DIM; ++d) xj[d] = s_xi[jj][d];
                const int tj = s_bt[jj];
                double Dj[DIM], q2 = 0.0;
#pragma unroll
                for (int d = 0; d < DIM; ++d) {
                    Dj[d] = xi[d] - xj[d];
                    q2 += Dj[d] * Dj[d];
                }
                double v = phi_r2_k<decltype(KC)::value>(B.eps, q2);
                if (bt == 2 || tj == 2) {
                    double nj[DIM];
#pragma unroll
                    for (int d = 0; d < DIM; ++d) nj[d] = s_bn[jj][d];
                    double Di, Djn, D2;
                    phi_grad_hess_dirs<DIM>(B, Dj, q2, bn, nj, Di, Djn, D2);
                    const double aj = s_ba[jj], bj = s_bb[jj];
                    if (bt != 2) v = aj * v - bj * Djn;
                    else if (tj != 2) v = ba * v + bb * Di;
                    else v = ba * aj * v - ba * bj * Djn + bb * aj * Di + bb * bj * D2;
                }
                Ai[M + jj] = v;
            }
        };
        switch (B.kind) {
        case RBFX_PHS1: point_cols(std::integral_constant<int, RBFX_PHS1>{}); break;
        case RBFX_PHS3: point_cols(std::integral_constant<int, RBFX_PHS3>{}); break;
        case RBFX_PHS5: point_cols(std::integral_constant<int, RBFX_PHS5>{}); break;
        case RBFX_PHS7: point_cols(std::integral_constant<int, RBFX_PHS7>{}); break;
        case RBFX_IMQ: point_cols(std::integral_constant<int, RBFX_IMQ>{}); break;
        default: point_cols(std::integral_constant<int, RBFX_GAUSSIAN>{}); break;
        }
        // right-hand sides
        double bcol[RC];
#pragma unroll
        for (int c = 0; c < RC; ++c) bcol[c] = 0.0;
        if (!is_poly) {
            double De[DIM], q2 = 0.0;
#pragma unroll
            for (int d = 0; d < DIM; ++d) {
                De[d] = -xi[d];
                q2 += De[d] * De[d];
            }
            for (int tt = 0; tt < n_terms; ++tt) {
                const TermDev tm = s_terms[tt];
                double v = phi_term<DIM>(B, tm.kind, tm.d1, tm.d2, De, q2);
                if (hermite && bt == 2) v = ba * v + bb * phi_term_normal<DIM>(B, tm.kind, tm.d1, De, q2, bn);
                const double sc = term_scale(tm, hinv);
#pragma unroll
                for (int c = 0; c < RC; ++c)
                    if (tm.col == c) bcol[c] += sc * v;
            }
        } else {
            double z[DIM];
#pragma unroll
            for (int d = 0; d < DIM; ++d) z[d] = 0.0;
            const int(&ea)[3] = s_mono[i];
            if (hermite && s_bt[eval_local] == 2) {
                // the eval node's boundary operator applied to P (assembly.jl:452-467)
                const double eav = s_ba[eval_local], ebv = s_bb[eval_local];
                double en[DIM];
#pragma unroll
                for (int d = 0; d < DIM; ++d) en[d] = s_bn[eval_local][d];
                const double v = eav * mono_op<DIM>(ea, RBFX_OP_VALUE, 0, 0, z) + ebv * mono_normal<DIM>(ea, en, z);
#pragma unroll
                for (int c = 0; c < RC; ++c) bcol[c] = v;
            } else {
                for (int tt = 0; tt < n_terms; ++tt) {
                    const TermDev tm = s_terms[tt];
                    const double v = term_scale(tm, hinv) * mono_op<DIM>(ea, tm.kind, tm.d1, tm.d2, z);
#pragma unroll
                    for (int c = 0; c < RC; ++c)
                        if (tm.col == c) bcol[c] += v;
                }
            }
        }
#pragma unroll
        for (int c = 0; c < RC; ++c) Ai[rhs0 + c] = bcol[c];
    }
    __syncthreads();

    // ---- factorisation with rook pivoting; rows never move, pivoted rows freeze
    const double alpha = 0.6403882032022076;  // (1 + sqrt(17)) / 8
    bool act[TWO];
    int myslot[TWO];
#pragma unroll
    for (int t = 0; t < TWO; ++t) {
        act[t] = owns(t);
        myslot[t] = 1 << 20;
    }
    int slot = 0;
    bool failed = false;
    auto A = [&](int i, int j) -> double { return s_A[(int64_t)i * lda + j]; };
    // Column c of the active rows goes to this lane's registers (v[t] = A(rowof(t), c)),
    // and the largest |A(r, c)| over the active rows r != excl comes back as a packed
    // (magnitude, row) key. The pivot tests then take single entries of that column from
    // their owning lanes (colval) instead of another LDS round trip.
    //
    // Column positions: the columns of the active rows sit in positions 0..n_act-1 of
    // every row (the right-hand sides at rhs0.., past the padding). Freezing a pivot swaps
    // its column with the last active position in every row, frozen rows included, so
    // the trailing update only touches the active prefix, and an entry (r, c) is always
    // at position pos(c) of row r. pos[t] is the position of column rowof(t).
    int pos[TWO];
#pragma unroll
    for (int t = 0; t < TWO; ++t) pos[t] = owns(t) ? rowof(t) : 1 << 20;
    int n_act = n;
    auto posof = [&](int c) -> int {
        const int cc = __builtin_amdgcn_readfirstlane(c);
        return slot_t(cc) ? rdlane(pos[TWO - 1], lane_of(cc)) : rdlane(pos[0], lane_of(cc));
    };
    double v[TWO];
    auto colkey = [&](int c, int excl) -> uint32_t {
        uint32_t k = 0u;
        const int pc = posof(c);
#pragma unroll
        for (int t = 0; t < TWO; ++t) {
            const int r = rowof(t);
            v[t] = act[t] ? A(r, pc) : 0.0;
            if (act[t] && r != excl) k = max(k, row_key(fabs(v[t]), r));
        }
        return wave_max_u32(k);
    };
    auto colval = [&](int r) -> double {
        const int rr = __builtin_amdgcn_readfirstlane(r);
        return slot_t(rr) ? rdlane(v[TWO - 1], lane_of(rr)) : rdlane(v[0], lane_of(rr));
    };
    for (;;) {
        const unsigned long long b0 = __ballot(act[0]), b1 = TWO == 2 ? __ballot(act[TWO - 1]) : 0ull;
        if (!b0 && !b1) break;
        // the lowest active row: slot 1 holds rows 0..m0-1, slot 0 rows m0..n-1
        const int c0 = b1 ? (int)__builtin_ctzll(b1) : m0 + (int)__builtin_ctzll(b0);
        // column c0 = row c0 by symmetry of the active block
        const uint32_t ck = colkey(c0, c0);
        int imax = ck ? 127 - (int)(ck & 127u) : c0;
        const double akk = colval(c0);
        double colmax = ck ? fabs(colval(imax)) : 0.0;
        const double absakk = fabs(akk);
        int kstep = 1, p = c0, kp = c0;
        // A(p, p), A(kp, kp) and, for a 2x2 pivot, A(p, kp) as the search ends
        double app = akk, akp = akk, apk = akk;
        bool need_rook = absakk < alpha * colmax;
        if (!(absakk > 0.0 || colmax > 0.0)) {
            failed = true;  // zero column: singular
            break;
        }
        for (int it = 0; it < 2 * ROWS && need_rook; ++it) {
            const uint32_t rk = colkey(imax, imax);
            const int ri = rk ? 127 - (int)(rk & 127u) : imax;
            const double rowmax = rk ? fabs(colval(ri)) : 0.0;
            const double aim = colval(imax);
            const double aii = fabs(aim);
            if (!(aii < alpha * rowmax)) {
                kp = imax;
                akp = aim;
                need_rook = false;
            } else if (p == ri || rowmax <= colmax || it == 2 * ROWS - 1) {
                kp = imax;
                kstep = 2;
                akp = aim;
                apk = colval(p);  // column imax holds A(p, imax)
                need_rook = false;
            } else {
                p = imax;
                app = aim;
                colmax = rowmax;
                imax = ri;
            }
        }
        // (the same on every lane; read from lane 0 so the compiler keeps the pivot
        // bookkeeping and the column masks below in scalar registers)
        kstep = __builtin_amdgcn_readfirstlane(kstep);
        const int p0 = __builtin_amdgcn_readfirstlane((kstep == 1) ? kp : p);
        const int p1 = __builtin_amdgcn_readfirstlane(kp);  // equals p0 for a 1x1 pivot
        // A(p0, p0), A(p1, p1), A(p0, p1)
        const double d0 = kstep == 1 ? akp : app, d1 = akp, bq = kstep == 1 ? akp : apk;
        const double det = d0 * d1 - bq * bq;
        if ((kstep == 1 && d0 == 0.0) || (kstep == 2 && det == 0.0)) {
            failed = true;
            break;
        }
        const double idet = 1.0 / det;
        if (L == 0) {
            s_piv[slot] = p0;
            s_blk[slot] = kstep;
            if (kstep == 2) {
                s_piv[slot + 1] = p1;
                s_blk[slot + 1] = 0;
            }
        }
        // freeze: the pivot columns move to the end of the active prefix in every row
        auto swap_to = [&](int c, int last) {
            const int pc = posof(c);
            if (pc == last) return;
#pragma unroll
            for (int t = 0; t < TWO; ++t) {
                if (!owns(t)) continue;
                const int r = rowof(t);
                double* Ar = s_A + (int64_t)r * lda;
                const double x0 = Ar[pc], x1 = Ar[last];
                Ar[pc] = x1;
                Ar[last] = x0;
                if (pos[t] == last) pos[t] = pc;
                else if (r == c) pos[t] = last;
            }
        };
        swap_to(p0, n_act - 1);
        if (kstep == 2) swap_to(p1, n_act - 2);
        n_act -= kstep;
        const double* U0 = s_A + (int64_t)p0 * lda;
        const double* U1 = s_A + (int64_t)p1 * lda;
        // The active prefix (rounded up to eight: the padding before rhs0 and the frozen
        // columns past the prefix are never read) and the right-hand sides are updated
        // eight columns at a time: uniform column offsets become immediate offsets of
        // paired LDS loads, all loads of a chunk are issued before its stores, and per
        // element the FMAs run in the same order as a column-by-column update.
        const int na8 = (n_act + 7) & ~7;
#pragma unroll
        for (int t = 0; t < TWO; ++t) {
            const int r = rowof(t);
            if (!act[t] || r == p0 || r == p1) continue;
            const double u0 = U0[pos[t]];
            double l0, l1 = 0.0;
            if (kstep == 1) {
                l0 = u0 / d0;
            } else {
                const double u1 = U1[pos[t]];
                l0 = (u0 * d1 - u1 * bq) * idet;
                l1 = (u1 * d0 - u0 * bq) * idet;
            }
            const double ml0 = -l0, ml1 = -l1;
            double* Ar = s_A + (int64_t)r * lda;
            // a 1x1 and a 2x2 pivot each have their own loop, so a chunk's loads stay together
            auto chunk1 = [&](auto W, int j0) __attribute__((always_inline)) {
                constexpr int CW = decltype(W)::value;
                double a[CW], w0[CW];
#pragma unroll
                for (int q = 0; q < CW; ++q) {
                    a[q] = Ar[j0 + q];
                    w0[q] = U0[j0 + q];
                }
#pragma unroll
                for (int q = 0; q < CW; ++q) Ar[j0 + q] = fma(ml0, w0[q], a[q]);
            };
            auto chunk2 = [&](auto W, int j0) __attribute__((always_inline)) {
                constexpr int CW = decltype(W)::value;
                double a[CW], w0[CW], w1[CW];
#pragma unroll
                for (int q = 0; q < CW; ++q) {
                    a[q] = Ar[j0 + q];
                    w0[q] = U0[j0 + q];
                    w1[q] = U1[j0 + q];
                }
#pragma unroll
                for (int q = 0; q < CW; ++q) Ar[j0 + q] = fma(ml1, w1[q], fma(ml0, w0[q], a[q]));
            };
            using C8 = std::integral_constant<int, 8>;
            using CR = std::integral_constant<int, RC>;
            if (kstep == 1) {
                for (int j0 = 0; j0 < na8; j0 += 8) chunk1(C8{}, j0);
                chunk1(CR{}, rhs0);
            } else {
                for (int j0 = 0; j0 < na8; j0 += 8) chunk2(C8{}, j0);
                chunk2(CR{}, rhs0);
            }
        }
#pragma unroll
        for (int t = 0; t < TWO; ++t) {
            const int r = rowof(t);
            if (act[t] && r == p0) {
                act[t] = false;
                myslot[t] = slot;
            }
            if (act[t] && kstep == 2 && r == p1) {
                act[t] = false;
                myslot[t] = slot + 1;
            }
        }
        slot += kstep;
        __syncthreads();
    }
    __syncthreads();

    // ---- back substitution over the frozen rows, last pivot first
    double x[TWO][RC], acc[TWO][RC];
#pragma unroll
    for (int t = 0; t < TWO; ++t)
#pragma unroll
        for (int c = 0; c < RC; ++c) {
            x[t][c] = 0.0;
            acc[t][c] = 0.0;
        }
    if (!failed) {
        const int nslots = slot;
        // the right-hand sides (final once every row has frozen) and the pivot list go to
        // registers: each slot then costs one round of LDS loads (the pivot block and the
        // lane's entries in the pivot columns), issued together
        double y[TWO][RC];
        int pv[TWO], bk[TWO];
#pragma unroll
        for (int t = 0; t < TWO; ++t) {
#pragma unroll
            for (int c = 0; c < RC; ++c) y[t][c] = owns(t) ? A(rowof(t), rhs0 + c) : 0.0;
            // slot sl of the pivot list sits in lane sl % 64, register sl / 64
            const int sl = L + 64 * t;
            pv[t] = sl < nslots ? s_piv[sl] : 0;
            bk[t] = sl < nslots ? s_blk[sl] : -1;
        }
        auto slot_of = [&](const int(&v)[TWO], int sl) -> int {
            return (TWO == 2 && sl >= 64) ? rdlane(v[TWO - 1], sl & 63) : rdlane(v[0], sl & 63);
        };
        for (int s = nslots - 1; s >= 0; --s) {
            const int blk = slot_of(bk, s);
            const int bprev = s > 0 ? slot_of(bk, s - 1) : -1;
            const bool one = blk == 1, two = (blk == 0) && (bprev == 2);
            if (!one && !two) continue;  // first slot of a 2x2 block: solved with the second
            const int p = slot_of(pv, one ? s : s - 1);
            const int q = two ? slot_of(pv, s) : p;
            const int pl = lane_of(p), pt = slot_t(p), ql = lane_of(q), qt = slot_t(q);
            const int pp = posof(p), pq = posof(q);
            const double dp = A(p, pp), dq = A(q, pq), bq = A(p, pq);
            double arp[TWO], arq[TWO];
#pragma unroll
            for (int t = 0; t < TWO; ++t) {
                const int r = rowof(t);
                arp[t] = owns(t) ? A(r, pp) : 0.0;
                arq[t] = (two && owns(t)) ? A(r, pq) : 0.0;
            }
            // (one division per pivot: a 1x1 pivot needs only 1/dp, a 2x2 only 1/det)
            double idet = 0.0, dinv = 0.0;
            if (two) idet = 1.0 / (dp * dq - bq * bq);
            else dinv = 1.0 / dp;
#pragma unroll
            for (int c = 0; c < RC; ++c) {
                if (c >= n_cols) continue;
                // y - acc of rows p and q, from their owning lanes
                const double rp0 = y[0][c] - acc[0][c];
                const double rp1 = TWO == 2 ? y[TWO - 1][c] - acc[TWO - 1][c] : 0.0;
                const double yp = pt ? rdlane(rp1, pl) : rdlane(rp0, pl);
                const double yq = qt ? rdlane(rp1, ql) : rdlane(rp0, ql);
                const double x0 = two ? (yp * dq - yq * bq) * idet : yp * dinv;
                const double x1 = two ? (yq * dp - yp * bq) * idet : 0.0;
#pragma unroll
                for (int t = 0; t < TWO; ++t) {
                    const int r = rowof(t);
                    if (!owns(t)) continue;
                    if (r == p) x[t][c] = x0;
                    if (two && r == q) x[t][c] = x1;
                    const bool upd = one ? (myslot[t] < s) : (myslot[t] < s - 1);
                    if (upd) acc[t][c] += two ? arp[t] * x0 + arq[t] * x1 : arp[t] * x0;
                }
            }
        }
    }

    // ---- outputs: weights of the point rows, multipliers of the polynomial rows
#pragma unroll
    for (int t = 0; t < TWO; ++t) {
        const int i = rowof(t);
        if (!owns(t)) continue;
#pragma unroll
        for (int c = 0; c < RC; ++c) {
            if (c >= n_cols) continue;
            const double v = failed ? __builtin_nan("") : x[t][c];
            if (i >= M) P.out_val[(int64_t)c * P.out_nnz + o0 + (i - M)] = v;
            else if (P.out_lambda) P.out_lambda[((int64_t)c * P.n_eval + e) * P.n_mono + i] = v;
        }
        // row i holds stencil point i - M
        if (i >= M && P.out_col) P.out_col[o0 + (i - M)] = P.adj_idx[s0 + (i - M)];
    }
    if (L == 0 && P.status) P.status[e] = failed ? RBFX_ST_SINGULAR : P.ok_status;
}

// ---------------------------------------------------------------- packed symmetric variant
//
// k_build_sym: the same build with half the LDS, for more wavefronts per CU. The
// saddle-point matrix is symmetric, and so is every trailing block of its elimination,
// so only the lower triangle is kept, by position: lane li owns position li (and
// li + 64), row j holding its entries at positions 0..j. Pivoting is a symmetric
// permutation: the pivot row and column move together to the end of the active prefix
// (rows and columns of two positions swap), so the active block is always positions
// 0..n_act-1, its pivot rows are the frozen rows just past it (contiguous, read as
// broadcasts by the update), and a frozen row keeps its entries at the positions of
// the rows frozen after it, which the back substitution reads. The original row index
// travels with each row (the pivot search starts from the active row of the lowest
// original index, as in k_build_wide; ties in the search go to the lower position).
// The stencil points take positions 0..k-1 and the monomials k..k+m-1, so for systems
// of more than 64 rows the second lane slot holds monomial rows, whose assembly is a
// zero fill, and which the first steps freeze (every step freezes the top active
// positions): the second update pass is skipped from then on.
//
// Bound by VALU issue (88% of the cycles on the 8M-stencil 3-D regrid of 34 rows, 4,937
// instructions a stencil), so everything is arranged to take fewer of them, each entry's
// arithmetic unchanged (the weights are the same bits):
//   - without boundary points each pair of points is evaluated once (8 evaluations a lane
//     for 30 points, not 30), and the basis kind is a constant around both loops;
//   - the update reads eight entries of the pivot row at once, one per lane, and the FMAs
//     broadcast them (DPP), where eight LDS broadcasts had taken a third of the LDS cycles;
//   - up to 32 active rows both halves of the wavefront share the rows;
//   - uniform work (the search's masks and maxima, where a row starts, 2x2 flags) is scalar;
//   - the back substitution takes the reciprocals of all diagonal entries in one division;
//   - systems of more than 64 rows leave the two-slot loop at 64 (51,000 of 65..70 rows: 4.55
//     -> 3.94 ms).
// 147.5 -> 83.5 ms there; 290,000 stencils of 33..70 rows of a disk with boundary points
// 18.9 -> 14.2 ms. LDS is allocated in steps of 1,280 bytes: 6,344 bytes (34 rows) hold 25
// wavefronts on a CU, 6,408 had held 21 (91.6 ms).
//
// Row starts: row j holds positions 0..j padded to a multiple of eight (the update's
// eight-column chunks stay inside the row), plus the fewest entries (0..31) that put the
// starts of each 16 consecutive rows in 16 different 8-byte bank pairs modulo 16 and of
// each 32 consecutive rows in 32 different ones modulo 32: a column read by the lanes of
// a wavefront is then free of bank conflicts whether the LDS serves 16 or 32 lanes of
// 8-byte reads per cycle.
constexpr int kSymRows = 128;
struct SymRowStarts {
    int rb[kSymRows + 1];
};
constexpr SymRowStarts make_sym_row_starts()
{
    SymRowStarts s{};
    bool u32[kSymRows / 32 + 1][32] = {};
    bool u16[kSymRows / 16 + 1][16] = {};
    s.rb[0] = 0;
    u32[0][0] = true;
    u16[0][0] = true;
    for (int j = 1; j <= kSymRows; ++j) {
        const int base = s.rb[j - 1] + ((j + 7) & ~7);  // row j - 1 holds j entries
        int p = 0;
        while (p < 31 && (u32[j / 32][(base + p) & 31] || u16[j / 16][(base + p) & 15])) ++p;
        s.rb[j] = base + p;
        u32[j / 32][(base + p) & 31] = true;
        u16[j / 16][(base + p) & 15] = true;
    }
    return s;
}
__constant__ SymRowStarts kSymRb = make_sym_row_starts();
constexpr SymRowStarts kSymRbHost = make_sym_row_starts();
static_assert(RBFX_MAX_N <= kSymRows, "positions fit the row-start table");
constexpr bool sym_rows_spread()
{
    for (int g = 0; g < kSymRows; g += 16) {
        bool seen[16] = {};
        for (int j = g; j < g + 16; ++j) {
            if (seen[kSymRbHost.rb[j] & 15]) return false;
            seen[kSymRbHost.rb[j] & 15] = true;
        }
    }
    for (int g = 0; g < kSymRows; g += 32) {
        bool seen[32] = {};
        for (int j = g; j < g + 32; ++j) {
            if (seen[kSymRbHost.rb[j] & 31]) return false;
            seen[kSymRbHost.rb[j] & 31] = true;
        }
    }
    return true;
}
static_assert(sym_rows_spread(), "row starts spread over the LDS banks");

// v where the lane's bit of a (uniform) mask is set, else 0
__device__ __forceinline__ uint32_t lanes_in(unsigned long long mask, uint32_t v)
{
    uint32_t r;
    asm("v_cndmask_b32_e64 %0, 0, %1, %2" : "=v"(r) : "v"(v), "s"(mask));
    return r;
}

// max on the scalar unit (the compiler takes max3 of the vector one for three operands)
__device__ __forceinline__ uint32_t smax_u32(uint32_t a, uint32_t b)
{
    uint32_t r;
    asm("s_max_u32 %0, %1, %2" : "=s"(r) : "s"(a), "s"(b) : "scc");
    return r;
}

// the largest key of the first `lanes` lanes (uniform; the others hold 0)
__device__ __forceinline__ uint32_t first_max_u32(uint32_t k, int lanes)
{
    k = max(k, (uint32_t)dpp_i<0x121>((int)k));
    k = max(k, (uint32_t)dpp_i<0x122>((int)k));
    k = max(k, (uint32_t)dpp_i<0x124>((int)k));
    k = max(k, (uint32_t)dpp_i<0x128>((int)k));
    uint32_t m = smax_u32((uint32_t)rdlane((int)k, 0), (uint32_t)rdlane((int)k, 16));
    if (lanes > 32) m = smax_u32(m, smax_u32((uint32_t)rdlane((int)k, 32), (uint32_t)rdlane((int)k, 48)));
    return m;
}

// lane l (uniform) of v set to x (uniform)
__device__ __forceinline__ int wrlane(int v, int x, int l)
{
    asm("s_mov_b32 m0, %2\n\tv_writelane_b32 %0, %1, m0" : "+v"(v) : "s"(x), "s"(l) : "m0");
    return v;
}
__device__ __forceinline__ double wrlane(double v, double x, int l)
{
    const unsigned long long u = (unsigned long long)__double_as_longlong(v);
    const unsigned long long w = (unsigned long long)__double_as_longlong(x);
    const unsigned lo = (unsigned)wrlane((int)(unsigned)u, (int)(unsigned)w, l);
    const unsigned hi = (unsigned)wrlane((int)(unsigned)(u >> 32), (int)(unsigned)(w >> 32), l);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// a[q] += m * (w of lane q of the row of 16 lanes), q < 8: the broadcast is the FMA's own
// DPP operand. All lanes are active wherever this runs; the wait states cover a write of w
// by the instruction before the block.
__device__ __forceinline__ void fma8_row(double (&a)[8], double w, double m)
{
#define RBFX_F8(D, Q) "v_fmac_f64_dpp %" D ", %8, %9 row_newbcast:" Q " row_mask:0xf bank_mask:0xf\n\t"
    asm("s_nop 1\n\t" RBFX_F8("0", "0") RBFX_F8("1", "1") RBFX_F8("2", "2") RBFX_F8("3", "3") RBFX_F8("4", "4")
            RBFX_F8("5", "5") RBFX_F8("6", "6") RBFX_F8("7", "7")
        : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(a[4]), "+v"(a[5]), "+v"(a[6]), "+v"(a[7])
        : "v"(w), "v"(m));
#undef RBFX_F8
}

// HERM: the build may carry boundary data. Launches without any (P.is_boundary null)
// whose LDS is small enough use the instantiation without the Hermite paths, whose
// smaller register allocation leaves room for more wavefronts per SIMD
template <int DIM, int RC, int TWO, bool HERM>
__global__ __attribute__((amdgpu_flat_work_group_size(64, 64))) void k_build_sym(const BuildDev P, int rows_cap,
                                                                                 int tri)
{
    constexpr int ROWS = 64 * TWO;
    static_assert(HERM || TWO == 1, "the instantiation without Hermite paths serves up to 64 rows");
    // the packed triangle (tri doubles) is the whole dynamic LDS: the right-hand sides,
    // the stencil points and their boundary data stay in the registers of the lanes that
    // own them and are read by the others with lane reads
    extern __shared__ __attribute__((aligned(16))) double s_T[];
    // (no static LDS, which would count toward the wavefronts per CU: the monomial exponents
    // and operator terms are read from the kernel arguments)

    const int L = threadIdx.x;
    const int n_cols = P.n_cols, n_terms = P.n_terms;
    auto mono_exps = [&](int a, int(&ex)[3]) {
        ex[0] = P.mono_e[a][0];
        ex[1] = P.mono_e[a][1];
        ex[2] = P.mono_e[a][2];
    };

    // one stencil per workgroup: every exit below is uniform over the workgroup
    const int64_t lb = xcd_contiguous_block(P.n_blocks);
    if (lb < 0) return;
    const int64_t n_work = P.list ? (int64_t)*P.list_len : P.n_eval;
    if (lb >= n_work) return;
    const int64_t e = P.list ? (int64_t)P.list[lb] : (P.order ? (int64_t)P.order[lb] : lb);
    if (e < 0 || e >= P.n_eval) return;
    const int64_t s0 = P.adj_ptr ? P.adj_ptr[e] : e * (int64_t)P.k;
    const int kk = P.adj_ptr ? (int)(P.adj_ptr[e + 1] - s0) : P.k;
    const int64_t o0 = P.out_ptr ? P.out_ptr[e] : e * (int64_t)P.k;
    const int M = stencil_n_mono(P, e, DIM);
    if (M < 0) {
        if (L == 0 && P.status) P.status[e] = RBFX_ST_INVALID;
        return;
    }
    if (kk < 1 || M + kk > rows_cap) {
        if (L == 0 && P.status) P.status[e] = RBFX_ST_TOO_LARGE;
        return;
    }
    const int n = M + kk;

    // ---- the stencil points this lane loads: q = L (and q = L + 64)
    double xe[DIM];
#pragma unroll
    for (int d = 0; d < DIM; ++d) xe[d] = P.eval[e * DIM + d];
    int gidx[TWO] = {};
    double D[TWO][DIM];
    double r2max = 0.0;
    bool ib[TWO] = {};
#pragma unroll
    for (int t = 0; t < TWO; ++t) {
        const int q = L + 64 * t;
#pragma unroll
        for (int d = 0; d < DIM; ++d) D[t][d] = 0.0;
        if (q < kk) {
            gidx[t] = P.adj_idx[s0 + q];
            double r2 = 0.0;
#pragma unroll
            for (int d = 0; d < DIM; ++d) {
                D[t][d] = P.data[(int64_t)gidx[t] * DIM + d] - xe[d];
                r2 += D[t][d] * D[t][d];
            }
            r2max = fmax(r2max, r2);
            ib[t] = HERM && P.is_boundary && P.is_boundary[gidx[t]];
        }
    }
    // stencil classification (types.jl:208-223)
    const bool hermite = HERM && P.is_boundary && (__ballot(ib[0] || ib[TWO - 1]) != 0ull);
    // a Dirichlet eval node is an identity row whatever its neighbours are (the row
    // length count_nonzeros gives it, execution.jl:39-69)
    if (HERM && P.is_boundary && e < P.n_data && P.is_boundary[e]) {
        const int bi = P.bnd_index[e];
        if (P.bc_alpha[bi] == 1.0 && P.bc_beta[bi] == 0.0) {
            // identity row (fill_dirichlet_entry!, execution.jl:297-303)
            if (L < n_cols) P.out_val[(int64_t)L * P.out_nnz + o0] = 1.0;
            if (L == 0) {
                if (P.out_col) P.out_col[o0] = (int32_t)e;
                if (P.status) P.status[e] = RBFX_ST_DIRICHLET;
            }
            return;
        }
    }
    double h = sqrt(group_max<64>(r2max));
    if (!(h > 0.0)) h = 1.0;
    const double hinv = 1.0 / h;
    unsigned long long at_eval[TWO];
    // this lane's points q = L + 64 t: the scaled coordinates and, for stencils with
    // boundary points, the boundary type (1 Dirichlet, 2 Neumann/Robin), the coefficients
    // (beta scaled by 1/h: it acts through a first derivative) and the normal
    double xo[TWO][DIM], bno[TWO][DIM], bao[TWO], bbo[TWO];
    int bto[TWO];
#pragma unroll
    for (int t = 0; t < TWO; ++t) {
        const int q = L + 64 * t;
        bool eq = false;
        bao[t] = 0.0;
        bbo[t] = 0.0;
        bto[t] = 0;
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            xo[t][d] = 0.0;
            bno[t][d] = 0.0;
        }
        if (q < kk) {
            if (hermite && ib[t]) {
                const int bi = P.bnd_index[gidx[t]];
                const double ba = P.bc_alpha[bi], bb = P.bc_beta[bi];
#pragma unroll
                for (int d = 0; d < DIM; ++d) bno[t][d] = P.normals[(int64_t)bi * DIM + d];
                bto[t] = (ba == 1.0 && bb == 0.0) ? 1 : 2;
                bao[t] = ba;
                bbo[t] = bb / h;
            }
            eq = hermite;
#pragma unroll
            for (int d = 0; d < DIM; ++d) {
                xo[t][d] = D[t][d] / h;
                eq = eq && (D[t][d] == 0.0);
            }
        }
        at_eval[t] = __ballot(eq);
    }
    // point q's data (q uniform), from the lane that loaded it
    auto pq_sel = [&](int q) -> int { return __builtin_amdgcn_readfirstlane(q); };
    auto px = [&](int q, int d) -> double {
        const int c = pq_sel(q);
        return (TWO == 2 && c >= 64) ? rdlane(xo[TWO - 1][d], c & 63) : rdlane(xo[0][d], c & 63);
    };
    auto pbn = [&](int q, int d) -> double {
        const int c = pq_sel(q);
        return (TWO == 2 && c >= 64) ? rdlane(bno[TWO - 1][d], c & 63) : rdlane(bno[0][d], c & 63);
    };
    auto pba = [&](int q) -> double {
        const int c = pq_sel(q);
        return (TWO == 2 && c >= 64) ? rdlane(bao[TWO - 1], c & 63) : rdlane(bao[0], c & 63);
    };
    auto pbb = [&](int q) -> double {
        const int c = pq_sel(q);
        return (TWO == 2 && c >= 64) ? rdlane(bbo[TWO - 1], c & 63) : rdlane(bbo[0], c & 63);
    };
    auto pbt = [&](int q) -> int {
        const int c = pq_sel(q);
        return (TWO == 2 && c >= 64) ? rdlane(bto[TWO - 1], c & 63) : rdlane(bto[0], c & 63);
    };
    int eval_local = 0;
    if (hermite) {
        const unsigned long long ae1 = TWO == 2 ? at_eval[TWO - 1] : 0ull;
        if (!at_eval[0] && !ae1) {
            if (L == 0 && P.status) P.status[e] = RBFX_ST_EVAL_NOT_FOUND;
            return;
        }
        eval_local = at_eval[0] ? __builtin_ctzll(at_eval[0]) : 64 + __builtin_ctzll(ae1);
    }
    __syncthreads();

    BasisDev B;
    B.kind = P.basis_kind;
    B.eps = (B.kind == RBFX_IMQ || B.kind == RBFX_GAUSSIAN) ? P.eps * h : P.eps;

    // positions: point q at q, monomial a at kk + a; orig: the row index of the
    // saddle-point system (monomials 0..M-1, then the points)
    int rbj[TWO], orig[TWO];
#pragma unroll
    for (int t = 0; t < TWO; ++t) {
        const int j = L + 64 * t;
        rbj[t] = kSymRb.rb[j] * 8;
        orig[t] = j < kk ? M + j : (j < n ? j - kk : 255);
    }
    // an entry by its byte offset (row starts are kept in bytes: no shifts on the way)
    auto T = [&](int off) -> double& { return *(double*)((char*)s_T + off); };
    // start of row c (c uniform): from the lane that owns position c
    auto rb_of = [&](int c) -> int {
        const int cc = __builtin_amdgcn_readfirstlane(c);
        return (TWO == 2 && cc >= 64) ? rdlane(rbj[TWO - 1], cc & 63) : rdlane(rbj[0], cc & 63);
    };

    // ---- assembly (FP64) of the lower triangle and the right-hand sides (registers: lane
    // L holds those of its positions)
    double bcol[RC][TWO];
#pragma unroll
    for (int t = 0; t < TWO; ++t)
#pragma unroll
        for (int c = 0; c < RC; ++c) bcol[c][t] = 0.0;
    // Without boundary points phi is symmetric, so each pair is computed once: the lane of
    // point j takes the points j + d (mod k) for d = 0..k/2, up to 32 points on both halves of
    // the wavefront, even and odd d (30 points: 8 evaluations a lane instead of 30)
    const bool around = !hermite && kk <= 64;
    auto point_pairs = [&](auto KC) __attribute__((always_inline)) {
        const int two = kk <= 32 ? 1 : 0, step = 1 + two;
        const int j = two ? L & 31 : L;
        double xj[DIM];
#pragma unroll
        for (int d = 0; d < DIM; ++d) xj[d] = __shfl(xo[0][d], j, 64);
        const int rb_own = __shfl(rbj[0], j, 64);
        int d = two ? L >> 5 : 0, jj = j + d;
        if (jj >= kk) jj -= kk;
        for (int d0 = 0; d0 <= kk / 2; d0 += step) {
            double q2 = 0.0;
#pragma unroll
            for (int x = 0; x < DIM; ++x) {
                const double t_ = xj[x] - __shfl(xo[0][x], jj, 64);
                q2 += t_ * t_;
            }
            const int rb_other = __shfl(rbj[0], jj, 64);
            const double v = phi_r2_k<decltype(KC)::value>(B.eps, q2);
            if (j < kk && d <= kk / 2) T(jj > j ? rb_other + 8 * j : rb_own + 8 * jj) = v;
            d += step;
            jj += step;
            if (jj >= kk) jj -= kk;
        }
    };
    // With boundary points (or more than 64): row j's entries one after another. The lane
    // reads stand outside the branches: a lane that a branch leaves out need not hold its
    // registers inside it.
    auto point_rows = [&](auto KC) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < TWO; ++t) {
            const int j = L + 64 * t;
            for (int jj = 0; jj < kk; ++jj) {
                double xj[DIM], nj[DIM];
#pragma unroll
                for (int d = 0; d < DIM; ++d) {
                    xj[d] = px(jj, d);
                    nj[d] = HERM ? pbn(jj, d) : 0.0;
                }
                const int tj = HERM ? pbt(jj) : 0;
                const double aj = HERM ? pba(jj) : 0.0, bj = HERM ? pbb(jj) : 0.0;
                if (j >= kk || jj > j) continue;
                double Dj[DIM], q2 = 0.0;
#pragma unroll
                for (int d = 0; d < DIM; ++d) {
                    Dj[d] = xo[t][d] - xj[d];
                    q2 += Dj[d] * Dj[d];
                }
                double v = phi_r2_k<decltype(KC)::value>(B.eps, q2);
                if (HERM && (bto[t] == 2 || tj == 2)) {
                    const double ba = bao[t], bb = bbo[t];
                    double Di, Djn, D2;
                    phi_grad_hess_dirs<DIM>(B, Dj, q2, bno[t], nj, Di, Djn, D2);
                    if (bto[t] != 2) v = aj * v - bj * Djn;
                    else if (tj != 2) v = ba * v + bb * Di;
                    else v = ba * aj * v - ba * bj * Djn + bb * aj * Di + bb * bj * D2;
                }
                T(rbj[t] + 8 * jj) = v;
            }
        }
    };
    // right-hand sides of the point rows
    auto point_rhs = [&](auto KC) __attribute__((always_inline)) {
        BasisDev Bk;
        Bk.kind = decltype(KC)::value;
        Bk.eps = B.eps;
#pragma unroll
        for (int t = 0; t < TWO; ++t) {
            if (L + 64 * t >= kk) continue;
            double De[DIM], q2 = 0.0;
#pragma unroll
            for (int d = 0; d < DIM; ++d) {
                De[d] = -xo[t][d];
                q2 += De[d] * De[d];
            }
            for (int tt = 0; tt < n_terms; ++tt) {
                const TermDev tm = P.terms[tt];
                // (or the roots and quotients of every term kind move out of the loop)
                double q2t = q2;
                asm volatile("" : "+v"(q2t));
                double v = phi_term<DIM>(Bk, tm.kind, tm.d1, tm.d2, De, q2t);
                if (hermite && bto[t] == 2)
                    v = bao[t] * v + bbo[t] * phi_term_normal<DIM>(Bk, tm.kind, tm.d1, De, q2t, bno[t]);
                const double sc = term_scale(tm, hinv);
#pragma unroll
                for (int c = 0; c < RC; ++c)
                    bcol[c][t] = tm.col == c ? bcol[c][t] + sc * v : bcol[c][t];
            }
        }
    };
    auto point_block = [&](auto KC) __attribute__((always_inline)) {
        if (around) point_pairs(KC);
        else point_rows(KC);
        point_rhs(KC);
    };
    switch (B.kind) {
    case RBFX_PHS1: point_block(std::integral_constant<int, RBFX_PHS1>{}); break;
    case RBFX_PHS3: point_block(std::integral_constant<int, RBFX_PHS3>{}); break;
    case RBFX_PHS5: point_block(std::integral_constant<int, RBFX_PHS5>{}); break;
    case RBFX_PHS7: point_block(std::integral_constant<int, RBFX_PHS7>{}); break;
    case RBFX_IMQ: point_block(std::integral_constant<int, RBFX_IMQ>{}); break;
    default: point_block(std::integral_constant<int, RBFX_GAUSSIAN>{}); break;
    }
    // the eval node's boundary condition (stencils with boundary points)
    const bool eval_normal = hermite && pbt(eval_local) == 2;
    const double eav = HERM ? pba(eval_local) : 0.0, ebv = HERM ? pbb(eval_local) : 0.0;
    double en[DIM];
#pragma unroll
    for (int d = 0; d < DIM; ++d) en[d] = HERM ? pbn(eval_local, d) : 0.0;
#pragma unroll
    for (int t = 0; t < TWO; ++t) {
        const int j = L + 64 * t;
        if (j >= n) continue;
        const bool is_poly = j >= kk;
        if (!is_poly) {
            // the point's monomial values: column j of monomial row a (position kk + a)
            for (int a = 0; a < M; ++a) {
                int ea[3];
                mono_exps(a, ea);
                double v = 1.0;
#pragma unroll
                for (int d = 0; d < DIM; ++d) {
                    double w = 1.0;
#pragma unroll 1
                    for (int q = 0; q < ea[d]; ++q) w *= xo[t][d];
                    v *= w;
                }
                if (hermite && bto[t] == 2) v = bao[t] * v + bbo[t] * mono_normal<DIM>(ea, bno[t], xo[t]);
                s_T[kSymRb.rb[kk + a] + j] = v;
            }
        } else {
            // monomial row a = j - kk: zero at the monomial positions kk..j, and its right-hand
            // sides
            for (int c = kk; c <= j; ++c) T(rbj[t] + 8 * c) = 0.0;
            double z[DIM];
#pragma unroll
            for (int d = 0; d < DIM; ++d) z[d] = 0.0;
            int ea[3];
            mono_exps(j - kk, ea);
            if (eval_normal) {
                // the eval node's boundary operator applied to P (assembly.jl:452-467)
                const double v = eav * mono_op<DIM>(ea, RBFX_OP_VALUE, 0, 0, z) + ebv * mono_normal<DIM>(ea, en, z);
#pragma unroll
                for (int c = 0; c < RC; ++c) bcol[c][t] = v;
            } else {
                for (int tt = 0; tt < n_terms; ++tt) {
                    const TermDev tm = P.terms[tt];
                    const double v = term_scale(tm, hinv) * mono_op<DIM>(ea, tm.kind, tm.d1, tm.d2, z);
#pragma unroll
                    for (int c = 0; c < RC; ++c)
                        bcol[c][t] = tm.col == c ? bcol[c][t] + v : bcol[c][t];
                }
            }
        }
    }
    __syncthreads();

    // ---- factorisation with rook pivoting and symmetric moves of the pivots
    const double alpha = 0.6403882032022076;  // (1 + sqrt(17)) / 8
    int n_act = n;
    bool failed = false;
    auto bits = [&](int count, int t) -> unsigned long long {
        const int c = count - 64 * t;
        return c >= 64 ? ~0ull : (c > 0 ? (1ull << c) - 1ull : 0ull);
    };
    // the original indices still active, and the positions where a 2x2 pivot starts
    unsigned long long om[TWO], twos[TWO];
#pragma unroll
    for (int t = 0; t < TWO; ++t) {
        om[t] = bits(n, t);
        twos[t] = 0ull;
    }
    // The trailing update's rows: lane L updates row jr; with up to 32 active rows, both
    // halves of the wavefront share the rows, the upper half eight columns on.
    int jr = L, rbu = rbj[0];
    bool shared = false;
    const int cadd = (L >> 2) & 8, cadd8 = 8 * cadd, wlane = 8 * (L & 7);
    auto share_rows = [&]() {
        jr = L & 31;
        rbu = __shfl(rbj[0], L & 31, 64);
        shared = true;
    };
    if (n_act <= 32) share_rows();
    // S: the slots that hold active rows. Systems of more than 64 rows start with two; once
    // 64 rows are left, the loop for one slot takes over, without the choices between them.
    auto factorise = [&](auto SL) __attribute__((always_inline)) {
        constexpr int S = decltype(SL)::value;
        auto row_at = [&](int c) __attribute__((always_inline)) -> int {
            if constexpr (S == 2) return rb_of(c);
            else return rdlane(rbj[0], c);
        };
        // Column c (uniform) of the active block to this lane's registers (v[t] = A(j, c)
        // for its positions j < n_act: row j's entry if c <= j, else row c's entry j), and
        // the largest |A(j, c)| over active j != c as a packed (magnitude, position) key.
        double v[S];
        auto colkey = [&](int c) -> uint32_t {
            const int cc = __builtin_amdgcn_readfirstlane(c);
            const int rbc = row_at(cc);
            uint32_t k = 0u;
#pragma unroll
            for (int t = 0; t < S; ++t) {
                const int j = L + 64 * t;
                unsigned long long m = bits(n_act, t);
                if (S == 1 || cc >> 6 == t) m &= ~(1ull << (cc & 63));
                // (lanes past the active rows read entry (0, cc) or of row cc, and are masked)
                v[t] = T(j >= cc ? (j < n_act ? rbj[t] : 0) + 8 * cc : rbc + 8 * j);
                k = max(k, lanes_in(m, row_key(v[t], j) & 0x7fffffffu));
            }
            return first_max_u32(k, n_act);
        };
        auto colval = [&](int r) -> double {
            const int rr = __builtin_amdgcn_readfirstlane(r);
            return (S == 2 && rr >= 64) ? rdlane(v[S - 1], rr & 63) : rdlane(v[0], rr & 63);
        };
        // symmetric swap of positions lo <= hi (both active): the rows and the columns, for
        // every row of the system (frozen rows keep their entries at the active positions);
        // each entry of the lower triangle that moves is moved by exactly one lane: lane k
        // swaps (k, lo) with (k, hi), lane lo the diagonal entries, lane hi nothing
        auto swap_entries = [&](int lo, int hi, int rhi) {
            const int rlo = row_at(lo);
#pragma unroll
            for (int t = 0; t < TWO; ++t) {
                const int k = L + 64 * t;
                if (k >= n || k == hi) continue;
                const int k8 = 8 * k;
                const int x0 = k >= lo ? rbj[t] + 8 * lo : rlo + k8;
                const int x1 = k > hi ? rbj[t] + 8 * hi : rhi + (k == lo ? 8 * hi : k8);
                const double y0 = T(x0), y1 = T(x1);
                T(x0) = y1;
                T(x1) = y0;
            }
        };
        auto lane_put = [&](auto& w, auto v_, int p) __attribute__((always_inline)) {
            if constexpr (S == 2) {
                const auto w0 = w[0], w1 = w[1];  // (by value: a choice of elements would go to memory)
                w[0] = p < 64 ? wrlane(w0, v_, p & 63) : w0;
                w[1] = p < 64 ? w1 : wrlane(w1, v_, p & 63);
            } else {
                w[0] = wrlane(w[0], v_, p);
            }
        };
        auto lane_get = [&](const auto& w, int p) __attribute__((always_inline)) {
            const auto w0 = w[0], w1 = w[S - 1];
            const auto a0 = rdlane(w0, p & 63);
            if constexpr (S == 2) return p < 64 ? a0 : rdlane(w1, p & 63);
            else return a0;
        };
        // The pivot of position p goes to the last active position q: its row start rq is
        // returned, its right-hand sides in vq.
        auto freeze = [&](int p, int q, double(&vq)[RC]) __attribute__((always_inline)) -> int {
            const int rq = row_at(q), o = lane_get(orig, p);
            if (TWO == 2 && o >= 64) om[TWO - 1] &= ~(1ull << (o & 63));
            else om[0] &= ~(1ull << (o & 63));
#pragma unroll
            for (int c = 0; c < RC; ++c) vq[c] = lane_get(bcol[c], p);
            if (p != q) {
                swap_entries(p, q, rq);
                lane_put(orig, lane_get(orig, q), p);
                lane_put(orig, o, q);
#pragma unroll
                for (int c = 0; c < RC; ++c) {
                    lane_put(bcol[c], lane_get(bcol[c], q), p);
                    lane_put(bcol[c], vq[c], q);
                }
            }
            return rq;
        };
        while (n_act > (S == 2 ? 64 : 0)) {
            // the active row of the lowest original index starts the search
            int c0;
            {
                const bool first = TWO == 1 || om[0] != 0ull;
                const int o = first ? __builtin_ctzll(om[0]) : 64 + __builtin_ctzll(om[TWO - 1]);
                const unsigned long long m0 = __ballot(orig[0] == o), m1 = S == 2 ? __ballot(orig[S - 1] == o) : 0ull;
                c0 = (S == 1 || m0) ? __builtin_ctzll(m0) : 64 + __builtin_ctzll(m1);
            }
            const uint32_t ck = colkey(c0);
            int imax = ck ? 127 - (int)(ck & 127u) : c0;
            const double akk = colval(c0);
            double colmax = ck ? fabs(colval(imax)) : 0.0;
            const double absakk = fabs(akk);
            int kstep = 1, p = c0, kp = c0;
            // A(p, p), A(kp, kp) and, for a 2x2 pivot, A(p, kp) as the search ends
            double app = akk, akp = akk, apk = akk;
            bool need_rook = absakk < alpha * colmax;
            if (!need_rook && !(absakk > 0.0 || colmax > 0.0)) {
                failed = true;  // zero column: singular (a search has colmax > 0)
                break;
            }
            for (int it = 0; it < 2 * ROWS && need_rook; ++it) {
                const uint32_t rk = colkey(imax);
                const int ri = rk ? 127 - (int)(rk & 127u) : imax;
                const double rowmax = rk ? fabs(colval(ri)) : 0.0;
                const double aim = colval(imax);
                const double aii = fabs(aim);
                if (!(aii < alpha * rowmax)) {
                    kp = imax;
                    akp = aim;
                    need_rook = false;
                } else if (p == ri || rowmax <= colmax || it == 2 * ROWS - 1) {
                    kp = imax;
                    kstep = 2;
                    akp = aim;
                    apk = colval(p);  // column imax holds A(p, imax)
                    need_rook = false;
                } else {
                    p = imax;
                    app = aim;
                    colmax = rowmax;
                    imax = ri;
                }
            }
            kstep = __builtin_amdgcn_readfirstlane(kstep);
            const int p0 = __builtin_amdgcn_readfirstlane((kstep == 1) ? kp : p);
            const int p1 = __builtin_amdgcn_readfirstlane(kp);  // equals p0 for a 1x1 pivot
            // A(p0, p0), A(p1, p1), A(p0, p1)
            const double d0 = kstep == 1 ? akp : app, d1 = akp, bq = kstep == 1 ? akp : apk;
            double idet = 0.0;
            if (kstep == 1) {
                failed = d0 == 0.0;
            } else {
                const double det = d0 * d1 - bq * bq;
                failed = det == 0.0;
                idet = 1.0 / det;
            }
            if (failed) break;
            // p0 to position n_act - 1, p1 (2x2) to n_act - 2
            double v0[RC], v1[RC];
            const int q0 = n_act - 1, r0 = freeze(p0, q0, v0);
            int r1 = r0;
#pragma unroll
            for (int c = 0; c < RC; ++c) v1[c] = 0.0;
            if (kstep == 2) {
                r1 = freeze(p1 == q0 ? p0 : p1, q0 - 1, v1);
                const unsigned long long bit = 1ull << ((q0 - 1) & 63);
                twos[0] |= S == 1 || q0 - 1 < 64 ? bit : 0ull;
                if (S == 2) twos[S - 1] |= q0 - 1 < 64 ? 0ull : bit;
            }
            n_act -= kstep;
            if (n_act <= 32 && !shared) share_rows();
            // The trailing update of the active rows j < n_act over their columns 0..j, eight at a
            // time (the chunk past the diagonal lands in the row's padding), and of their
            // right-hand sides; per element the FMAs run in the same order as in k_build_wide. The
            // pivot row's eight entries are one read, spread over the lanes and broadcast by the
            // FMAs. Every lane reads and multiplies (lanes without a row: row 0), those whose
            // chunk lies in their row write.
            const int na = S == 2 ? min(n_act, 64) : n_act;
            const bool on = jr < na;
            const int row = on ? rbu : 0;
            auto update = [&](auto KS) __attribute__((always_inline)) {
                constexpr int K = decltype(KS)::value;
                auto factors = [&](int j, double& ml0, double& ml1) __attribute__((always_inline)) {
                    const double u0 = T(r0 + 8 * j);
                    double l0, l1 = 0.0;
                    if (K == 1) {
                        l0 = u0 / d0;
                    } else {
                        const double u1 = T(r1 + 8 * j);
                        l0 = (u0 * d1 - u1 * bq) * idet;
                        l1 = (u1 * d0 - u0 * bq) * idet;
                    }
                    ml0 = -l0;
                    ml1 = -l1;
                };
                double ml0, ml1;
                factors(jr, ml0, ml1);
                auto chunk = [&](int A, int W, int cc) __attribute__((always_inline)) {
                    double a[8], w1 = 0.0;
                    const double w0 = T(r0 + W);
                    if (K == 2) w1 = T(r1 + W);
#pragma unroll
                    for (int q = 0; q < 8; ++q) a[q] = T(A + 8 * q);
                    fma8_row(a, w0, ml0);
                    if (K == 2) fma8_row(a, w1, ml1);
                    if (on && cc <= jr) {
#pragma unroll
                        for (int q = 0; q < 8; ++q) T(A + 8 * q) = a[q];
                    }
                };
                if (n_act <= 32) {
                    if (n_act > 0) chunk(row + cadd8, wlane + cadd8, cadd);
                    if (n_act > 16) chunk(row + cadd8 + 128, wlane + cadd8 + 128, cadd + 16);
                } else {
                    for (int cc = 0; cc < na; cc += 8) chunk(row + 8 * cc, wlane + 8 * cc, cc);
                }
#pragma unroll
                for (int c = 0; c < RC; ++c) {
                    const double b0 = fma(ml0, v0[c], bcol[c][0]);
                    const double b = K == 1 ? b0 : fma(ml1, v1[c], b0);
                    bcol[c][0] = L < na ? b : bcol[c][0];
                }
                if constexpr (S == 2) {
                    // rows 64.. (the first steps of a system of more than 64 rows)
                    const int j = L + 64;
                    if (j < n_act) {
                        factors(j, ml0, ml1);
                        for (int j0 = 0; j0 <= j; j0 += 8) {
#pragma unroll
                            for (int q = 0; q < 8; ++q) {
                                const int o = 8 * (j0 + q);
                                const double a0 = fma(ml0, T(r0 + o), T(rbj[1] + o));
                                T(rbj[1] + o) = K == 1 ? a0 : fma(ml1, T(r1 + o), a0);
                            }
                        }
#pragma unroll
                        for (int c = 0; c < RC; ++c)
                            bcol[c][1] = K == 1 ? fma(ml0, v0[c], bcol[c][1])
                                                 : fma(ml1, v1[c], fma(ml0, v0[c], bcol[c][1]));
                    }
                }
            };
            if (kstep == 1) update(std::integral_constant<int, 1>{});
            else update(std::integral_constant<int, 2>{});
            __syncthreads();
        }
    };
    if constexpr (TWO == 2) factorise(std::integral_constant<int, 2>{});
    if (!failed) factorise(std::integral_constant<int, 1>{});
    __syncthreads();

    // ---- back substitution, last pivot (position 0) first: the rows frozen before a pivot
    // are the positions above it. A lane holds the reciprocal of its own diagonal entry and
    // its right-hand side less what the solved positions below it contribute: its weight,
    // once those are all solved, is the product.
    double x[TWO][RC], acc[TWO][RC], dinv[TWO];
    unsigned long long in_two[TWO];  // positions of 2x2 pivots (solved explicitly)
#pragma unroll
    for (int t = 0; t < TWO; ++t) {
        const int j = L + 64 * t;
        dinv[t] = 0.0;
        in_two[t] = twos[t] << 1 | twos[t] | (t ? twos[0] >> 63 : 0ull);
#pragma unroll
        for (int c = 0; c < RC; ++c) {
            x[t][c] = 0.0;
            acc[t][c] = 0.0;
        }
        if (!failed && j < n) dinv[t] = 1.0 / T(rbj[t] + 8 * j);
    }
    auto lane_get = [&](const auto& w, int p) __attribute__((always_inline)) {
        const auto w0 = w[0], w1 = w[TWO - 1];
        const auto a0 = rdlane(w0, p & 63);
        if constexpr (TWO == 2) return p < 64 ? a0 : rdlane(w1, p & 63);
        else return a0;
    };
    if (!failed) {
        for (int pq = 0; pq < n;) {
            const bool two = ((TWO == 1 || pq < 64 ? twos[0] : twos[TWO - 1]) >> (pq & 63)) & 1ull;
            // the block's pivots: pp (p0) and, for a 2x2, pq (p1) below it
            const int pp = two ? pq + 1 : pq;
            if (!two) {
                double arp[TWO];
#pragma unroll
                for (int t = 0; t < TWO; ++t) {
                    const int j = L + 64 * t;
                    arp[t] = (j > pp && j < n) ? T(rbj[t] + 8 * pp) : 0.0;
                }
#pragma unroll
                for (int c = 0; c < RC; ++c) {
                    if (c >= n_cols) continue;
                    double r[TWO];
#pragma unroll
                    for (int t = 0; t < TWO; ++t) r[t] = (bcol[c][t] - acc[t][c]) * dinv[t];
                    const double x0 = lane_get(r, pp);
#pragma unroll
                    for (int t = 0; t < TWO; ++t) {
                        const int j = L + 64 * t;
                        if (j > pp && j < n) acc[t][c] += arp[t] * x0;
                    }
                }
                pq += 1;
                continue;
            }
            const int rbp = rb_of(pp), rbq = rb_of(pq);
            const double dp = T(rbp + 8 * pp), dq = T(rbq + 8 * pq), bq = T(rbp + 8 * pq);
            double arp[TWO], arq[TWO];
#pragma unroll
            for (int t = 0; t < TWO; ++t) {
                const int j = L + 64 * t;
                const bool above = j > pp && j < n;
                arp[t] = above ? T(rbj[t] + 8 * pp) : 0.0;
                arq[t] = above ? T(rbj[t] + 8 * pq) : 0.0;
            }
            const double idet = 1.0 / (dp * dq - bq * bq);
#pragma unroll
            for (int c = 0; c < RC; ++c) {
                if (c >= n_cols) continue;
                double r[TWO];
#pragma unroll
                for (int t = 0; t < TWO; ++t) r[t] = bcol[c][t] - acc[t][c];
                const double yp = lane_get(r, pp), yq = lane_get(r, pq);
                const double x0 = (yp * dq - yq * bq) * idet;
                const double x1 = (yq * dp - yp * bq) * idet;
#pragma unroll
                for (int t = 0; t < TWO; ++t) {
                    const int j = L + 64 * t;
                    if (j == pp) x[t][c] = x0;
                    if (j == pq) x[t][c] = x1;
                    if (j > pp && j < n) acc[t][c] += arp[t] * x0 + arq[t] * x1;
                }
            }
            pq += 2;
        }
#pragma unroll
        for (int t = 0; t < TWO; ++t) {
            if ((in_two[t] >> L) & 1ull) continue;
#pragma unroll
            for (int c = 0; c < RC; ++c) x[t][c] = (bcol[c][t] - acc[t][c]) * dinv[t];
        }
    }

    // ---- outputs: weights of the point rows, multipliers of the monomial rows
#pragma unroll
    for (int t = 0; t < TWO; ++t) {
        const int j = L + 64 * t;
        if (j >= n) continue;
        const int i = orig[t];
#pragma unroll
        for (int c = 0; c < RC; ++c) {
            if (c >= n_cols) continue;
            const double v_ = failed ? __builtin_nan("") : x[t][c];
            if (i >= M) P.out_val[(int64_t)c * P.out_nnz + o0 + (i - M)] = v_;
            else if (P.out_lambda) P.out_lambda[((int64_t)c * P.n_eval + e) * P.n_mono + i] = v_;
        }
        if (i >= M && P.out_col) P.out_col[o0 + (i - M)] = P.adj_idx[s0 + (i - M)];
    }
    if (L == 0 && P.status) P.status[e] = failed ? RBFX_ST_SINGULAR : P.ok_status;
}

static int rc_class(int n_cols) { return n_cols <= 1 ? 1 : (n_cols <= 4 ? 4 : 8); }
// odd: the columns rounded up to a multiple of eight, then the right-hand sides
static int wide_lda(int rows_cap, int n_cols) { return (((rows_cap + 7) & ~7) + rc_class(n_cols)) | 1; }
// dynamic LDS: the system, then per row the scaled point and, for builds with boundary
// data, the normal, two boundary coefficients and a boundary type
static size_t wide_lds(int rows_cap, int n_cols, int dim, bool bnd)
{
    return (size_t)rows_cap * wide_lda(rows_cap, n_cols) * 8 + (size_t)rows_cap * dim * 8 +
           (bnd ? (size_t)rows_cap * (dim + 2) * 8 + (size_t)rows_cap * 4 : 0);
}

// the system plus the kernel's static tables within 64 KB of LDS
constexpr int64_t kWideStaticLds = 2 * 1024;
bool wide_fits(int rows_cap, int n_cols)
{
    return rows_cap >= 1 && rows_cap <= RBFX_MAX_N &&
           (int64_t)wide_lds(rows_cap, n_cols, 3, true) + kWideStaticLds <= 65536;
}

template <int DIM, int RC>
static hipError_t launch_wide_rc(const BuildDev& P, int rows_cap, int64_t n_work, hipStream_t s)
{
    BuildDev Q = P;
    Q.n_blocks = n_work;
    const int lda = wide_lda(rows_cap, P.n_cols);
    const size_t lds = wide_lds(rows_cap, P.n_cols, DIM, P.is_boundary != nullptr);
    if (rows_cap <= 64)
        hipLaunchKernelGGL((k_build_wide<DIM, RC, 1>), dim3((unsigned)pad_to_xcds(n_work)), dim3(64), lds, s, Q,
                           rows_cap, lda);
    else
        hipLaunchKernelGGL((k_build_wide<DIM, RC, 2>), dim3((unsigned)pad_to_xcds(n_work)), dim3(64), lds, s, Q,
                           rows_cap, lda);
    return hipGetLastError();
}

template <int DIM>
static hipError_t launch_wide_dim(const BuildDev& P, int rows_cap, int64_t n_work, hipStream_t s)
{
    switch (rc_class(P.n_cols)) {
    case 1: return launch_wide_rc<DIM, 1>(P, rows_cap, n_work, s);
    case 4: return launch_wide_rc<DIM, 4>(P, rows_cap, n_work, s);
    default: return launch_wide_rc<DIM, 8>(P, rows_cap, n_work, s);
    }
}

hipError_t launch_build_wide(const BuildDev& P, int dim, int rows_cap, int64_t n_work, hipStream_t s)
{
    if (n_work <= 0) return hipSuccess;
    if (!wide_fits(rows_cap, P.n_cols)) return hipErrorInvalidValue;
    switch (dim) {
    case 1: return launch_wide_dim<1>(P, rows_cap, n_work, s);
    case 2: return launch_wide_dim<2>(P, rows_cap, n_work, s);
    case 3: return launch_wide_dim<3>(P, rows_cap, n_work, s);
    default: return hipErrorInvalidValue;
    }
}

// dynamic LDS of k_build_sym: the packed triangle, and the entries that lanes
// without a row may read past it in the trailing update (position 31 of row 0 at most, and
// eight past a row's end)
static int sym_tri(int rows_cap) { return kSymRbHost.rb[rows_cap] + 24; }
static size_t sym_lds(int rows_cap, int n_cols)
{
    (void)n_cols;  // (the right-hand sides live in registers)
    return (size_t)sym_tri(rows_cap) * 8;
}

bool sym_fits(int rows_cap, int n_cols)
{
    return rows_cap >= 1 && rows_cap <= RBFX_MAX_N &&
           (int64_t)sym_lds(rows_cap, n_cols) + kWideStaticLds <= 65536;
}

template <int DIM, int RC>
static hipError_t launch_sym_rc(const BuildDev& P, int rows_cap, int64_t n_work, hipStream_t s)
{
    BuildDev Q = P;
    Q.n_blocks = n_work;
    const int tri = sym_tri(rows_cap);
    // the instantiation without Hermite paths (fewer VGPRs) where the LDS leaves room for
    // more than the 12 wavefronts per CU of the other's registers
    const size_t lds = sym_lds(rows_cap, P.n_cols);
    const bool lean = !P.is_boundary && rows_cap <= 64 && 160 * 1024 / (lds + kWideStaticLds) > 12;
    if (lean)
        hipLaunchKernelGGL((k_build_sym<DIM, RC, 1, false>), dim3((unsigned)pad_to_xcds(n_work)), dim3(64), lds, s, Q,
                           rows_cap, tri);
    else if (rows_cap <= 64)
        hipLaunchKernelGGL((k_build_sym<DIM, RC, 1, true>), dim3((unsigned)pad_to_xcds(n_work)), dim3(64), lds, s, Q,
                           rows_cap, tri);
    else
        hipLaunchKernelGGL((k_build_sym<DIM, RC, 2, true>), dim3((unsigned)pad_to_xcds(n_work)), dim3(64), lds, s, Q,
                           rows_cap, tri);
    return hipGetLastError();
}

template <int DIM>
static hipError_t launch_sym_dim(const BuildDev& P, int rows_cap, int64_t n_work, hipStream_t s)
{
    switch (rc_class(P.n_cols)) {
    case 1: return launch_sym_rc<DIM, 1>(P, rows_cap, n_work, s);
    case 4: return launch_sym_rc<DIM, 4>(P, rows_cap, n_work, s);
    default: return launch_sym_rc<DIM, 8>(P, rows_cap, n_work, s);
    }
}

hipError_t launch_build_sym(const BuildDev& P, int dim, int rows_cap, int64_t n_work, hipStream_t s)
{
    if (n_work <= 0) return hipSuccess;
    if (!sym_fits(rows_cap, P.n_cols)) return hipErrorInvalidValue;
    switch (dim) {
    case 1: return launch_sym_dim<1>(P, rows_cap, n_work, s);
    case 2: return launch_sym_dim<2>(P, rows_cap, n_work, s);
    case 3: return launch_sym_dim<3>(P, rows_cap, n_work, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace rbfx
