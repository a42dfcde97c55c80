// rc_wave.hpp -- recompression of a low-rank gemm update by ONE wave.
//
// A task is the update C_mn -= A_mk A_nk^T of three low-rank tiles (the
// reference's hcore_dgemm QR + SVD recompression, hicma_parsec_core.c).  The
// wave owns its task from start to end: every reduction over the NB tile rows
// is a wave reduction (permlane / DPP / readlane), LDS is private to the wave
// and no barrier is shared with other waves, so a CU works on four tasks at
// once and a step with thousands of tasks fills all CUs.
//
// Mathematics (the reference's up to rounding):
//   X = Av^T Bv,  Qn = -Bu X^T,  P = [Cu Au],  Q = [Cv Qn]        (NB x s)
//   Rp, Rq = R factors of P, Q (Householder, panels of WV_PW columns)
//   M = Rp Rq^T (s x s) = Q1 R;  one-sided Jacobi on the rows of R:  R^T J = Vs S
//   -> right singular vectors Vs and singular values S of M;
//   r' = #{S >= acc} (or the fixed rank), capped at maxrank;
//   U' = P (Rq^T Vs_r)   ( = Qp Us_r S_r because P = Qp Rp, M Vs = Us S )
//   V' = Q (Rq^-1 Vs_r)  ( = Qq Vs_r     because Q = Qq Rq )
// so neither orthogonal factor is ever formed.
//
// Layout: lane l holds rows l, l+64, ... of every tall (NB-row) operand, so
// tall data is read and written coalesced and row-locally.
//
// What bounds it: FP64 VALU issue of one wave per SIMD and, in the Jacobi, the
// LDS crossbar (s doubles per lane and round); the two tall QR are 37 % of a
// task at NB = 900.  The rows of the unpivoted R are graded, which takes about half the
// sweeps that the rows of M took, and a sweep pairs only rows above the
// truncation floor: per panel step of N=90000 tile 900 (thousands of tasks)
// 3.3 -> 2.7 ms, of N=8100 tile 465 (tens) 1.45 -> 1.02 ms.
#pragma once
#include "blk.hpp"
#include "rc_task.hpp"

// Per-class sizes: SM = largest stack width of the class (32, 48 or 64).
template <int SM>
struct WvCfg {
    static constexpr int LDJ = SM + 2;             // column stride in LDS
    static constexpr int SIG = SM * LDJ;           // offset of the singular values
    static constexpr int LDS = SIG + 2 * SM;       // doubles of LDS
};
#define WV_LDS (WvCfg<WV_SMAX>::LDS)  // doubles per wave: those of the widest class

// FP64 matrix core tile C += A B with A 16x4, B 4x16, C 16x16 (gfx950
// V_MFMA_F64_16X16X4_F64).  Operand layout on the wave: A[i][k] on lane
// i + 16k, B[k][j] on lane j + 16k; result C[i][j] on lane j + 16 (i & 3),
// register i >> 2.
typedef double wv_d4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ wv_d4 mfma16(double a, double b, wv_d4 c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Columns of a tall operand: c0 columns at s0, the rest at s1, column
// stride lda (rows 0 .. NB - 1 of each are used).
struct WvSrc {
    const double *s0;
    int c0;
    const double *s1;
    int lda;
};

// One batch of A rows by buffer loads.  Column group kk (columns 4 kk ..
// 4 kk + 3, one per 16 lanes) is read from the block that holds it; when c0
// is not a multiple of 4 the group that straddles the blocks reads its
// block-0 columns into av and its block-1 columns into ax, and the MFMA
// chain takes both.  A lane outside its block reads 0, so there is neither
// a branch nor a select after a load, and loads are waited for at their use.
template <int SM, int RT>
__device__ __forceinline__ void wv_tall_ld(double (&av)[RT][SM / 4], double (&ax)[RT], int NB, int kd, wv_rsrc r0s,
                                           wv_rsrc r1s, int c0, int lda, int r0, int rstep)
{
    const int lane = threadIdx.x & 63, i16 = lane & 15, k4 = lane >> 4;
    const int cx = 4 * (c0 >> 2) + k4;  // this lane's column of the straddling group
    const bool mix = (c0 & 3) != 0 && cx >= c0 && cx < kd;
#pragma unroll
    for (int t = 0; t < RT; t++) {
        const int row = r0 + rstep * t + i16;
#pragma unroll
        for (int kk = 0; kk < SM / 4; kk++) {
            const int c = 4 * kk + k4;
            const bool b1 = 4 * kk >= c0;  // the whole group is in block 1
            const bool in = row < NB && c < kd && (b1 || c < c0);
            av[t][kk] = wv_ld(b1 ? r1s : r0s, in ? ((b1 ? c - c0 : c) * lda + row) * 8 : WV_OOB);
        }
        ax[t] = wv_ld(r1s, (mix && row < NB) ? ((cx - c0) * lda + row) * 8 : WV_OOB);
    }
}

// This lane's K operands: kv[kk][tn] = K[4 kk + k4][16 tn + i16] and
// kx[tn] = the same for the straddling group's block-1 columns, 0 where
// there is no such row.
template <int SM>
__device__ __forceinline__ void wv_tall_k(double (&kv)[SM / 4][SM / 16], double (&kx)[SM / 16], int kd, int c0,
                                          const double *Kl, int ldk)
{
    const int lane = threadIdx.x & 63, i16 = lane & 15, k4 = lane >> 4;
#pragma unroll
    for (int kk = 0; kk < SM / 4; kk++)
#pragma unroll
        for (int tn = 0; tn < SM / 16; tn++) {
            const int kr = 4 * kk + k4;
            const double v = Kl[(kr < kd ? kr : 0) * ldk + 16 * tn + i16];
            kv[kk][tn] = kr < kd ? v : 0.0;
        }
    const int cx = 4 * (c0 >> 2) + k4;
    const bool mix = (c0 & 3) != 0 && cx >= c0 && cx < kd;
#pragma unroll
    for (int tn = 0; tn < SM / 16; tn++) {
        const double v = Kl[(mix ? cx : 0) * ldk + 16 * tn + i16];
        kx[tn] = mix ? v : 0.0;
    }
}

// D rows of one batch from its loaded A rows and the K operands in
// registers: for each 16-column block of D (a uniform branch on nc), the
// MFMA chain over K runs in chunks of 16 rows (a uniform branch on kd per
// chunk), so the accumulators stay in place between MFMAs.  Stores go
// through a buffer over D's nc columns (those past it are dropped).
template <int SM, int RT>
__device__ __forceinline__ void wv_tall_mul(const double (&av)[RT][SM / 4], const double (&ax)[RT],
                                            const double (&kv)[SM / 4][SM / 16], const double (&kx)[SM / 16], int NB,
                                            int kd, int nc, double alpha, wv_rsrc dr, int r0, int rstep)
{
    const int lane = threadIdx.x & 63, i16 = lane & 15, k4 = lane >> 4;
    constexpr int KS = SM / 4, TN = SM / 16;
#pragma unroll
    for (int tn = 0; tn < TN; tn++) {
        if (16 * tn < nc) {
            wv_d4 acc[RT];
#pragma unroll
            for (int t = 0; t < RT; t++) acc[t] = mfma16(ax[t], kx[tn], wv_d4{0.0, 0.0, 0.0, 0.0});
#pragma unroll
            for (int kc = 0; kc < KS; kc += 4) {
                if (4 * kc < kd) {
#pragma unroll
                    for (int kk = kc; kk < kc + 4; kk++)
#pragma unroll
                        for (int t = 0; t < RT; t++) acc[t] = mfma16(av[t][kk], kv[kk][tn], acc[t]);
                }
            }
            const int j = 16 * tn + i16;
#pragma unroll
            for (int t = 0; t < RT; t++) {
                const int rt = r0 + rstep * t;
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int i = rt + k4 + 4 * r;
                    wv_st(alpha * acc[t][r], dr, (j < nc && i < NB) ? (i + j * NB) * 8 : WV_OOB);
                }
            }
        }
    }
}

// Tall product D (NB x nc, ld NB) = alpha * A (NB x kd) K (kd x nc) with A's
// columns given by a WvSrc and K in LDS (K[c][j] at Kl[c * ldk + j]).  Work
// goes in batches of RT 16-row tiles (tiles t0, t0 + tstep, ... when several
// waves share the product); a batch's A loads are all issued before its
// first MFMA.  K is held in registers and batches alternate
// between two register sets: batch i + 1 loads while batch i multiplies and
// stores.  Rows of a batch are read before any of them is written, so D may
// overwrite A's storage row for row.
template <int SM, int RT = (SM <= 32 ? 2 : 1)>
__device__ __forceinline__ void wv_tall_mm(int NB, int kd, int nc, double alpha, WvSrc A, const double *Kl, int ldk,
                                           double *D, int t0 = 0, int tstep = 1)
{
    const int rstep = 16 * tstep, bstep = rstep * RT;  // rows between tiles, between batches
    int r0 = 16 * t0;
    const wv_rsrc dr = wv_col_rsrc(D, NB * nc * 8);
    const int c0 = A.c0 < kd ? A.c0 : kd;
    const wv_rsrc r0s = wv_col_rsrc(A.s0, c0 * A.lda * 8), r1s = wv_col_rsrc(A.s1, (kd - c0) * A.lda * 8);
    double kv[SM / 4][SM / 16], kx[SM / 16];
    wv_tall_k<SM>(kv, kx, kd, c0, Kl, ldk);
    double a0[RT][SM / 4], x0[RT], a1[RT][SM / 4], x1[RT];
    if (r0 < NB) wv_tall_ld<SM, RT>(a0, x0, NB, kd, r0s, r1s, c0, A.lda, r0, rstep);
#pragma unroll 1
    for (; r0 < NB; r0 += 2 * bstep) {
        if (r0 + bstep < NB) wv_tall_ld<SM, RT>(a1, x1, NB, kd, r0s, r1s, c0, A.lda, r0 + bstep, rstep);
        wv_tall_mul<SM, RT>(a0, x0, kv, kx, NB, kd, nc, alpha, dr, r0, rstep);
        if (r0 + bstep >= NB) break;
        if (r0 + 2 * bstep < NB) wv_tall_ld<SM, RT>(a0, x0, NB, kd, r0s, r1s, c0, A.lda, r0 + 2 * bstep, rstep);
        wv_tall_mul<SM, RT>(a1, x1, kv, kx, NB, kd, nc, alpha, dr, r0 + bstep, rstep);
    }
}

// reduce-scatter of N = 4, 8 or 16 values: lane l returns the wave total of
// value l / (64 / N)
template <int N>
__device__ __forceinline__ double wrsN(double (&p)[N])
{
    static_assert(N == 4 || N == 8 || N == 16, "reduce-scatter width");
    if constexpr (N == 4) return wrs4(p[0], p[1], p[2], p[3]);
    else if constexpr (N == 8) return wrs8(p);
    else return wrs16(p);
}

// Buffer resources of the columns of a stack [src0 (c0 columns) | src1] in
// its first pass and of the workspace W afterwards (the fields are plain
// scalars: no indexed access to a structure in private memory).
struct WvRs {
    const double *src0, *src1, *W;
    int c0, NB;
    // column c (no bytes when !valid: loads give 0)
    __device__ __forceinline__ wv_rsrc rd(int c, bool first, bool valid) const
    {
        const double *p = !first ? W + (size_t)c * NB
                                 : (c < c0 ? src0 + (size_t)c * NB : src1 + (size_t)(c - c0) * NB);
        return wv_col_rsrc(valid ? p : W, valid ? NB * 8 : 0);
    }
    // W's column c (no bytes when !valid: stores are dropped)
    __device__ __forceinline__ wv_rsrc wr(int c, bool valid) const
    {
        return wv_col_rsrc(W + (size_t)(valid ? c : 0) * NB, valid ? NB * 8 : 0);
    }
};

// One trailing pair (b0, b1) of a panel: b -= V (T^T (V^T b)), V = the
// panel's reflectors (row block 0 in v0, the rest in a), result to W.
template <int KR>
__device__ __forceinline__ void wv_qr_pair(const double (&a)[KR][WV_PW], const double (&v0)[WV_PW],
                                           const double (&T)[WV_PW][WV_PW], double (&b0)[KR], double (&b1)[KR],
                                           wv_rsrc w0, wv_rsrc w1, int lane)
{
    double p[2 * WV_PW];
#pragma unroll
    for (int c = 0; c < WV_PW; c++) {
        double a0 = v0[c] * b0[0], a1 = v0[c] * b1[0];
#pragma unroll
        for (int k = 1; k < KR; k++) {
            a0 = fma(a[k][c], b0[k], a0);
            a1 = fma(a[k][c], b1[k], a1);
        }
        p[c] = a0;
        p[c + WV_PW] = a1;
    }
    const double red = wrsN<2 * WV_PW>(p);
    double w0v[WV_PW], w1v[WV_PW];
    {
        double d0[WV_PW], d1[WV_PW];
#pragma unroll
        for (int c = 0; c < WV_PW; c++) {
            d0[c] = rdlane(red, (32 / WV_PW) * c);
            d1[c] = rdlane(red, (32 / WV_PW) * (c + WV_PW));
        }
#pragma unroll
        for (int c = 0; c < WV_PW; c++) {
            double x0 = 0.0, x1 = 0.0;
#pragma unroll
            for (int q = 0; q <= c; q++) {
                x0 = fma(T[q][c], d0[q], x0);
                x1 = fma(T[q][c], d1[q], x1);
            }
            w0v[c] = x0;
            w1v[c] = x1;
        }
    }
    {
        double x0 = b0[0], x1 = b1[0];
#pragma unroll
        for (int c = 0; c < WV_PW; c++) {
            x0 = fma(-v0[c], w0v[c], x0);
            x1 = fma(-v0[c], w1v[c], x1);
        }
        b0[0] = x0;
        b1[0] = x1;
    }
#pragma unroll
    for (int k = 1; k < KR; k++) {
        double x0 = b0[k], x1 = b1[k];
#pragma unroll
        for (int c = 0; c < WV_PW; c++) {
            x0 = fma(-a[k][c], w0v[c], x0);
            x1 = fma(-a[k][c], w1v[c], x1);
        }
        b0[k] = x0;
        b1[k] = x1;
    }
    wv_st_col(b0, w0, lane);
    wv_st_col(b1, w1, lane);
}

// R factor of the NB x s stack (NB <= 64 KR; s <= SM <= 64, so pivot row j is on
// lane j of the first row block).  Panels of WV_PW columns live in registers,
// trailing columns stream through W in pairs: the pair after the current
// one is loaded while the current one is updated (two register sets used in
// turn, so no load is waited for before its use), and a panel's first pair
// is loaded before the panel is factored.  R (row-major, ld WV_SMAX, zeros
// below the diagonal) is written to Rout.
template <int SM, int KR>
__device__ __forceinline__ void wv_geqrf_r(int s, const double *src0, const double *src1, int c0, double *W, int NB,
                                           double *Rout)
{
    const int lane = threadIdx.x & 63;
    const WvRs A{src0, src1, W, c0, NB};
    for (int j0 = 0; j0 < s; j0 += WV_PW) {
        const int jb = min(WV_PW, s - j0);
        const bool first = (j0 == 0);
        double a[KR][WV_PW];
#pragma unroll
        for (int c = 0; c < WV_PW; c++) {
            const wv_rsrc r = A.rd(j0 + c, first, c < jb);
#pragma unroll
            for (int k = 0; k < KR; k++) a[k][c] = wv_ld(r, (lane + 64 * k) * 8);
        }
        const int t0 = j0 + jb;
        double p0[KR], p1[KR], q0[KR], q1[KR];
        wv_ld_col(p0, A.rd(t0, first, t0 < s), lane);
        wv_ld_col(p1, A.rd(t0 + 1, first, t0 + 1 < s), lane);
        double T[WV_PW][WV_PW];
#pragma unroll
        for (int r = 0; r < WV_PW; r++)
#pragma unroll
            for (int c = 0; c < WV_PW; c++) T[r][c] = 0.0;
        // ---- panel factorization ----
#pragma unroll
        for (int jj = 0; jj < WV_PW; jj++) {
            if (jj < jb) {
                const int j = j0 + jj;
                // x = column jj; y = its part strictly below the pivot row j
                const double x0 = a[0][jj];
                const double y0 = (lane > j) ? x0 : 0.0;
                double p[WV_PW];
#pragma unroll
                for (int c = 0; c < WV_PW; c++) p[c] = y0 * (c == jj ? y0 : a[0][c]);
#pragma unroll
                for (int k = 1; k < KR; k++)
#pragma unroll
                    for (int c = 0; c < WV_PW; c++) p[c] = fma(a[k][jj], a[k][c], p[c]);
                const double red = wrsN<WV_PW>(p);
                double S[WV_PW], prow[WV_PW];
#pragma unroll
                for (int c = 0; c < WV_PW; c++) {
                    S[c] = rdlane(red, (64 / WV_PW) * c);
                    prow[c] = rdlane(a[0][c], j);
                }
                const double alpha = prow[jj], xn2 = S[jj];
                double tau = 0.0, beta = alpha, scal = 0.0;
                if (xn2 > 0.0) {
                    beta = -copysign(sqrt(alpha * alpha + xn2), alpha);
                    tau = (beta - alpha) / beta;
                    scal = 1.0 / (alpha - beta);
                }
                // reflector v in place of column jj: 1 at the pivot, y * scal below
                a[0][jj] = (lane == j) ? 1.0 : y0 * scal;
#pragma unroll
                for (int k = 1; k < KR; k++) a[k][jj] *= scal;
#pragma unroll
                for (int c = 0; c < WV_PW; c++) {
                    if (c > jj) {
                        const double td = tau * (prow[c] + S[c] * scal);  // tau * v^T a_c
#pragma unroll
                        for (int k = 0; k < KR; k++) a[k][c] = fma(-td, a[k][jj], a[k][c]);
                    }
                }
                // row block 0 of column jj: beta at the pivot, R entries above it
                a[0][jj] = (lane == j) ? beta : ((lane > j) ? a[0][jj] : x0);
                // T(0:jj, jj) = -tau T(0:jj, 0:jj) w,  w_q = v_q^T v_jj = prow[q] + S[q] * scal
#pragma unroll
                for (int l = 0; l < WV_PW; l++) {
                    if (l < jj) {
                        double acc = 0.0;
#pragma unroll
                        for (int q = 0; q < WV_PW; q++)
                            if (q >= l && q < jj) acc = fma(T[l][q], prow[q] + S[q] * scal, acc);
                        T[l][jj] = -tau * acc;
                    }
                }
                T[jj][jj] = tau;
            }
        }
        // R entries of the panel columns: rows <= j0 + c on lanes of row block 0
#pragma unroll
        for (int c = 0; c < WV_PW; c++)
            if (c < jb && lane < s) Rout[lane * SM + j0 + c] = (lane <= j0 + c) ? a[0][c] : 0.0;
        // reflector entries of row block 0: 1 at the pivot, 0 above
        double v0[WV_PW];
#pragma unroll
        for (int c = 0; c < WV_PW; c++)
            v0[c] = (c < jb) ? ((lane == j0 + c) ? 1.0 : (lane > j0 + c ? a[0][c] : 0.0)) : 0.0;
        // ---- trailing pairs: (t, t + 1) in p while (t + 2, t + 3) loads into q,
        //      then the roles swap ----
        for (int t = t0; t < s; t += 4) {
            wv_ld_col(q0, A.rd(t + 2, first, t + 2 < s), lane);
            wv_ld_col(q1, A.rd(t + 3, first, t + 3 < s), lane);
            wv_qr_pair(a, v0, T, p0, p1, A.wr(t, true), A.wr(t + 1, t + 1 < s), lane);
            if (t + 2 >= s) break;
            wv_ld_col(p0, A.rd(t + 4, first, t + 4 < s), lane);
            wv_ld_col(p1, A.rd(t + 5, first, t + 5 < s), lane);
            wv_qr_pair(a, v0, T, q0, q1, A.wr(t + 2, true), A.wr(t + 3, t + 3 < s), lane);
        }
    }
}

// Lane q holds column q of the s x s matrix M in x (zero beyond s): R of the
// Householder QR of M in place (rows i <= q; below is rounding noise).  Column j
// reaches the other lanes by readlane, every lane forms its own column's product
// with the reflector: no cross-lane sum.
template <int SM>
__device__ __forceinline__ void wv_qr_cols(double (&x)[SM], int s)
{
#pragma unroll
    for (int c = 0; c < SM; c += 8) {
        const int je = min(8, s - 1 - c);  // the last column needs no reflector
#pragma unroll 1
        for (int jj = 0; jj < je; jj++) {
            const int j = c + jj;
            double d4[4] = {0.0, 0.0, 0.0, 0.0}, xj = 0.0;
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const double v = rdlane(x[c + u], j);
                d4[u & 3] = fma(u >= jj ? v : 0.0, x[c + u], d4[u & 3]);
                xj = u == jj ? x[c + u] : xj;
            }
#pragma unroll
            for (int i8 = c + 8; i8 < SM; i8 += 8)
                if (i8 < s) {
#pragma unroll
                    for (int i = i8; i < i8 + 8; i++) d4[i & 3] = fma(rdlane(x[i], j), x[i], d4[i & 3]);
                    __builtin_amdgcn_sched_barrier(0);  // 8 values in scalar registers at a time
                }
            const double d = (d4[0] + d4[1]) + (d4[2] + d4[3]);
            const double alpha = rdlane(xj, j), nrm2 = rdlane(d, j);
            if (nrm2 > 1e-290) {
                // w = x_j with alpha - beta at row j;  H = I - w w^T / (nrm2 - alpha beta)
                const double beta = -copysign(sqrt(nrm2), alpha);
                const double g = (d - beta * xj) / (nrm2 - alpha * beta);
#pragma unroll
                for (int u = 0; u < 8; u++) {
                    const double v = rdlane(x[c + u], j);
                    x[c + u] = fma(u > jj ? -v : (u == jj ? beta - alpha : 0.0), g, x[c + u]);
                }
#pragma unroll
                for (int i8 = c + 8; i8 < SM; i8 += 8)
                    if (i8 < s) {
#pragma unroll
                        for (int i = i8; i < i8 + 8; i++) x[i] = fma(-rdlane(x[i], j), g, x[i]);
                        __builtin_amdgcn_sched_barrier(0);
                    }
            }
        }
    }
}

// One-sided Jacobi on the rows of R (lane r owns row r in xm, zero beyond s),
// round-robin pairs; a lane reads its partner's row with ds_bpermute (no LDS
// storage, no wave barrier).  Loops cover the first W entries (W >= s); f2 =
// ||R||_F^2.  Counts a run out of sweeps in *unconv.
template <int SM, int W>
__device__ __forceinline__ void wv_jacobi(double (&xm)[SM], int s, double f2, double acc, int fixed_rk, int *unconv)
{
    const int lane = threadIdx.x & 63;
    const double tol = 4.0e-16 * sqrt((double)s);
    // A pair is left alone when its smaller row is below the
    // rounding-noise floor (2.3e-16 s)^2 ||M||_F^2, or, when truncating
    // at acc, below (1e-3 acc)^2: such rows stay below the
    // truncation threshold (all of them together hold less than
    // 0.012 acc of energy) and rotating them moves a kept row by
    // less than one rounding of its norm.  A sweep pairs only the rows
    // above the floor (the others never change again).
    const double nz = wv_skip_floor(f2, s, acc, fixed_rk);
    int sweep = 0;
    for (; sweep < BLK_JACOBI_SWEEPS; sweep++) {
        double al = 0.0;  // exact norms once per sweep
#pragma unroll
        for (int q = 0; q < W; q++) al = fma(xm[q], xm[q], al);
        const bool act = lane < s && !(al <= nz);
        const unsigned long long am = __ballot(act);
        const int na = __popcll(am), npad = na + (na & 1);
        const int idx = __builtin_amdgcn_mbcnt_hi((unsigned)(am >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)am, 0));
        // row of the i-th active one, on lane i
        const int row = __builtin_amdgcn_ds_permute(4 * (act ? idx : na + lane - idx), lane);
        int rot_any = 0;
        int pos = idx;  // row at position p in round r: ((p - 1 + r) mod (npad - 1)) + 1
        for (int r = 0; r < npad - 1; r++) {
            const int pp = npad - 1 - pos;
            int pc = 0;
            if (pp != 0) {
                pc = pp + r;
                if (pc > npad - 1) pc -= npad - 1;
            }
            const int src = 4 * __builtin_amdgcn_ds_bpermute(4 * pc, row);
            double yv[W];
#pragma unroll
            for (int q = 0; q < W; q++) yv[q] = wv_bperm(src, xm[q]);
            const double be = wv_bperm(src, al);
            if (act && pc < na) {
                double g4[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int q = 0; q < W; q++) g4[q & 3] = fma(xm[q], yv[q], g4[q & 3]);
                const double ga = (g4[0] + g4[1]) + (g4[2] + g4[3]);
                const bool lo_ = idx < pc;
                double cs, sn;
                if (fmin(al, be) > nz && jacobi_rot(lo_ ? al : be, lo_ ? be : al, ga, tol, cs, sn)) {
                    rot_any = 1;
                    const double ss = lo_ ? -sn : sn;
#pragma unroll
                    for (int q = 0; q < W; q++) xm[q] = fma(ss, yv[q], cs * xm[q]);
                    // squared norm after the rotation
                    al = lo_ ? (cs * cs * al - 2.0 * cs * sn * ga + sn * sn * be)
                             : (sn * sn * be + 2.0 * cs * sn * ga + cs * cs * al);
                }
            }
            // next round: every row but the first moves one position down
            if (idx > 0) pos = (pos == 1) ? npad - 1 : pos - 1;
        }
        if (__ballot(rot_any) == 0) break;
    }
    if (sweep >= BLK_JACOBI_SWEEPS && lane == 0) atomicAdd(unconv, 1);
}

// The update of tile (m, n) = k + 1 + (hi, lo) of the packed triangle's entry e;
// L: the wave's LDS, Wq: its workspace.
template <int SM, int KR>
__device__ __forceinline__ void rc_wave_task(const TLR &t, int k, int e, double *Wq, double *L, int *redo, int *nredo,
                                             double acc, int fixed_rk, int maxrank, const OpLog &o, int *ovf,
                                             const double *qn_dense)
{
    using Cf = WvCfg<SM>;
    // opaque here, so that masks and offsets of one class are not kept live
    // across the task loop (they would take the registers of all)
    int lane = threadIdx.x & 63, NB = t.NB;
    asm volatile("" : "+v"(lane));
    asm volatile("" : "+s"(NB));
    double *sg = L + Cf::SIG;
    const int NT = t.NT;
    double *Qn = Wq + (size_t)NB * SM;
    double *Out = Qn + (size_t)NB * SM;
    double *Rp = Out + (size_t)NB * 2 * SM;
    double *Rq = Rp + SM * SM;
    double *Ku = Rq + SM * SM;
    int hi, lo;
    tri_decode(e, hi, lo);
    const int m = uni(k + 1 + hi), n = uni(k + 1 + lo);
    const bool bdense = (n - k < t.band_size);
    const int ra = uni(*rank_at(t, m, k)), rc = uni(*rank_at(t, m, n)), rb = bdense ? 0 : uni(*rank_at(t, n, k));
    const int s = rc + ra;
    const double *Au = lr_tile(t, m, k), *Av = Au + (size_t)NB * ra;
    const double *Bu = bdense ? Au : lr_tile(t, n, k), *Bv = Bu + (size_t)NB * rb;
    double *C = lr_tile(t, m, n);
    // Q's second block: formed below, or precomputed for a dense B
    const double *Qs = bdense ? qn_dense + qn_slot(NT, NB, k, m, n) : Qn;

    // ---- X = Av^T Bv (ra x rb) on the matrix cores: 16x16 tiles of X,
    //      k runs over the NB rows four at a time ----
    if (!bdense) {
        const int i16 = lane & 15, k4 = lane >> 4;
        constexpr int TT = SM / 16, U = SM <= 32 ? 4 : (SM <= 48 ? 2 : 4);
        wv_d4 xacc[TT][TT];
#pragma unroll
        for (int ta = 0; ta < TT; ta++)
#pragma unroll
            for (int tb = 0; tb < TT; tb++) xacc[ta][tb] = wv_d4{0.0, 0.0, 0.0, 0.0};
        // rows r0 .. r0 + 4U - 1 of Av's and Bv's columns by buffer loads;
        // out-of-range lanes read 0 (no branch, no select)
        const wv_rsrc ar = wv_col_rsrc(Av, ra * NB * 8), br = wv_col_rsrc(Bv, rb * NB * 8);
        auto ldx = [&](double (&av)[U][TT], double (&bv)[U][TT], int r0) {
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int row = r0 + 4 * u + k4;
#pragma unroll
                for (int tt = 0; tt < TT; tt++) {
                    const int a = 16 * tt + i16;
                    av[u][tt] = wv_ld(ar, (a < ra && row < NB) ? (row + a * NB) * 8 : WV_OOB);
                    bv[u][tt] = wv_ld(br, (a < rb && row < NB) ? (row + a * NB) * 8 : WV_OOB);
                }
            }
        };
        auto mulx = [&](const double (&av)[U][TT], const double (&bv)[U][TT]) {
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int ta = 0; ta < TT; ta++)
                    if (16 * ta < ra) {
#pragma unroll
                        for (int tb = 0; tb < TT; tb++)
                            if (16 * tb < rb) xacc[ta][tb] = mfma16(av[u][ta], bv[u][tb], xacc[ta][tb]);
                    }
        };
        if constexpr (SM <= 48) {
            // two register sets in turn: rows of the next step load
            // while the current ones multiply
            double av0[U][TT], bv0[U][TT], av1[U][TT], bv1[U][TT];
            ldx(av0, bv0, 0);
#pragma unroll 1
            for (int r0 = 0; r0 < NB; r0 += 8 * U) {
                if (r0 + 4 * U < NB) ldx(av1, bv1, r0 + 4 * U);
                mulx(av0, bv0);
                if (r0 + 4 * U >= NB) break;
                if (r0 + 8 * U < NB) ldx(av0, bv0, r0 + 8 * U);
                mulx(av1, bv1);
            }
        } else {  // one set (the registers of the widest class are taken)
#pragma unroll 1
            for (int r0 = 0; r0 < NB; r0 += 4 * U) {
                double av[U][TT], bv[U][TT];
                ldx(av, bv, r0);
                mulx(av, bv);
            }
        }
        // X^T into LDS as Xl[b * SM + a], zero outside ra x rb
        double *Xl = L;
        for (int q = lane; q < SM * SM; q += 64) Xl[q] = 0.0;
        wv_sync();
#pragma unroll
        for (int ta = 0; ta < TT; ta++)
#pragma unroll
            for (int tb = 0; tb < TT; tb++)
                if (16 * ta < ra && 16 * tb < rb) {
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const int a = 16 * ta + k4 + 4 * r, bb = 16 * tb + i16;
                        if (a < ra && bb < rb) Xl[bb * SM + a] = xacc[ta][tb][r];
                    }
                }
        wv_sync();
    }
    // ---- Qn = -Bu X^T (NB x ra): K = X^T, K[b][a] = Xl[b * SM + a] ----
    if (!bdense) wv_tall_mm<SM>(NB, rb, ra, -1.0, WvSrc{Bu, rb, Bu, NB}, L, SM, Qn);
    wv_sync();
    // ---- R factors of P = [Cu Au] and Q = [Cv Qn] ----
    for (int side = 0; side < 2; side++) {
        wv_geqrf_r<SM, KR>(s, side ? C + (size_t)NB * rc : C, side ? Qs : Au, rc, Wq, NB, side ? Rq : Rp);
    }
    wv_sync();
    // ---- columns of M = Rp Rq^T: lane q holds M(:, q) ----
    double xm[SM];
    {
        for (int q = lane; q < s * SM; q += 64) {
            const int l = q / SM, c = q - l * SM;
            L[q] = (c < s) ? Rp[c * SM + l] : 0.0;  // L[l][c] = Rp(c, l)
        }
        wv_sync();
#pragma unroll
        for (int q = 0; q < SM; q++) xm[q] = 0.0;
        // this lane's row of Rq, 16 entries per batch of loads
        const wv_rsrc rqr = wv_col_rsrc(Rq, SM * SM * 8);
        for (int l0 = 0; l0 < s; l0 += 16) {
            double rv[16];
#pragma unroll
            for (int u = 0; u < 16; u++) {
                const int l = l0 + u;
                rv[u] = wv_ld(rqr, (lane < s && l < s && l >= lane) ? (lane * SM + l) * 8 : WV_OOB);
            }
#pragma unroll
            for (int u = 0; u < 16; u++)
                if (l0 + u < s) {
                    const double *rp = L + (l0 + u) * SM;
#pragma unroll
                    for (int q8 = 0; q8 < SM; q8 += 8)
                        if (q8 < s) {
#pragma unroll
                            for (int q = q8; q < q8 + 8; q++) xm[q] = fma(rv[u], rp[q], xm[q]);
                        }
                }
        }
        wv_sync();
    }
    // ---- M = Q1 R, rows of R to the lanes, one-sided Jacobi on them: R^T J =
    //      Vs S.  Loops run over SM - 8 entries when s fits in them (entries
    //      beyond s are zero, so the width changes no bit) ----
    double f2 = 0.0;
#pragma unroll
    for (int q = 0; q < SM; q++) f2 = fma(xm[q], xm[q], f2);
    f2 = wsum(f2);
    const double fro = sqrt(f2);
    wv_qr_cols<SM>(xm, s);
#pragma unroll
    for (int q = 0; q < SM; q++)
        if (q < s && lane < s) L[q * Cf::LDJ + lane] = q <= lane ? xm[q] : 0.0;
    wv_sync();
#pragma unroll
    for (int q = 0; q < SM; q++) xm[q] = (lane < s && q < s) ? L[lane * Cf::LDJ + q] : 0.0;
    wv_sync();
    if constexpr (SM <= 48) {
        constexpr int WJ = SM - 8;
        if (s <= WJ) wv_jacobi<SM, WJ>(xm, s, f2, acc, fixed_rk, o.unconv);
        else wv_jacobi<SM, SM>(xm, s, f2, acc, fixed_rk, o.unconv);
    } else {  // one width: a second copy costs the widest class registers
        wv_jacobi<SM, SM>(xm, s, f2, acc, fixed_rk, o.unconv);
    }
    // ---- singular values, order, rank ----
    double sig = 0.0;
#pragma unroll
    for (int q = 0; q < SM; q++) sig = fma(xm[q], xm[q], sig);
    sig = sqrt(sig);
    if (lane < s) sg[lane] = sig;
    wv_sync();
    int pos = 0;
    for (int q = 0; q < s; q++) {
        const double o2 = sg[q];
        pos += (o2 > sig) || (o2 == sig && q < lane);
    }
    int nr;
    if (fixed_rk > 0) nr = fixed_rk < s ? fixed_rk : s;
    else nr = __popcll(__ballot(lane < s && sig >= acc));
    if (nr > maxrank) {
        if (lane == 0) atomicAdd(ovf, 1);
        nr = maxrank;
    }
    nr = uni(nr);
    wv_sync();
    if (nr > 0) {
        // Vs_r into LDS, row-major: Vl[l * SM + pos]; sigma by position
        double *Vl = L;
        double *sgp = sg + SM;
        if (lane < s && pos < nr) {
            const double inv = sig > 0.0 ? 1.0 / sig : 0.0;
#pragma unroll
            for (int q = 0; q < SM; q++)
                if (q < s) Vl[q * SM + pos] = xm[q] * inv;
            sgp[pos] = sig;
        }
        wv_sync();
        // Ku = Rq^T Vs_r: lane c computes row c -> Ku[c * SM + j]
        {
            double ac[SM];
#pragma unroll
            for (int j = 0; j < SM; j++) ac[j] = 0.0;
            // column `lane` of Rq, 16 entries per batch of loads
            const wv_rsrc rqr = wv_col_rsrc(Rq, SM * SM * 8);
            for (int l0 = 0; l0 < s; l0 += 16) {
                double rv[16];
#pragma unroll
                for (int u = 0; u < 16; u++) {
                    const int l = l0 + u;
                    rv[u] = wv_ld(rqr, (lane < s && l < s && l <= lane) ? (l * SM + lane) * 8 : WV_OOB);
                }
#pragma unroll
                for (int u = 0; u < 16; u++)
                    if (l0 + u < s) {
                        const double *vr = Vl + (l0 + u) * SM;
#pragma unroll
                        for (int j8 = 0; j8 < SM; j8 += 8)
                            if (j8 < nr) {
#pragma unroll
                                for (int j = j8; j < j8 + 8; j++) ac[j] = fma(rv[u], vr[j], ac[j]);
                            }
                    }
            }
            if (lane < s) {
#pragma unroll
                for (int j = 0; j < SM; j++)
                    if (j < nr) Ku[lane * SM + j] = ac[j];
            }
        }
        wv_sync();
        // Kv = Rq^-1 Vs_r in place (lane j solves column j) by plain back
        // substitution.  Q Kv = Qq Vs_r for any Kv with Rq Kv = Vs_r, and
        // the substitution is backward stable, so the tiny pivots of a
        // numerically rank-deficient Q are divided by, not dropped (dropping
        // one breaks the solve when its row carries other entries).  Column
        // j then errs in the tile by at most
        // sigma_j s eps max_q sum_l |Rq(q,l)| |Kv(l,j)|; a task over the
        // tolerance, or with an exactly zero pivot, is left untouched and
        // handed to the Householder path (k_rc_big).
        // Row q of Rq is loaded across the lanes (lane l: Rq(q, l), one
        // load per row, the next row's issued ahead) and read by readlane.
        bool bad = false;
        {
            const wv_rsrc rqr = wv_col_rsrc(Rq, SM * SM * 8);
            double gmax = 0.0;
            double rnext = wv_ld(rqr, (lane < s) ? ((s - 1) * SM + lane) * 8 : WV_OOB);
            for (int q = s - 1; q >= 0; q--) {
                const double rrow = rnext;
                rnext = wv_ld(rqr, (q > 0 && lane < s) ? ((q - 1) * SM + lane) * 8 : WV_OOB);
                double v = Vl[q * SM + lane], gq = 0.0;
                for (int l = q + 1; l < s; l++) {
                    const double rql = rdlane(rrow, l), xl = Vl[l * SM + lane];
                    v = fma(-rql, xl, v);
                    gq = fma(fabs(rql), fabs(xl), gq);
                }
                const double d = rdlane(rrow, q);
                const bool ok = fabs(d) > 1e-300;
                const double x = ok ? v / d : 0.0;
                bad = bad || !ok;
                gmax = fmax(gmax, fma(fabs(d), fabs(x), gq));
                if (lane < nr) Vl[q * SM + lane] = x;
            }
            bad = lane < nr && (bad || !(sgp[lane] * s * 2.3e-16 * gmax <= rc_solve_tol(acc, fixed_rk, fro)));
        }
        if (__ballot(bad) != 0) {
            if (lane == 0) redo[atomicAdd(nredo, 1)] = e;
            wv_sync();
            return;
        }
        wv_sync();
        // ---- outputs, written in place into the tile.  A product reads a
        //      batch of rows of all its sources before writing those rows,
        //      and every column of the tile has stride NB, so an output
        //      may overwrite its own sources.  The two products are
        //      ordered so that neither overwrites the other's sources:
        //      U' = P Ku (columns 0 .. nr-1, sources Cu = columns
        //      0 .. rc-1) and V' = Q Kv (columns nr .. 2nr-1, sources
        //      Cv = columns rc .. 2rc-1): U' first when nr <= rc, V'
        //      first otherwise. ----
        auto v_out = [&]() {  // Kv in LDS
            wv_tall_mm<SM>(NB, s, nr, 1.0, WvSrc{C + (size_t)rc * NB, rc, Qs, NB}, Vl, SM, C + (size_t)nr * NB);
            wv_sync();
        };
        auto u_out = [&]() {  // stages Ku into LDS
            for (int q = lane; q < s * SM; q += 64) {
                const int c = q / SM, j = q - c * SM;
                Vl[q] = (j < nr) ? Ku[c * SM + j] : 0.0;
            }
            wv_sync();
            wv_tall_mm<SM>(NB, s, nr, 1.0, WvSrc{C, rc, Au, NB}, Vl, SM, C);
            wv_sync();
        };
        if (nr > rc) {
            v_out();
            u_out();
        } else {
            for (int q = lane; q < s * SM; q += 64) Out[q] = Vl[q];  // Kv aside while Ku uses the LDS
            u_out();
            for (int q = lane; q < s * SM; q += 64) Vl[q] = Out[q];
            wv_sync();
            v_out();
        }
    }
    if (lane == 0) {
        *rank_at(t, m, n) = nr;
        rank_hist(o, NT, m, n, nr);
        rc_oplog(o, t, m, n, ra, rb, rc, nr, bdense);
    }
    wv_sync();
}
