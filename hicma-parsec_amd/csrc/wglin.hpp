// wglin.hpp -- dense factorizations by one 256-thread workgroup (four waves,
// one per SIMD with the full register file): Householder QR with the panel in
// registers and the trailing update on the FP64 matrix cores, application of
// the reflectors, and a one-sided Jacobi SVD whose columns live in LDS.
// Matrices are column major in global memory (one workgroup's share stays in
// L2); every routine is called by all threads and begins and ends with its
// data visible to the workgroup.
#pragma once
#include "blk.hpp"

#define WQ_PW 16       // panel width (= QRB: one T factor of 16 x 16 per panel)
#define WQ_MAIN 18432  // doubles of the shared region: V panel, Jacobi columns, gemm staging
#define WQ_AUX 768     // T, G, tau, reduction slots
#define WQ_LDS (WQ_MAIN + WQ_AUX)
#define WQ_MAXROWS 2048  // tallest matrix (8 rows per thread)

struct WqLds {
    double *main;  // WQ_MAIN
    double *T;     // 16 x 17, row major
    double *G;     // 16 x 17: G[c + 17 j] = v_c^T v_j, c < j
    double *tau;   // 16
    double *red;   // 2 x 64
    double *prow;  // 2 x 16
};
__device__ __forceinline__ WqLds wq_lds(double *sm)
{
    double *x = sm + WQ_MAIN;
    return WqLds{sm, x, x + 272, x + 544, x + 560, x + 688};
}

// column stride of the V panel: 17 mod 32 keeps both reads of the panel
// (16 consecutive rows of 4 columns, 4 rows of 16 columns) at two bank cycles
__device__ __forceinline__ int wq_ldv(int m) { return ((m + 63) & ~63) + 17; }

// T (upper, 16 x 16) of H = I - V T V^T from G and tau, by lanes 0 .. 15 of
// wave 0: lane i forms row i.  Into S.T and Tsave (column major).
__device__ __forceinline__ void wq_build_t(int jb, const WqLds &S, double *Tsave)
{
    const int i = threadIdx.x;
    if (i < WQ_PW) {
        double tr[WQ_PW];
#pragma unroll
        for (int j = 0; j < WQ_PW; j++) {
            double v = 0.0;
            if (j < jb) {
                const double tj = S.tau[j];
                double s = 0.0;
#pragma unroll
                for (int l = 0; l < j; l++) s = fma(l >= i ? tr[l] : 0.0, S.G[l + 17 * j], s);
                v = (i == j) ? tj : (i < j ? -tj * s : 0.0);
            }
            tr[j] = v;
            S.T[i * 17 + j] = v;
            Tsave[i + WQ_PW * j] = v;
        }
    }
}

// Householder factorization of the mr x jb panel at Ap (jb <= 16, mr <= 256 R),
// thread t holding rows t, t + 256, ...: one reduction per column gives its
// norm below the pivot, the products with the panel's later columns and with
// the earlier reflectors (for T).  R entries and reflectors go back in place,
// the reflectors with explicit ones and zeros to V (ld ldv, rows padded with
// zeros to a multiple of 64), T to S.T and Tsave.
template <int R>
__device__ __forceinline__ void wq_panel(int mr, int jb, double *Ap, int lda, double *V, int ldv, double *Tsave,
                                         const WqLds &S)
{
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    double a[R][WQ_PW];
#pragma unroll
    for (int c = 0; c < WQ_PW; c++)
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int row = tid + BS * r;
            a[r][c] = (c < jb && row < mr) ? Ap[row + (size_t)c * lda] : 0.0;
        }
#pragma unroll
    for (int jj = 0; jj < WQ_PW; jj++) {
        if (jj < jb) {
            const int buf = jj & 1;
            const double x0 = a[0][jj], y0 = (tid > jj) ? x0 : 0.0;
            double p[WQ_PW];
#pragma unroll
            for (int c = 0; c < WQ_PW; c++) p[c] = y0 * a[0][c];
#pragma unroll
            for (int r = 1; r < R; r++)
#pragma unroll
                for (int c = 0; c < WQ_PW; c++) p[c] = fma(a[r][jj], a[r][c], p[c]);
            const double part = wrs16(p);
            if ((lane & 3) == 0) S.red[64 * buf + 16 * w + (lane >> 2)] = part;
            if (tid == jj) {
#pragma unroll
                for (int c = 0; c < WQ_PW; c++) S.prow[16 * buf + c] = a[0][c];
            }
            __syncthreads();
            // lanes 4c .. 4c+3: value c, one wave's part each
            double sc = S.red[64 * buf + 16 * (lane & 3) + (lane >> 2)];
            sc += dppd<DPP_XOR1>(sc);
            sc += dppd<DPP_XOR2>(sc);
            const double pr = S.prow[16 * buf + (lane >> 2)];
            const double alpha = rdlane(pr, 4 * jj), xn2 = rdlane(sc, 4 * jj);
            double tau = 0.0, beta = alpha, scal = 0.0;
            if (xn2 > 0.0) {
                beta = -copysign(sqrt(alpha * alpha + xn2), alpha);
                tau = (beta - alpha) / beta;
                scal = 1.0 / (alpha - beta);
            }
            const double wv = fma(sc, scal, pr);  // v_jj^T (column c), or v_c^T v_jj for c < jj
            if (w == 0 && (lane & 3) == 0 && (lane >> 2) < jj) S.G[(lane >> 2) + 17 * jj] = wv;
            if (tid == 0) S.tau[jj] = tau;
            const double td = tau * wv;
            const double v0 = (tid == jj) ? 1.0 : y0 * scal;
#pragma unroll
            for (int r = 1; r < R; r++) a[r][jj] *= scal;
#pragma unroll
            for (int c = jj + 1; c < WQ_PW; c++) {
                const double tc = rdlane(td, 4 * c);
                a[0][c] = fma(-tc, v0, a[0][c]);
#pragma unroll
                for (int r = 1; r < R; r++) a[r][c] = fma(-tc, a[r][jj], a[r][c]);
            }
            a[0][jj] = (tid == jj) ? beta : (tid > jj ? v0 : x0);
        }
    }
    const int mrp = (mr + 63) & ~63;
#pragma unroll
    for (int c = 0; c < WQ_PW; c++)
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int row = tid + BS * r;
            if (c < jb && row < mr) Ap[row + (size_t)c * lda] = a[r][c];
            const double v = (c < jb && row < mr) ? (row > c ? a[r][c] : (row == c ? 1.0 : 0.0)) : 0.0;
            if (row < mrp) V[c * ldv + row] = v;
        }
    __syncthreads();  // G, tau are complete
    wq_build_t(jb, S, Tsave);
    __syncthreads();  // V, T for every wave
}

// C (mr x nc) <- (I - V op(T) V^T) C, op(T) = T^T if TR else T: 16-column
// tiles of C over the waves, each one W = V^T C, op(T) W and C - V W on the
// matrix cores (the result layout of one product is the operand layout of
// the next, so W stays in registers).
template <bool TR>
__device__ __forceinline__ void wq_reflect(int mr, int nc, const double *V, int ldv, const double *T, double *C,
                                           int ldc)
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, i16 = lane & 15, k4 = lane >> 4;
    for (int c0 = 16 * w; c0 < nc; c0 += 64) {
        const wv_rsrc cr = wv_col_rsrc(C + (size_t)c0 * ldc, (min(16, nc - c0) - 1) * ldc * 8 + mr * 8);
        const bool cok = c0 + i16 < nc;
        mk_d4 w0 = mk_d4{0.0, 0.0, 0.0, 0.0}, w1 = w0;
#pragma unroll 1
        for (int r0 = 0; r0 < mr; r0 += 64) {
            double b[16];
#pragma unroll
            for (int u = 0; u < 16; u++) {
                const int row = r0 + 4 * u + k4;
                b[u] = wv_ld(cr, (cok && row < mr) ? (row + i16 * ldc) * 8 : WV_OOB);
            }
            const double *vp = V + i16 * ldv + r0 + k4;
#pragma unroll
            for (int u = 0; u < 16; u += 2) {
                w0 = mk_mfma(vp[4 * u], b[u], w0);
                w1 = mk_mfma(vp[4 * u + 4], b[u + 1], w1);
            }
        }
        mk_d4 q = mk_d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int kk = 0; kk < 4; kk++) {
            const int kr = 4 * kk + k4;
            q = mk_mfma(TR ? T[kr * 17 + i16] : T[i16 * 17 + kr], w0[kk] + w1[kk], q);
        }
#pragma unroll 1
        for (int r0 = 0; r0 < mr; r0 += 64) {
            mk_d4 x[4];
#pragma unroll
            for (int s = 0; s < 4; s++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int row = r0 + 16 * s + i16, col = 4 * e + k4;
                    x[s][e] = wv_ld(cr, (c0 + col < nc && row < mr) ? (row + col * ldc) * 8 : WV_OOB);
                }
#pragma unroll
            for (int kk = 0; kk < 4; kk++)
#pragma unroll
                for (int s = 0; s < 4; s++)
                    x[s] = mk_mfma(-q[kk], V[(4 * kk + k4) * ldv + r0 + 16 * s + i16], x[s]);
#pragma unroll
            for (int s = 0; s < 4; s++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int row = r0 + 16 * s + i16, col = 4 * e + k4;
                    wv_st(x[s][e], cr, (c0 + col < nc && row < mr) ? (row + col * ldc) * 8 : WV_OOB);
                }
        }
    }
}

// QR of A (m x n, m <= 256 R), LAPACK storage; T factor of panel p at
// Tsave + 256 p.  Vb: global room for the V panel (16 wq_ldv(m) doubles)
// when it does not fit the LDS (R > 4).
template <int R>
__device__ __forceinline__ void wq_geqrf(int m, int n, double *A, int lda, double *Tsave, double *Vb, const WqLds &S)
{
    const int kmax = m < n ? m : n;
    __syncthreads();
    for (int j0 = 0; j0 < kmax; j0 += WQ_PW) {
        const int jb = min(WQ_PW, kmax - j0), mr = m - j0, ldv = wq_ldv(mr), nt = n - j0 - jb;
        double *Ap = A + j0 + (size_t)j0 * lda, *Ts = Tsave + (size_t)(j0 / WQ_PW) * WQ_PW * WQ_PW;
        if constexpr (R <= 4) {
            wq_panel<R>(mr, jb, Ap, lda, S.main, ldv, Ts, S);
            wq_reflect<true>(mr, nt, S.main, ldv, S.T, Ap + (size_t)jb * lda, lda);
        } else {
            wq_panel<R>(mr, jb, Ap, lda, Vb, ldv, Ts, S);
            wq_reflect<true>(mr, nt, Vb, ldv, S.T, Ap + (size_t)jb * lda, lda);
        }
        __syncthreads();
    }
}

// C (m x nc) <- Q C, Q = H_0 .. H_{k-1} of wq_geqrf.  With TRI, C starts as
// the first nc columns of the identity and panel p touches columns 16 p ..
// only (nc <= k).
template <int R, bool TRI = false>
__device__ __forceinline__ void wq_apply(int m, int nc, int k, const double *A, int lda, const double *Tsave,
                                         double *C, int ldc, double *Vb, const WqLds &S)
{
    if (nc <= 0 || k <= 0) return;
    const int tid = threadIdx.x;
    double *V = R <= 4 ? S.main : Vb;
    for (int p = (k + WQ_PW - 1) / WQ_PW - 1; p >= 0; p--) {
        const int j0 = WQ_PW * p, jb = min(WQ_PW, k - j0), mr = m - j0, ldv = wq_ldv(mr), mrp = (mr + 63) & ~63;
        const double *Ap = A + j0 + (size_t)j0 * lda;
        __syncthreads();
        for (int c = 0; c < WQ_PW; c++)
            for (int row = tid; row < mrp; row += BS) {
                const double v = (c < jb && row < mr) ? (row > c ? Ap[row + (size_t)c * lda] : (row == c ? 1.0 : 0.0)) : 0.0;
                V[c * ldv + row] = v;
            }
        S.T[(tid & 15) * 17 + (tid >> 4)] = Tsave[(size_t)p * WQ_PW * WQ_PW + tid];
        __syncthreads();
        const int cs = TRI ? j0 : 0;
        if (nc > cs) {
            if constexpr (R <= 4) wq_reflect<false>(mr, nc - cs, S.main, ldv, S.T, C + j0 + (size_t)cs * ldc, ldc);
            else wq_reflect<false>(mr, nc - cs, Vb, ldv, S.T, C + j0 + (size_t)cs * ldc, ldc);
        }
    }
    __syncthreads();
}

// ---- one-sided Jacobi -----------------------------------------------------

#define WJ_ROWS 40        // rows per lane
#define WJ_SMALL2 1e-20   // squared cosine below which a rotation counts as small

// One pair by a group of G lanes (lane sub of the group holds rows sub,
// sub + G, ...; `nch` chunks of two such rows, rows past the matrix hold zeros):
// the pair is read once, rotated in registers and written back if it turned.
// Returns 0 (left alone), 1 (turned by a small angle) or 3.
template <int G>
__device__ __forceinline__ int wj_pair(double *x, double *y, int nch, int sub, double tol, double nz)
{
    double xv[WJ_ROWS], yv[WJ_ROWS], al[2] = {0.0, 0.0}, be[2] = {0.0, 0.0}, ga[2] = {0.0, 0.0};
#pragma unroll
    for (int c = 0; c < WJ_ROWS / 2; c++)
        if (c < nch) {
#pragma unroll
            for (int u = 0; u < 2; u++) {
                xv[2 * c + u] = x[sub + G * (2 * c + u)];
                yv[2 * c + u] = y[sub + G * (2 * c + u)];
            }
#pragma unroll
            for (int u = 0; u < 2; u++) {
                al[u] = fma(xv[2 * c + u], xv[2 * c + u], al[u]);
                be[u] = fma(yv[2 * c + u], yv[2 * c + u], be[u]);
                ga[u] = fma(xv[2 * c + u], yv[2 * c + u], ga[u]);
            }
        }
    const double a = gsum<G>(al[0] + al[1]), b = gsum<G>(be[0] + be[1]), g = gsum<G>(ga[0] + ga[1]);
    double cs, sn;
    if (!(fmin(a, b) > nz) || !jacobi_rot(a, b, g, tol, cs, sn)) return 0;
#pragma unroll
    for (int c = 0; c < WJ_ROWS / 2; c++)
        if (c < nch) {
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const double xo = xv[2 * c + u], yo = yv[2 * c + u];
                x[sub + G * (2 * c + u)] = cs * xo - sn * yo;
                y[sub + G * (2 * c + u)] = sn * xo + cs * yo;
            }
        }
    return g * g > WJ_SMALL2 * a * b ? 3 : 1;
}

// LDS column stride of m-row columns: multiples of 2 G rows, and columns of
// consecutive pairs start G banks apart
template <int G>
__host__ __device__ __forceinline__ int wj_ldc(int m)
{
    const int rows = (m + 2 * G - 1) / (2 * G) * (2 * G);
    return G < 32 ? rows + G : rows;
}
// whether G lanes per pair take columns of m rows: WJ_ROWS rows per lane, and
// 512 / G columns of LDS (or all n of them, when those are fewer)
template <int G>
__host__ __device__ __forceinline__ bool wj_takes(int m, int n)
{
    const int nc = 2 * BS / G, ldc = wj_ldc<G>(m);
    return (m + 2 * G - 1) / (2 * G) * 2 <= WJ_ROWS && (long)(n < nc ? n + (n & 1) : nc) * ldc <= WQ_MAIN;
}

// One-sided Jacobi on the n columns of M (m x n, ld ldm, in place): on return
// the columns are orthogonal.  Columns live in LDS, 256 / G pairs at a time.
// n <= 512 / G columns stay there throughout; otherwise the columns form
// blocks of 256 / G, and a sweep visits every pair of blocks (all pairs of
// both blocks on the first visit of each, the cross pairs afterwards),
// which moves a column once per 256 / G rotations instead of once per
// rotation.  Pairs whose smaller squared norm is <= nz are left alone.  A sweep
// whose rotations all had cosines below 1e-10 is the last one (convergence is
// quadratic, so what it leaves is below rounding).  Fixed order; returns the
// number of sweeps (BLK_JACOBI_SWEEPS: not converged).
template <int G>
__device__ __forceinline__ int wj_jacobi(int m, int n, double *M, int ldm, double nz, double *L)
{
    constexpr int NP = BS / G, NC = 2 * NP;
    const int tid = threadIdx.x, kp = tid / G, sub = tid % G;
    const int nch = (m + 2 * G - 1) / (2 * G), rows = nch * 2 * G, ldc = wj_ldc<G>(m);
    const double tol = 4.0e-16 * sqrt((double)m);
    auto move_in = [&](int c0, int g0, int nc) {  // LDS columns c0 .. c0 + nc - 1 <- columns g0 ..
        for (int c = 0; c < nc; c++)
            for (int r = tid; r < rows; r += BS)
                L[(c0 + c) * ldc + r] = (g0 + c < n && r < m) ? M[r + (size_t)(g0 + c) * ldm] : 0.0;
    };
    auto move_out = [&](int c0, int g0, int nc) {
        for (int c = 0; c < nc; c++)
            if (g0 + c < n)
                for (int r = tid; r < m; r += BS) M[r + (size_t)(g0 + c) * ldm] = L[(c0 + c) * ldc + r];
    };
    // every pair of the first nc (even) LDS columns once
    auto all_pairs = [&](int nc) {
        int any = 0;
        for (int r = 0; r < nc - 1; r++) {
            if (kp < nc / 2) {
                int ca = kp == 0 ? 0 : kp - 1 + r, cb = nc - 2 - kp + r;
                if (kp) {
                    if (ca >= nc - 1) ca -= nc - 1;
                    ca++;
                }
                if (cb >= nc - 1) cb -= nc - 1;
                cb++;
                any |= wj_pair<G>(L + ca * ldc, L + cb * ldc, nch, sub, tol, nz);
            }
            __syncthreads();
        }
        return any;
    };
    int sweep = 0;
    if (n <= NC) {
        const int ne = n + (n & 1);
        move_in(0, 0, ne);
        __syncthreads();
        for (; sweep < BLK_JACOBI_SWEEPS; sweep++)
            if (!__syncthreads_or(all_pairs(ne) & 2)) break;
        move_out(0, 0, n);
        __syncthreads();
        return sweep;
    }
    const int nb = (n + NP - 1) / NP, nbe = nb + (nb & 1);
    for (; sweep < BLK_JACOBI_SWEEPS; sweep++) {
        int any = 0;
        for (int rd = 0; rd < nbe - 1; rd++)
            for (int q = 0; q < nbe / 2; q++) {
                int ba = q == 0 ? 0 : (q - 1 + rd) % (nbe - 1) + 1, bb = (nbe - 2 - q + rd) % (nbe - 1) + 1;
                if (ba > bb) {
                    const int s = ba;
                    ba = bb;
                    bb = s;
                }
                if (bb >= nb && rd > 0) continue;  // a block without a partner: its own pairs in round 0
                move_in(0, ba * NP, NP);
                move_in(NP, bb * NP, NP);
                __syncthreads();
                int rot = 0;
                if (rd == 0) {
                    rot = all_pairs(NC);
                } else {
                    for (int r = 0; r < NP; r++) {
                        const int cb = NP + ((kp + r) & (NP - 1));
                        rot |= wj_pair<G>(L + kp * ldc, L + cb * ldc, nch, sub, tol, nz);
                        __syncthreads();
                    }
                }
                any |= rot & 2;
                if (__syncthreads_or(rot)) {
                    move_out(0, ba * NP, NP);
                    move_out(NP, bb * NP, NP);
                }
                __syncthreads();
            }
        if (!__syncthreads_or(any)) break;
    }
    return sweep;
}

// tallest matrix wj_svd takes (64 lanes per pair, 8 columns of LDS)
#define WJ_MAXN 2304
__device__ __forceinline__ int wj_svd(int m, int n, double *M, int ldm, double nz, double *L)
{
    if (n <= 1) return 0;
    if (n <= 32 && wj_takes<16>(m, n)) return wj_jacobi<16>(m, n, M, ldm, nz, L);
    if (n <= 64 && wj_takes<8>(m, n)) return wj_jacobi<8>(m, n, M, ldm, nz, L);
    if (n <= 128 && wj_takes<4>(m, n)) return wj_jacobi<4>(m, n, M, ldm, nz, L);
    if (wj_takes<8>(m, n)) return wj_jacobi<8>(m, n, M, ldm, nz, L);
    if (wj_takes<16>(m, n)) return wj_jacobi<16>(m, n, M, ldm, nz, L);
    if (wj_takes<32>(m, n)) return wj_jacobi<32>(m, n, M, ldm, nz, L);
    return wj_jacobi<64>(m, n, M, ldm, nz, L);
}

// squared Frobenius norm of M (n x n, ld ldm), the same on every thread
__device__ __forceinline__ double wq_fro2(int n, const double *M, int ldm, double *red)
{
    double s = 0.0;
    for (int c = threadIdx.x >> 6; c < n; c += NWAVE)
        for (int r = threadIdx.x & 63; r < n; r += 64) s = fma(M[r + (size_t)c * ldm], M[r + (size_t)c * ldm], s);
    return blk_sum(s, red);
}

// sig[j] = norm of column j of M (m x n), pos[j] = its rank in descending
// order (ties by index); sig and pos in LDS
__device__ __forceinline__ void wq_sigma(int m, int n, const double *M, int ldm, double *sig, int *pos)
{
    const int lane = threadIdx.x & 63;
    for (int c = threadIdx.x >> 6; c < n; c += NWAVE) {
        double s = 0.0;
        for (int r = lane; r < m; r += 64) s = fma(M[r + (size_t)c * ldm], M[r + (size_t)c * ldm], s);
        s = wsum(s);
        if (lane == 0) sig[c] = sqrt(s);
    }
    __syncthreads();
    blk_sort_pos(n, sig, pos);
}

// Right singular vectors of M (n x n, ld ldm): M = Q1 R, and one-sided Jacobi
// on the columns of R^T (the rows of R) gives R^T J = Vs S.  The rows of an
// (unpivoted) R are graded, which takes 5 .. 8 sweeps where the columns of M
// or M^T take 8 .. 22 (stacks of 44 .. 115 columns of 2-D sqexp updates), and
// the rows after the last one above the floor nz2 (a squared norm, see
// wv_skip_floor) take no part.  M is overwritten by its QR; X (n x n, ld n)
// returns Vs S in columns 0 .. n - 1 (unsorted).  Returns the sweeps.
template <int R>
__device__ __forceinline__ int wq_right_svd(int n, double *M, int ldm, double *X, double nz, double *Tsave, double *Vb,
                                            const WqLds &S)
{
    wq_geqrf<R>(n, n, M, ldm, Tsave, Vb, S);
    for (int i = threadIdx.x >> 6; i < n; i += NWAVE)
        for (int r = threadIdx.x & 63; r < n; r += 64) X[r + (size_t)i * n] = r >= i ? M[i + (size_t)r * ldm] : 0.0;
    __syncthreads();
    __shared__ int s_ke;
    if (threadIdx.x == 0) s_ke = 0;
    __syncthreads();
    for (int i = threadIdx.x >> 6; i < n; i += NWAVE) {
        double s = 0.0;
        for (int r = threadIdx.x & 63; r < n; r += 64) s = fma(X[r + (size_t)i * n], X[r + (size_t)i * n], s);
        s = wsum(s);
        if ((threadIdx.x & 63) == 0 && !(s <= nz)) atomicMax(&s_ke, i + 1);
    }
    __syncthreads();
    return wj_svd(n, s_ke, X, n, nz, S.main);
}

// dst (n x n) <- upper triangle of src, zeros below the diagonal
__device__ __forceinline__ void wq_triu(int n, const double *src, int lds, double *dst, int ldd)
{
    for (int c = threadIdx.x >> 6; c < n; c += NWAVE)
        for (int r = threadIdx.x & 63; r < n; r += 64) dst[r + (size_t)c * ldd] = r <= c ? src[r + (size_t)c * lds] : 0.0;
}
