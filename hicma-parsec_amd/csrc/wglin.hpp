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
    // the small parts first: their addresses are then immediates of the LDS instructions
    return WqLds{sm + WQ_AUX, sm, sm + 272, sm + 544, sm + 560, sm + 688};
}

// f(r, c, g(r, c)) for the rows r < rows of the columns c < nc, a thread on
// consecutive rows: eight columns' loads g are issued before the first store f,
// so that a copy costs one latency per eight columns.
template <typename Ld, typename St>
__device__ __forceinline__ void wq_cols(int rows, int nc, Ld g, St f)
{
    for (int r = threadIdx.x; r < rows; r += BS)
        for (int c = 0; c < nc; c += 8) {
            double v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = (c + u < nc) ? g(r, c + u) : 0.0;
#pragma unroll
            for (int u = 0; u < 8; u++)
                if (c + u < nc) f(r, c + u, v[u]);
        }
}

__device__ __forceinline__ void wq_copy(int rows, int nc, const double *src, int lds, double *dst, int ldd)
{
    wq_cols(
        rows, nc, [&](int r, int c) { return src[r + (size_t)c * lds]; },
        [&](int r, int c, double v) { dst[r + (size_t)c * ldd] = v; });
}

// column stride of the V panel: 17 mod 32 keeps both reads of the panel
// (16 consecutive rows of 4 columns, 4 rows of 16 columns) at two bank cycles
__device__ __forceinline__ int wq_ldv(int m) { return ((m + 63) & ~63) + 17; }

// T (upper, 16 x 16) of H = I - V T V^T from G and tau, by lanes 0 .. 15 of
// wave 0: lane i forms row i.  Into S.T and Tsave (column major).
__device__ __forceinline__ void wq_build_t(const WqLds &S, double *Tsave)
{
    int i = threadIdx.x;
    asm volatile("" : "+v"(i));
    if (i < WQ_PW) {
        double tr[WQ_PW];
#pragma unroll
        for (int j = 0; j < WQ_PW; j++) {
            const double tj = S.tau[j];
            double s = 0.0;
#pragma unroll
            for (int l = 0; l < j; l++) s = fma(l >= i ? tr[l] : 0.0, S.G[l + 17 * j], s);
            const double v = (i == j) ? tj : (i < j ? -tj * s : 0.0);
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
    // opaque, so that the comparisons with it are not hoisted out of the panel
    // loop into scalar registers that then spill
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63, w = tid >> 6;
    // columns past jb are zero throughout: they read 0, and their tau comes out 0
    const wv_rsrc ar = wv_col_rsrc(Ap, ((jb - 1) * lda + mr) * 8);
    int off[R];
#pragma unroll
    for (int r = 0; r < R; r++) off[r] = tid + BS * r < mr ? 8 * (tid + BS * r) : WV_OOB;
    double a[R][WQ_PW];
#pragma unroll
    for (int c = 0; c < WQ_PW; c++)
#pragma unroll
        for (int r = 0; r < R; r++) a[r][c] = wv_ldc(ar, off[r], c < jb ? 8 * c * lda : WV_OOB);
#pragma unroll
    for (int jj = 0; jj < WQ_PW; jj++) {
        {
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
            wv_stc(a[r][c], ar, off[r], c < jb ? 8 * c * lda : WV_OOB);
            if (row < mrp) V[c * ldv + row] = row > c ? a[r][c] : (row == c ? 1.0 : 0.0);
        }
    __syncthreads();  // G, tau are complete
    wq_build_t(S, Tsave);
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
        wq_cols(
            mrp, WQ_PW, [&](int r, int c) { return (c < jb && r < mr && r > c) ? Ap[r + (size_t)c * lda] : 0.0; },
            [&](int r, int c, double v) { V[c * ldv + r] = (r == c && c < jb) ? 1.0 : v; });
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

// jacobi_rot by the hardware's approximate roots: the angle's relative error
// (2^-23) only leaves that part of the inner product for the next sweep, and
// c = (1 + t^2)^-1/2 gets one third-order step, so c^2 + s^2 = 1 to rounding.
// 14 dependent instructions instead of some 50.
__device__ __forceinline__ bool wj_rotation(double al, double be, double ga, double tol, double &c, double &s)
{
    if (ga == 0.0 || !(ga * ga > (tol * tol) * (al * be))) return false;
    const double diff = be - al, g2 = 2.0 * ga, h = fma(diff, diff, g2 * g2);
    const double den = fabs(diff) + h * __builtin_amdgcn_rsq(h);
    if (!(den > 0.0)) return false;
    const double t = (diff >= 0.0 ? g2 : -g2) * __builtin_amdgcn_rcp(den);
    const double u = fma(t, t, 1.0), r = __builtin_amdgcn_rsq(u), e = fma(-u * r, r, 1.0);
    c = fma(r * e, fma(0.375, e, 0.5), r);
    s = c * t;
    return true;
}

#define WJ_ROWS 40        // rows per lane
#define WJ_SMALL2 1e-20   // squared cosine below which a rotation counts as small

// One pair by a group of G lanes (lane sub of the group holds rows sub,
// sub + G, ...; `nch` chunks of four such rows, rows past the matrix hold zeros):
// the pair is read once, rotated in registers and written back if it turned.
// Returns 0 (left alone), 1 (turned by a small angle) or 3.
template <int G>
__device__ __forceinline__ int wj_pair(double *x, double *y, int nch, int sub, double tol, double nz)
{
    asm volatile("" : "+s"(nch));  // no hoisted comparison per chunk
    constexpr int CH = 4;          // rows per chunk
    double xv[WJ_ROWS], yv[WJ_ROWS], al[2] = {0.0, 0.0}, be[2] = {0.0, 0.0}, ga[2] = {0.0, 0.0};
    // every load first, then the products, so that the loads' latencies overlap
#pragma unroll
    for (int c = 0; c < WJ_ROWS / CH; c++)
        if (c < nch) {
#pragma unroll
            for (int u = 0; u < CH; u++) {
                xv[CH * c + u] = x[sub + G * (CH * c + u)];
                yv[CH * c + u] = y[sub + G * (CH * c + u)];
            }
        }
#pragma unroll
    for (int c = 0; c < WJ_ROWS / CH; c++)
        if (c < nch) {
#pragma unroll
            for (int u = 0; u < CH; u++) {
                al[u & 1] = fma(xv[CH * c + u], xv[CH * c + u], al[u & 1]);
                be[u & 1] = fma(yv[CH * c + u], yv[CH * c + u], be[u & 1]);
                ga[u & 1] = fma(xv[CH * c + u], yv[CH * c + u], ga[u & 1]);
            }
        }
    const double a = gsum<G>(al[0] + al[1]), b = gsum<G>(be[0] + be[1]), g = gsum<G>(ga[0] + ga[1]);
    double cs, sn;
    if (!(fmin(a, b) > nz) || !wj_rotation(a, b, g, tol, cs, sn)) return 0;
#pragma unroll
    for (int c = 0; c < WJ_ROWS / CH; c++)
        if (c < nch) {
#pragma unroll
            for (int u = 0; u < CH; u++) {
                const double xo = xv[CH * c + u], yo = yv[CH * c + u];
                x[sub + G * (CH * c + u)] = cs * xo - sn * yo;
                y[sub + G * (CH * c + u)] = sn * xo + cs * yo;
            }
        }
    return g * g > WJ_SMALL2 * a * b ? 3 : 1;
}

// LDS column stride of m-row columns: multiples of 4 G rows, and columns of
// consecutive pairs start G banks apart
template <int G>
__host__ __device__ __forceinline__ int wj_ldc(int m)
{
    const int rows = (m + 4 * G - 1) / (4 * G) * (4 * G);
    return G < 32 ? rows + G : rows;
}
// whether G lanes per pair take columns of m rows: WJ_ROWS rows per lane, and
// 512 / G columns of LDS (or all n of them, when those are fewer)
template <int G>
__host__ __device__ __forceinline__ bool wj_takes(int m, int n)
{
    const int nc = 2 * BS / G, ldc = wj_ldc<G>(m);
    return (m + 4 * G - 1) / (4 * G) * 4 <= WJ_ROWS && (long)(n < nc ? n + (n & 1) : nc) * ldc <= WQ_MAIN;
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
    const int nch = (m + 4 * G - 1) / (4 * G), rows = nch * 4 * G, ldc = wj_ldc<G>(m);
    const double tol = 4.0e-16 * sqrt((double)m);
    auto move_in = [&](int c0, int g0, int nc) {  // LDS columns c0 .. c0 + nc - 1 <- columns g0 ..
        wq_cols(
            rows, nc, [&](int r, int c) { return (g0 + c < n && r < m) ? M[r + (size_t)(g0 + c) * ldm] : 0.0; },
            [&](int r, int c, double v) { L[(c0 + c) * ldc + r] = v; });
    };
    auto move_out = [&](int c0, int g0, int nc) {
        wq_cols(
            m, min(nc, n - g0), [&](int r, int c) { return L[(c0 + c) * ldc + r]; },
            [&](int r, int c, double v) { M[r + (size_t)(g0 + c) * ldm] = v; });
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

// ---- the same with 4 x 4 column blocks per group --------------------------
// A group of G lanes holds eight columns (two blocks of four) in registers
// and turns all pairs across the blocks, four independent rotations at a time, so
// a column crosses the LDS once per four rotations (one per rotation bounds
// wj_jacobi: 16 bytes per row each way at about 64 bytes per cycle).  The four
// inner products are reduce-scattered over the lanes of each quad, lane j
// (mod 4) computes rotation j, and DPP gives every lane all four.
// What bounds it: the chain of dependent instructions of a step (one wave per SIMD,
// about 350 instructions of 3.4 ns a step).  One workgroup per matrix, N=2700
// tile 270 band 1: 33 -> 27 ms against wj_jacobi; 28 sketches of 266 columns
// 43 -> 33 ms, of 160 13 -> 9 ms.

#define WJ4_ROWS 10  // rows per lane

__device__ __forceinline__ double wj_quad(double v, int j)
{
    switch (j) {
    case 0: return dppd<0x00>(v);  // quad_perm [j, j, j, j]
    case 1: return dppd<0x55>(v);
    case 2: return dppd<0xAA>(v);
    default: return dppd<0xFF>(v);
    }
}

// Four independent rotations (u_j, v_j); nu, nv: squared norms, the same on
// every lane.  nch chunks of two rows.  Returns as wj_pair.
template <int G>
__device__ __forceinline__ int wj_rot4(double (&u0)[WJ4_ROWS], double (&v0)[WJ4_ROWS], double (&u1)[WJ4_ROWS],
                                       double (&v1)[WJ4_ROWS], double (&u2)[WJ4_ROWS], double (&v2)[WJ4_ROWS],
                                       double (&u3)[WJ4_ROWS], double (&v3)[WJ4_ROWS], double &nu0, double &nv0,
                                       double &nu1, double &nv1, double &nu2, double &nv2, double &nu3, double &nv3,
                                       int nch, int sub, double tol, double nz)
{
    double p0 = 0.0, p1 = 0.0, p2 = 0.0, p3 = 0.0;
#pragma unroll
    for (int c = 0; c < WJ4_ROWS / 2; c++)
        if (c < nch) {
#pragma unroll
            for (int q = 2 * c; q < 2 * c + 2; q++) {
                p0 = fma(u0[q], v0[q], p0);
                p1 = fma(u1[q], v1[q], p1);
                p2 = fma(u2[q], v2[q], p2);
                p3 = fma(u3[q], v3[q], p3);
            }
        }
    const bool b0 = sub & 1, b1 = sub & 2;
    const double q0 = (b0 ? p1 : p0) + dppd<DPP_XOR1>(b0 ? p0 : p1);
    const double q1 = (b0 ? p3 : p2) + dppd<DPP_XOR1>(b0 ? p2 : p3);
    double ga = (b1 ? q1 : q0) + dppd<DPP_XOR2>(b1 ? q0 : q1);  // product sub & 3 of this quad
    ga += xor4d(ga);
    ga += dppd<DPP_ROR8>(ga);
    if (G >= 32) {
        double x = ga, y = ga;
        swap16d(x, y);
        ga = x + y;
    }
    if (G >= 64) {
        double x = ga, y = ga;
        swap32d(x, y);
        ga = x + y;
    }
    const double al = b1 ? (b0 ? nu3 : nu2) : (b0 ? nu1 : nu0), be = b1 ? (b0 ? nv3 : nv2) : (b0 ? nv1 : nv0);
    double cs = 1.0, sn = 0.0;
    bool rot = false;
    if (fmin(al, be) > nz) rot = wj_rotation(al, be, ga, tol, cs, sn);
    if (!rot) {
        cs = 1.0;
        sn = 0.0;
    }
    if (__ballot(rot) == 0) return 0;
    const double na = rot ? cs * cs * al - 2.0 * cs * sn * ga + sn * sn * be : al;
    const double nb = rot ? sn * sn * al + 2.0 * cs * sn * ga + cs * cs * be : be;
    nu0 = wj_quad(na, 0), nu1 = wj_quad(na, 1), nu2 = wj_quad(na, 2), nu3 = wj_quad(na, 3);
    nv0 = wj_quad(nb, 0), nv1 = wj_quad(nb, 1), nv2 = wj_quad(nb, 2), nv3 = wj_quad(nb, 3);
    const double c0 = wj_quad(cs, 0), c1 = wj_quad(cs, 1), c2 = wj_quad(cs, 2), c3 = wj_quad(cs, 3);
    const double s0 = wj_quad(sn, 0), s1 = wj_quad(sn, 1), s2 = wj_quad(sn, 2), s3 = wj_quad(sn, 3);
    auto turn = [](double &x, double &y, double c, double s) {
        const double xo = x, yo = y;
        x = fma(c, xo, -(s * yo));
        y = fma(s, xo, c * yo);
    };
#pragma unroll
    for (int c = 0; c < WJ4_ROWS / 2; c++)
        if (c < nch) {
#pragma unroll
            for (int q = 2 * c; q < 2 * c + 2; q++) {
                turn(u0[q], v0[q], c0, s0);
                turn(u1[q], v1[q], c1, s1);
                turn(u2[q], v2[q], c2, s2);
                turn(u3[q], v3[q], c3, s3);
            }
        }
    return !rot ? 0 : (ga * ga > WJ_SMALL2 * al * be ? 3 : 1);
}

// rows and column stride in LDS; columns of neighbouring groups (G = 16) lie
// sixteen banks apart
template <int G>
__host__ __device__ __forceinline__ int wj4_rows(int m) { return (m + 2 * G - 1) / (2 * G) * (2 * G); }
template <int G>
__host__ __device__ __forceinline__ int wj4_ldc(int m) { return wj4_rows<G>(m) + (G == 16 ? 4 : 0); }
// LDS columns (a multiple of eight), 0 when a lane would hold too many rows
template <int G>
__host__ __device__ __forceinline__ int wj4_cols(int m)
{
    if (wj4_rows<G>(m) > WJ4_ROWS * G) return 0;
    const int c = WQ_MAIN / wj4_ldc<G>(m) / 8 * 8, most = BS / G * 8;
    return c < most ? c : most;
}

// wj_jacobi's contract.  The n columns stay in LDS when they fit; otherwise
// blocks of up to half of the LDS columns take turns, as there.  Norms are
// kept up to date through the rotations and computed anew in every sweep.
template <int G>
__device__ __forceinline__ int wj4_jacobi(int m, int n, double *M, int ldm, double nz, const WqLds &S)
{
    double *L = S.main, *nrm = S.T;  // 128 norms
    const int tid = threadIdx.x, kp = tid / G, sub = tid % G;
    const int rows = wj4_rows<G>(m), nch = rows / (2 * G), ldc = wj4_ldc<G>(m), cap = wj4_cols<G>(m);
    const double tol = 4.0e-16 * sqrt((double)m);
    auto move_in = [&](int c0, int g0, int nc) {
        wq_cols(
            rows, nc, [&](int r, int c) { return (g0 + c < n && r < m) ? M[r + (size_t)(g0 + c) * ldm] : 0.0; },
            [&](int r, int c, double v) { L[(c0 + c) * ldc + r] = v; });
    };
    auto move_out = [&](int c0, int g0, int nc) {
        wq_cols(
            m, min(nc, n - g0), [&](int r, int c) { return L[(c0 + c) * ldc + r]; },
            [&](int r, int c, double v) { M[r + (size_t)(g0 + c) * ldm] = v; });
    };
    auto norms = [&](int nc) {
        const int lane = tid & 63;
        for (int c = tid >> 6; c < nc; c += NWAVE) {
            double s = 0.0;
            for (int r = lane; r < rows; r += 64) s = fma(L[c * ldc + r], L[c * ldc + r], s);
            s = wsum(s);
            if (lane == 0) nrm[c] = s;
        }
        __syncthreads();
    };
    // blocks of four columns at ca and cb: all pairs across, and within both if `own`
    auto visit = [&](int ca, int cb, bool own) -> int {
        double *xa = L + ca * ldc + sub, *xb = L + cb * ldc + sub;
        int nc_ = nch;
        asm volatile("" : "+s"(nc_));  // no hoisted comparison per chunk
        double x0[WJ4_ROWS], x1[WJ4_ROWS], x2[WJ4_ROWS], x3[WJ4_ROWS], y0[WJ4_ROWS], y1[WJ4_ROWS], y2[WJ4_ROWS],
            y3[WJ4_ROWS];
#pragma unroll
        for (int c = 0; c < WJ4_ROWS / 2; c++)
            if (c < nc_) {
#pragma unroll
                for (int q = 2 * c; q < 2 * c + 2; q++) {
                    x0[q] = xa[G * q], x1[q] = xa[ldc + G * q], x2[q] = xa[2 * ldc + G * q], x3[q] = xa[3 * ldc + G * q];
                    y0[q] = xb[G * q], y1[q] = xb[ldc + G * q], y2[q] = xb[2 * ldc + G * q], y3[q] = xb[3 * ldc + G * q];
                }
            }
        double a0 = nrm[ca], a1 = nrm[ca + 1], a2 = nrm[ca + 2], a3 = nrm[ca + 3];
        double b0 = nrm[cb], b1 = nrm[cb + 1], b2 = nrm[cb + 2], b3 = nrm[cb + 3];
        int any = 0;
        if (own) {
            any |= wj_rot4<G>(x0, x1, x2, x3, y0, y1, y2, y3, a0, a1, a2, a3, b0, b1, b2, b3, nc_, sub, tol, nz);
            any |= wj_rot4<G>(x0, x2, x1, x3, y0, y2, y1, y3, a0, a2, a1, a3, b0, b2, b1, b3, nc_, sub, tol, nz);
            any |= wj_rot4<G>(x0, x3, x1, x2, y0, y3, y1, y2, a0, a3, a1, a2, b0, b3, b1, b2, nc_, sub, tol, nz);
        }
        any |= wj_rot4<G>(x0, y0, x1, y1, x2, y2, x3, y3, a0, b0, a1, b1, a2, b2, a3, b3, nc_, sub, tol, nz);
        any |= wj_rot4<G>(x0, y1, x1, y2, x2, y3, x3, y0, a0, b1, a1, b2, a2, b3, a3, b0, nc_, sub, tol, nz);
        any |= wj_rot4<G>(x0, y2, x1, y3, x2, y0, x3, y1, a0, b2, a1, b3, a2, b0, a3, b1, nc_, sub, tol, nz);
        any |= wj_rot4<G>(x0, y3, x1, y0, x2, y1, x3, y2, a0, b3, a1, b0, a2, b1, a3, b2, nc_, sub, tol, nz);
        if (__ballot(any) == 0) return 0;
#pragma unroll
        for (int c = 0; c < WJ4_ROWS / 2; c++)
            if (c < nc_) {
#pragma unroll
                for (int q = 2 * c; q < 2 * c + 2; q++) {
                    xa[G * q] = x0[q], xa[ldc + G * q] = x1[q], xa[2 * ldc + G * q] = x2[q], xa[3 * ldc + G * q] = x3[q];
                    xb[G * q] = y0[q], xb[ldc + G * q] = y1[q], xb[2 * ldc + G * q] = y2[q], xb[3 * ldc + G * q] = y3[q];
                }
            }
        if (sub == 0) {
            nrm[ca] = a0, nrm[ca + 1] = a1, nrm[ca + 2] = a2, nrm[ca + 3] = a3;
            nrm[cb] = b0, nrm[cb + 1] = b1, nrm[cb + 2] = b2, nrm[cb + 3] = b3;
        }
        return any;
    };
    // every pair of the first 4 nb4 LDS columns (nb4 even)
    auto all_pairs = [&](int nb4) {
        int any = 0;
        for (int r = 0; r < nb4 - 1; r++) {
            if (kp < nb4 / 2) {
                int ca = kp == 0 ? 0 : kp - 1 + r, cb = nb4 - 2 - kp + r;
                if (kp) {
                    if (ca >= nb4 - 1) ca -= nb4 - 1;
                    ca++;
                }
                if (cb >= nb4 - 1) cb -= nb4 - 1;
                cb++;
                any |= visit(4 * ca, 4 * cb, r == 0);
            }
            __syncthreads();
        }
        return any;
    };
    int sweep = 0;
    if (n <= cap) {
        const int nb4 = (n + 7) / 8 * 2;
        move_in(0, 0, 4 * nb4);
        __syncthreads();
        for (; sweep < BLK_JACOBI_SWEEPS; sweep++) {
            norms(4 * nb4);
            if (!__syncthreads_or(all_pairs(nb4) & 2)) break;
        }
        move_out(0, 0, n);
        __syncthreads();
        return sweep;
    }
    // blocks of W columns, as many as needed and of even widths
    const int nb = (n + cap / 2 - 1) / (cap / 2), W = ((n + nb - 1) / nb + 3) / 4 * 4, nbe = nb + (nb & 1);
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
                move_in(0, ba * W, W);
                move_in(W, bb < nb ? bb * W : n, W);
                __syncthreads();
                norms(2 * W);
                int rot = 0;
                const int w4 = W / 4;
                if (rd == 0) {
                    rot = all_pairs(2 * w4);
                } else {
                    for (int r = 0; r < w4; r++) {
                        if (kp < w4) {
                            const int cb = kp + r < w4 ? kp + r : kp + r - w4;
                            rot |= visit(4 * kp, W + 4 * cb, false);
                        }
                        __syncthreads();
                    }
                }
                any |= rot & 2;
                if (__syncthreads_or(rot)) {
                    move_out(0, ba * W, W);
                    move_out(W, bb < nb ? bb * W : n, W);
                }
                __syncthreads();
            }
        if (!__syncthreads_or(any)) break;
    }
    return sweep;
}

// tallest matrix wj_svd takes (64 lanes per pair, 8 columns of LDS)
#define WJ_MAXN 2304
__device__ __forceinline__ int wj_svd(int m, int n, double *M, int ldm, double nz, const WqLds &S)
{
    if (n <= 1) return 0;
    // all columns resident with the fewest lanes per block pair, else the widest blocks
    const int c16 = wj4_cols<16>(m), c32 = wj4_cols<32>(m), c64 = wj4_cols<64>(m);
    if (n > 64 || c32 < n) {
        if (c16 >= 64) return wj4_jacobi<16>(m, n, M, ldm, nz, S);
    }
    if (c32 >= 32) return wj4_jacobi<32>(m, n, M, ldm, nz, S);
    if (c64 >= 16) return wj4_jacobi<64>(m, n, M, ldm, nz, S);
    if (wj_takes<32>(m, n)) return wj_jacobi<32>(m, n, M, ldm, nz, S.main);
    return wj_jacobi<64>(m, n, M, ldm, nz, S.main);
}

// squared Frobenius norm of M (n x n, ld ldm), the same on every thread
__device__ __forceinline__ double wq_fro2(int n, const double *M, int ldm, double *red)
{
    double s = 0.0;
    wq_cols(
        n, n, [&](int r, int c) { return M[r + (size_t)c * ldm]; }, [&](int, int, double v) { s = fma(v, v, s); });
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

// Jacobi on the columns of X (n x n, ld n), graded by rows of an R factor:
// the columns after the last one above the floor nz (a squared norm) take no
// part.  Returns the sweeps.
__device__ __forceinline__ int wq_graded_svd(int n, double *X, double nz, const WqLds &S)
{
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
    return wj_svd(n, s_ke, X, n, nz, S);
}

// Right singular vectors of M (n x n, ld ldm): M = Q1 R, and one-sided Jacobi
// on the columns of R^T (the rows of R) gives R^T J = Vs S.  The rows of an
// (unpivoted) R are graded, which takes 5 .. 8 sweeps where the columns of M
// or M^T take 8 .. 22 (stacks of 44 .. 115 columns of 2-D sqexp updates).  M is
// overwritten by its QR; X (n x n, ld n) returns Vs S in columns 0 .. n - 1
// (unsorted).  Returns the sweeps.
template <int R>
__device__ __forceinline__ int wq_right_svd(int n, double *M, int ldm, double *X, double nz, double *Tsave, double *Vb,
                                            const WqLds &S)
{
    wq_geqrf<R>(n, n, M, ldm, Tsave, Vb, S);
    // X(r, i) = R(i, r): threads run down the columns of R
    wq_cols(
        n, n, [&](int i, int r) { return r >= i ? M[i + (size_t)r * ldm] : 0.0; },
        [&](int i, int r, double v) { X[r + (size_t)i * n] = v; });
    return wq_graded_svd(n, X, nz, S);
}

// dst (n x n) <- upper triangle of src, zeros below the diagonal
__device__ __forceinline__ void wq_triu(int n, const double *src, int lds, double *dst, int ldd)
{
    wq_cols(
        n, n, [&](int r, int c) { return r <= c ? src[r + (size_t)c * lds] : 0.0; },
        [&](int r, int c, double v) { dst[r + (size_t)c * ldd] = v; });
}
