// gen.hpp -- compression of the off-band covariance tiles by one 256-thread
// workgroup per tile (STARS-H's starsh_dense_dlrrsdd restated):
//   Y = D Omega, Y = Q R;  X = D^T Q, X = Qx Rx;  Rx = Us S Vr^T (Jacobi);
//   rank by the relative Frobenius tail; U = Q Vr, V = Qx [Us S; 0].
// The sketch width is adaptive: see k_compress.
// What bounds it: with thousands of tiles the two products (matrix cores and the
// covariance's exponentials) and the panels' reductions, with the few tiles of a
// wide sketch the Jacobi rounds of one workgroup.  The kernel it replaced kept D
// and every intermediate in global memory, built panels column by column there
// and ran the Jacobi on the columns of Rx, both sets of vectors accumulated, one
// lane per pair at 266 columns.  Measured: 4,950 tiles of 900 rows, sketch 64:
// 229 -> 88 ms; 496 tiles of 512 rows, sketches 64 and 160: 90 -> 12 ms; 28 tiles of
// 512 rows of 3-D exp, sketches 64, 160 and 266: 637 -> 42 ms.
#pragma once
#include "rc_big.hpp"

// tiles and sketches k_compress_wg takes
__host__ __device__ inline bool gw_fits(int NB, int p) { return NB <= WQ_MAXROWS && p <= NB; }
// widest sketch whose two products form D on the fly (one 64-column tile of
// the result, so every entry of D is formed once per product)
#define GW_FUSED 64

__host__ __device__ inline size_t gw_slot_doubles(int NB, int p)
{
    const size_t nt = (size_t)(p + WQ_PW - 1) / WQ_PW;
    return (p > GW_FUSED ? (size_t)NB * NB : 0) + 3 * (size_t)NB * p + 2 * nt * WQ_PW * WQ_PW + 3 * (size_t)p * p +
           (size_t)WQ_PW * (((size_t)NB + 63) / 64 * 64 + 17);
}

// tiles of the next pass: every off-band tile (redo = 0), or those a narrower
// sketch marked; n[0] counts them, n[1] is their next-task counter
__global__ void k_gen_list(TLR t, int redo, int *list, int *n)
{
    const long long ntask = (long long)t.NT * (t.NT - 1) / 2;
    const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= ntask) return;
    int hi, lo;
    tri_decode(e, hi, lo);
    if (hi - lo < t.band_size || (redo && *rank_at(t, hi, lo) != GEN_REDO)) return;
    list[atomicAdd(n, 1)] = (int)e;
}

// C (NB x p, p <= 64, ld ldc) = K B, K(i, k) the covariance of row point
// rt NB + i and column point kt NB + k, formed in the operand staging: thread t
// holds the coordinates of row t % 64 of the tile and evaluates four of a
// chunk's sixteen columns (wave-uniform points) while the previous chunk is
// multiplied.  B (NB x p, ld ldb).
__device__ __forceinline__ void gw_gemm(const TLR &t, int rt, int kt, const double *B, int ldb, int p, double *C,
                                        int ldc, double *sm)
{
    double *As = sm, *Bs = sm + MK_KC * MK_LD;  // As[k][j]: B^T, Bs[k][i]: K
    const int NB = t.NB, tid = threadIdx.x, lane = tid & 63, w = uni(tid >> 6);
    const int wi = 32 * (w & 1), wj = 32 * (w >> 1), i16 = lane & 15, k4 = lane >> 4;
    const double cexp = (t.kind == 4) ? -1.0 / t.beta : -1.0 / (2.0 * t.beta * t.beta);
    const double *xs = t.xyz, *ys = xs + t.N, *zs = (t.ndim == 3) ? ys + t.N : xs;
    for (int i0 = 0; i0 < NB; i0 += MK_T) {
        const int row = i0 + lane, gi = rt * NB + row;
        const bool rok = row < NB && gi < t.N;
        const int gic = rok ? gi : 0;
        const double xi = xs[gic], yi = ys[gic], zi = zs[gic];
        double pa[4], pb[4];
        auto load = [&](int kc) {
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int e = tid + 256 * q, kk = e & (MK_KC - 1), jj = e >> 4;
                pa[q] = (jj < p && kc + kk < NB) ? B[kc + kk + (size_t)jj * ldb] : 0.0;
            }
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int k = kc + w + 4 * q, gj = kt * NB + k;  // uniform
                const bool kok = k < NB && gj < t.N;
                const int gjc = kok ? gj : 0;
                const double dx = xi - xs[gjc], dy = yi - ys[gjc], dz = (t.ndim == 3) ? zi - zs[gjc] : 0.0;
                const double d2 = dx * dx + dy * dy + dz * dz;
                const double v = t.sigma2 * exp(cexp * (t.kind == 4 ? sqrt(d2) : d2));
                pb[q] = (rok && kok) ? v : 0.0;
            }
        };
        mk_d4 acc[2][2];
        mk_zero(acc);
        load(0);
        for (int kc = 0; kc < NB; kc += MK_KC) {
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int e = tid + 256 * q;
                As[(e & (MK_KC - 1)) * MK_LD + (e >> 4)] = pa[q];
                Bs[(w + 4 * q) * MK_LD + lane] = pb[q];
            }
            __syncthreads();
            if (kc + MK_KC < NB) load(kc + MK_KC);
#pragma unroll
            for (int ks = 0; ks < MK_KC; ks += 4) {
                const double a0 = As[(ks + k4) * MK_LD + wi + i16], a1 = As[(ks + k4) * MK_LD + wi + 16 + i16];
                const double b0 = Bs[(ks + k4) * MK_LD + wj + i16], b1 = Bs[(ks + k4) * MK_LD + wj + 16 + i16];
                acc[0][0] = mk_mfma(a0, b0, acc[0][0]);
                acc[0][1] = mk_mfma(a0, b1, acc[0][1]);
                acc[1][0] = mk_mfma(a1, b0, acc[1][0]);
                acc[1][1] = mk_mfma(a1, b1, acc[1][1]);
            }
            __syncthreads();
        }
        mk_store(acc, [&](int j, int i, double v) {
            if (j < p && i0 + i < NB) C[i0 + i + (size_t)j * ldc] = v;
        });
    }
    __syncthreads();
}

template <int R>
__global__ void __launch_bounds__(BS, 1)
k_compress_wg(TLR t, const double *Om, const int *list, int *n, double *ws, size_t stride, int P, int p, double tol,
              int maxrank, int *info)
{
    extern __shared__ double sm[];
    __shared__ int s_idx, s_r;
    const WqLds S = wq_lds(sm);
    const int NB = t.NB, tid = threadIdx.x;
    const bool fused = p <= GW_FUSED;
    double *Y = ws + (size_t)blockIdx.x * stride, *Qm = Y + (size_t)NB * p, *X = Qm + (size_t)NB * p;
    const size_t nt = (size_t)(p + WQ_PW - 1) / WQ_PW;
    double *TY = X + (size_t)NB * p, *TX = TY + nt * WQ_PW * WQ_PW;
    double *Rx = TX + nt * WQ_PW * WQ_PW, *J = Rx + (size_t)p * p, *Vs = J + (size_t)p * p;
    double *Vb = Vs + (size_t)p * p, *D = Vb + (size_t)WQ_PW * wq_ldv(NB);
    const int cnt = n[0];
    for (;;) {
        if (tid == 0) s_idx = atomicAdd(n + 1, 1);
        __syncthreads();
        const int idx = s_idx;
        __syncthreads();
        if (idx >= cnt) break;
        int m, c;
        tri_decode(list[idx], m, c);
        if (fused) {
            gw_gemm(t, m, c, Om, NB, p, Y, NB, S.main);
        } else {
            for (size_t e = tid; e < (size_t)NB * NB; e += BS) D[e] = kval(t, m * NB + (int)(e % NB), c * NB + (int)(e / NB));
            __syncthreads();
            blk_gemm<false, false>(NB, p, NB, 1.0, D, NB, Om, NB, 0.0, Y, NB, S.main);
        }
        wq_geqrf<R>(NB, p, Y, NB, TY, Vb, S);
        wq_cols(
            NB, p, [&](int i, int j) { return (i == j) ? 1.0 : 0.0; },
            [&](int i, int j, double v) { Qm[i + (size_t)j * NB] = v; });
        wq_apply<R, true>(NB, p, p, Y, NB, TY, Qm, NB, Vb, S);
        if (fused) gw_gemm(t, c, m, Qm, NB, p, X, NB, S.main);
        else blk_gemm<true, false>(NB, p, NB, 1.0, D, NB, Qm, NB, 0.0, X, NB, S.main);
        wq_geqrf<R>(NB, p, X, NB, TX, Vb, S);
        wq_triu(p, X, NB, Rx, p);
        __syncthreads();
        // the rows of Rx are the columns of J = Rx^T = Vr S Us^T: graded already,
        // since Q's leading columns carry D's dominant directions.  A pair is left
        // alone below rounding noise or 1e-3 of the smallest column that the tail
        // rule can keep, tol ||D|| / sqrt(p).
        wq_cols(
            p, p, [&](int i, int r) { return Rx[i + (size_t)r * p]; },
            [&](int i, int r, double v) { J[r + (size_t)i * p] = v; });
        const double f2 = wq_fro2(p, Rx, p, S.red);
        const double nz = fmax((2.3e-16 * p) * (2.3e-16 * p), 1e-6 * tol * tol / p) * f2;
        __syncthreads();
        if (wq_graded_svd(p, J, nz, S) >= BLK_JACOBI_SWEEPS && tid == 0) atomicAdd(info + 2, 1);
        double *sig = S.main, *ssig = sig + p;
        int *pos = (int *)(ssig + p);
        wq_sigma(p, p, J, p, sig, pos);
        for (int j = tid; j < p; j += BS) ssig[pos[j]] = sig[j];
        __syncthreads();
        if (tid == 0) {
            double tot = 0.0, acc = 0.0;
            for (int i = 0; i < p; i++) tot += ssig[i] * ssig[i];
            const double stop = tot * tol * tol;
            int r = 0;
            for (int i = p - 1; i >= 0; i--) {
                acc += ssig[i] * ssig[i];
                if (acc > stop) {
                    r = i + 1;
                    break;
                }
            }
            const int rows = tdim(t, m), cols = tdim(t, c), mn = rows < cols ? rows : cols;
            if (p < P && r > p - GEN_OVS) r = GEN_REDO;
            else if (!(r < mn / 2 && r <= maxrank)) r = -1;
            *rank_at(t, m, c) = r;
            if (r == -1) atomicExch(info, -1);
            s_r = r;
        }
        __syncthreads();
        const int r = s_r;
        if (r <= 0) continue;
        double *U = lr_tile(t, m, c), *V = U + (size_t)NB * r;
        for (int j = tid >> 6; j < p; j += NWAVE) {
            const int q = pos[j];
            if (q >= r) continue;
            const double inv = sig[j] > 0.0 ? 1.0 / sig[j] : 0.0;
            for (int i = tid & 63; i < p; i += 64) Vs[i + (size_t)q * p] = J[i + (size_t)j * p] * inv;
            for (int i = p + (tid & 63); i < NB; i += 64) V[i + (size_t)q * NB] = 0.0;
        }
        __syncthreads();
        blk_gemm<false, false>(NB, r, p, 1.0, Qm, NB, Vs, p, 0.0, U, NB, S.main);
        blk_gemm<false, false>(p, r, p, 1.0, Rx, p, Vs, p, 0.0, V, NB, S.main);
        wq_apply<R>(NB, r, p, X, NB, TX, V, NB, Vb, S);
    }
}
