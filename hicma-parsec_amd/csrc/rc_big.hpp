// rc_big.hpp -- recompression of a low-rank gemm update by one 256-thread
// workgroup per task, for any stack width (wglin.hpp's QR and Jacobi).
//
// C' = Cu Cv^T - A B^T:  (v) A, B low rank: Qn = -Bu (Av^T Bv)^T;  (iv) B dense:
// Qn = -B Av.  P = [Cu Au], Q = [Cv Qn];  P = Qp Rp, Q = Qq Rq (Householder);
// M = Rp Rq^T = Us S Vs^T: wq_right_svd gives Vs, and M Vs = Us S;  keep sigma >= acc (or the fixed rank) capped at maxrank;
// U' = Qp [Us S; 0], V' = Qq [Vs; 0] by applying the reflectors.
//
// What bounds it: the chains of one task (a reduction and a barrier per
// panel column and per Jacobi round), since the steps that need it have few
// tasks; hence one workgroup with the whole register file and LDS of a CU per
// task, panels in registers and Jacobi columns in LDS.  The kernel it replaced
// ran the Jacobi in global memory with one lane per pair and accumulated both
// sets of vectors.  Factorization of N=2700 tile 270 band 1 (stacks up to 150):
// 889 -> 33 ms; N=4096 tile 512 3-D sqexp band 3 (stacks up to 350): 1637 ->
// 83 ms.  Against the four-wave kernel with back substitution that took
// stacks of 61 .. 128 columns: N=2600 tile 270 band 3 33 -> 15 ms, N=90000 tile
// 900 552 -> 460 ms (37 such tasks a step), so it takes every stack above
// WV_S2MAX.
//
// The tasks come from a list filled on the device (order irrelevant: tasks of
// a step are independent) and are taken one at a time from a counter.
#pragma once
#include "tlr_kernels.hpp"
#include "wglin.hpp"

struct RbWs {
    size_t stride;  // doubles per workgroup
    int smax;       // 2 cap
};

__host__ __device__ inline size_t rb_slot_doubles(int NB, int cap)
{
    const size_t smax = 2 * (size_t)cap, nt = (smax + WQ_PW - 1) / WQ_PW;
    return 2 * (size_t)NB * smax + 3 * nt * WQ_PW * WQ_PW + (size_t)cap * cap + 3 * smax * smax +
           (size_t)WQ_PW * (((smax > (size_t)NB ? smax : NB) + 63) / 64 * 64 + 17);
}

// whether k_rc_big takes tiles of NB rows with ranks up to cap
__host__ __device__ inline bool rb_fits(int NB, int cap) { return NB <= WQ_MAXROWS && 2 * cap <= WQ_MAXROWS; }

template <int R>
__global__ void __launch_bounds__(BS, 1)
k_rc_big(TLR t, int k, const int *list, const int *count, int *next, double *ws, RbWs g, double acc, int fixed_rk,
         int maxrank, OpLog o, int *ovf, const double *qn_dense)
{
    extern __shared__ double sm[];
    __shared__ int s_idx, s_nr;
    const WqLds S = wq_lds(sm);
    const int NB = t.NB, NT = t.NT, cap = t.cap, b = t.band_size, tid = threadIdx.x, smax = g.smax;
    double *P = ws + (size_t)blockIdx.x * g.stride, *Q = P + (size_t)NB * smax;
    const size_t nt = (smax + WQ_PW - 1) / WQ_PW;
    double *Tp = Q + (size_t)NB * smax, *Tq = Tp + nt * WQ_PW * WQ_PW;
    double *Tm = Tq + nt * WQ_PW * WQ_PW, *Xr = Tm + nt * WQ_PW * WQ_PW;
    double *B1 = Xr + (size_t)cap * cap, *B2 = B1 + (size_t)smax * smax, *Ms = B2 + (size_t)smax * smax;
    double *Vb = Ms + (size_t)smax * smax;
    const int cnt = *count;
    for (;;) {
        if (tid == 0) s_idx = atomicAdd(next, 1);
        __syncthreads();
        const int idx = s_idx;
        __syncthreads();
        if (idx >= cnt) break;
        int hi, lo;
        tri_decode(list[idx], hi, lo);
        const int m = k + 1 + hi, n = k + 1 + lo;
        const bool bdense = (n - k < b);
        const int ra = *rank_at(t, m, k), rc = *rank_at(t, m, n);
        const int rb = bdense ? 0 : *rank_at(t, n, k);
        const int s = rc + ra;
        const double *Au = lr_tile(t, m, k), *Av = Au + (size_t)NB * ra;
        double *C = lr_tile(t, m, n);
        // stacks
        double *Qn = Q + (size_t)rc * NB;
        wq_copy(NB, rc, C, NB, P, NB);
        wq_copy(NB, ra, Au, NB, P + (size_t)rc * NB, NB);
        wq_copy(NB, rc, C + (size_t)NB * rc, NB, Q, NB);
        __syncthreads();
        if (!bdense) {
            const double *Bu = lr_tile(t, n, k), *Bv = Bu + (size_t)NB * rb;
            blk_gemm<true, false>(ra, rb, NB, 1.0, Av, NB, Bv, NB, 0.0, Xr, ra, S.main);
            blk_gemm<false, true>(NB, ra, rb, -1.0, Bu, NB, Xr, ra, 0.0, Qn, NB, S.main);
        } else if (qn_dense && ra > 0 && s <= QN_COLS) {
            wq_copy(NB, ra, qn_dense + qn_slot(NT, NB, k, m, n), NB, Qn, NB);  // formed by k_qn_dense
        } else {
            blk_gemm<false, false>(NB, ra, NB, -1.0, band_tile(t, n, k), NB, Av, NB, 0.0, Qn, NB, S.main);
        }
        int nr = 0;
        if (s > 0) {
            wq_geqrf<R>(NB, s, P, NB, Tp, Vb, S);
            wq_geqrf<R>(NB, s, Q, NB, Tq, Vb, S);
            wq_triu(s, P, NB, B1, s);
            wq_triu(s, Q, NB, B2, s);
            __syncthreads();
            blk_gemm<false, true>(s, s, s, 1.0, B1, s, B2, s, 0.0, Ms, s, S.main);  // M = Rp Rq^T
            wq_copy(s, s, Ms, s, B1, s);
            const double f2 = wq_fro2(s, Ms, s, S.red);
            __syncthreads();
            if (wq_right_svd<R>(s, B1, s, B2, wv_skip_floor(f2, s, acc, fixed_rk), Tm, Vb, S) >= BLK_JACOBI_SWEEPS &&
                tid == 0)
                atomicAdd(o.unconv, 1);
            double *sig = S.main;
            int *pos = (int *)(sig + smax);
            wq_sigma(s, s, B2, s, sig, pos);
            if (tid < 64) {
                int c = 0;
                if (fixed_rk > 0) {
                    c = fixed_rk < s ? fixed_rk : s;
                } else {
                    for (int j = tid; j < s; j += 64) c += (sig[j] >= acc);
                    c = (int)wsum((double)c);
                }
                if (tid == 0) {
                    if (c > maxrank) {
                        atomicAdd(ovf, 1);
                        c = maxrank;
                    }
                    s_nr = c;
                }
            }
            __syncthreads();
            nr = s_nr;
            // V' <- [Vs_r; 0], U' <- [M Vs_r; 0], then the reflectors
            double *Un = C, *Vn = C + (size_t)NB * nr;
            for (int j = tid >> 6; j < s; j += NWAVE) {
                const int q = pos[j];
                if (q >= nr) continue;
                const double inv = sig[j] > 0.0 ? 1.0 / sig[j] : 0.0;
                for (int i = tid & 63; i < NB; i += 64) {
                    Vn[i + (size_t)q * NB] = (i < s) ? B2[i + (size_t)j * s] * inv : 0.0;
                    if (i >= s) Un[i + (size_t)q * NB] = 0.0;
                }
            }
            __syncthreads();
            blk_gemm<false, false>(s, nr, s, 1.0, Ms, s, Vn, NB, 0.0, Un, NB, S.main);
            wq_apply<R>(NB, nr, s, P, NB, Tp, Un, NB, Vb, S);
            wq_apply<R>(NB, nr, s, Q, NB, Tq, Vn, NB, Vb, S);
        }
        if (tid == 0) {
            *rank_at(t, m, n) = nr;
            rank_hist(o, NT, m, n, nr);
            rc_oplog(o, t, m, n, ra, rb, rc, nr, bdense);
        }
        __syncthreads();
    }
}

// Qn = -B Av for the dense-B tasks of step k that the wave kernels take
// (ra > 0, s <= 128); grid (64x64 tiles of an NB x 128 slot, (band - 1) T).
__global__ void __launch_bounds__(BS) k_qn_dense(TLR t, int k, double *qn)
{
    __shared__ double sm[BLK_GEMM_SMEM];
    const int NB = t.NB, NT = t.NT, b = t.band_size, T = NT - 1 - k;
    const int m = k + 1 + (int)(blockIdx.y % T), n = k + 1 + (int)(blockIdx.y / T);
    if (m - n < b) return;
    const int ra = *rank_at(t, m, k), rc = *rank_at(t, m, n);
    if (ra <= 0 || rc + ra > 128) return;
    const int nrt = (NB + GT - 1) / GT;
    const int ti = blockIdx.x % nrt, tj = blockIdx.x / nrt;
    if (tj * GT >= ra) return;
    const double *Av = lr_tile(t, m, k) + (size_t)NB * ra;
    gemm_tile<false, false>(ti * GT, tj * GT, NB, ra, NB, -1.0, band_tile(t, n, k), NB, Av, NB, 0.0,
                            qn + qn_slot(NT, NB, k, m, n), NB, sm);
}

// Sorts the low-rank results of step k into task lists (the order inside a
// list is irrelevant: tasks of one step are independent): 0 (s, rb <= 32),
// 1 (<= 48), 2 (s <= WV_S2MAX, rb <= WV_SMAX) run on one wave each; 3, every other
// task, on one workgroup each (k_rc_big).  A dense B (band tile) needs its
// Qn = -B Av from k_qn_dense to run on a wave.  With big_only every task goes to
// list 3.  A low-rank update by a rank-0 factor changes nothing and is skipped.
// wcount: [0..3] list lengths, [4..7] next-task counters, [8] length and [9]
// next task of the redo list (list 4).
__global__ void k_classify_wave(TLR t, int k, int *wlist, int *wcount, int cap, int big_only, int qn_dense)
{
    const int T = t.NT - 1 - k;
    const long long ntask = (long long)T * (T - 1) / 2;
    long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= ntask) return;
    int hi, lo;
    tri_decode(e, hi, lo);
    const int m = k + 1 + hi, n = k + 1 + lo, b = t.band_size;
    if (m - n < b) return;
    const bool bdense = (n - k < b);
    const int ra = *rank_at(t, m, k), rc = *rank_at(t, m, n), rb = bdense ? 0 : *rank_at(t, n, k);
    const int s = rc + ra;
    if (ra < 0 || rb < 0 || rc < 0 || (!bdense && (ra == 0 || rb == 0))) return;
    int l = 3;
    if (!big_only && ra > 0 && (!bdense || qn_dense))
        l = (s <= 32 && rb <= 32) ? 0 : ((s <= 48 && rb <= 48) ? 1 : (s <= WV_S2MAX && rb <= WV_SMAX ? 2 : 3));
    wlist[(size_t)l * cap + atomicAdd(wcount + l, 1)] = (int)e;
}
