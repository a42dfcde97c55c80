// hicma_solve.hip -- triangular solves with the TLR factor, Sigma^-1 B and
// the Gaussian log-likelihood -1/2 (z^T Sigma^-1 z + log det Sigma + N log 2 pi).
//
// No counterpart in the reference (it stops at the factor); the solves read
// the factor in the layout HiCMA_dpotrf_L leaves (dense band tiles, compact
// [U | V] off-band tiles, each in the type the precision map gives) and the
// inverses of its diagonal tiles, which the factorization keeps (a descriptor
// without them has them formed first, k_tri_inv and k_tile_inv).
//
// One pass (L^-1 B or L^-T B, in place) is one launch, k_solve_flow: by tile rows
// in the order of the substitution (first to last forward, last to first
// backward), row m has 8 or 16 update tasks, each summing its share of every
// L_mk x_k, k before m, in that order, and one diagonal task per 32 rows of
// x_m = L_mm^-1 (b_m - sum).  Workgroups claim tasks in this order from a
// counter; a task waits only for tasks before it, so the schedule cannot
// deadlock whatever is resident, and each wait is bounded all the same.  While an
// update task waits for x_k it already holds its share of tile (m, k) in
// registers, so the chain per row is one small product, a sum over the shares
// and the block product with L_mm^-1.  All sums run in a fixed order: the
// results do not depend on scheduling.
//
// What bounds it: the chain of 2 NT hand-overs between compute units through the
// memory's coherence point.  The pass it replaced launched two kernels per tile
// row and formed the inverses in every call.  One vector at N=90000 band 1
// 7.5 -> 2.1 ms (0.55 TB/s of factor); Sigma^-1 b at N=2700 1.00 -> 0.21 ms; eight
// right-hand sides at N=30011 band 16 7.7 -> 4.6 ms; twenty backward at N=8091
// band 10 2.8 -> 0.9 ms.
#include "internal.hpp"
#include "mfma.hpp"
#include "wave.hpp"

#include <math.h>
#include <algorithm>
#include <utility>

#define SV_BK 64               // diagonal block edge
#define SF_T 512               // threads of the flow kernel
#define SF_W (SF_T / 64)
#define SF_GMAX 16             // update tasks per tile row: sf_shares()
#define SF_RB 32               // rows of x per diagonal task
#define SF_PF 4                // blocks of L_mm^-1 a diagonal task loads ahead
#define SF_SPIN_LIMIT (1 << 21)

// W = L_bb^-1 for every 64 x 64 diagonal block b of every diagonal tile k,
// into block (b, b) of its inverse (rows and columns beyond the tile, NB not
// a multiple of 64, hold the identity).  One wave per block: lane c forms
// column c of W by forward substitution, W(i, c) = (e_c(i) - sum_{c <= l < i}
// L(i, l) W(l, c)) / L(i, i), with L and W in LDS.
__global__ void __launch_bounds__(64) k_tri_inv(TLR t, double *Xinv)
{
    __shared__ double Lr[SV_BK * (SV_BK + 1)];  // L(i, l) at Lr[i * 65 + l]
    __shared__ double Ws[SV_BK * (SV_BK + 1)];  // W(i, c) at Ws[i * 65 + c]
    const int NB = t.NB, nbk = (NB + SV_BK - 1) / SV_BK;
    const int k = blockIdx.x / nbk, b = blockIdx.x % nbk, j0 = SV_BK * b;
    const int jb = min(SV_BK, NB - j0), lane = threadIdx.x;
    const double *Lk = band_tile(t, k, k) + j0 + (size_t)j0 * NB;
    for (int c = 0; c < SV_BK; c++) {
        double v = (lane == c) ? 1.0 : 0.0;
        if (lane < jb && c < jb) v = (c <= lane) ? Lk[lane + (size_t)c * NB] : 0.0;
        Lr[lane * (SV_BK + 1) + c] = v;
    }
    wv_sync();
    const int c = lane;
    for (int i = 0; i < SV_BK; i++) {
        double s = (i == c) ? 1.0 : 0.0;
        for (int l = c; l < i; l++) s = fma(-Lr[i * (SV_BK + 1) + l], Ws[l * (SV_BK + 1) + c], s);
        Ws[i * (SV_BK + 1) + c] = (i >= c) ? s / Lr[i * (SV_BK + 1) + i] : 0.0;
    }
    wv_sync();
    double *W = Xinv + (size_t)k * inv_tile(nbk) + inv_blk(b, b) * SV_BK * SV_BK;
    for (int j = 0; j < SV_BK; j++) W[lane + j * SV_BK] = Ws[lane * (SV_BK + 1) + j];
}

// The off-diagonal blocks of L_kk^-1, block column c of tile k per
// workgroup (grid NT nb): X_bc = -W_b sum_{j=c}^{b-1} L_bj X_jc for
// b = c+1 .. nb-1, the sum on the matrix cores, stored into block (b, c),
// then multiplied by W_b.
__global__ void __launch_bounds__(256) k_tile_inv(TLR t, double *Xinv)
{
    __shared__ double sm[MK_SMEM];
    const int NB = t.NB, nb = (NB + SV_BK - 1) / SV_BK;
    const int k = blockIdx.x / nb, c = blockIdx.x % nb;
    double *X0 = Xinv + (size_t)k * inv_tile(nb);
    const double *Lk = band_tile(t, k, k);
    for (int b = c + 1; b < nb; b++) {
        mk_d4 acc[2][2];
        mk_zero(acc);
        for (int j = c; j < b; j++) {
            const MkOps<false, true> op{Lk + (size_t)SV_BK * j * NB, NB, X0 + inv_blk(j, c) * SV_BK * SV_BK, SV_BK};
            mk_accum(op, NB, SV_BK, SV_BK * b, 0, 0, SV_BK, acc, sm);
        }
        double *Sb = X0 + inv_blk(b, c) * SV_BK * SV_BK;
        mk_store(acc, [&](int i, int j, double v) { Sb[i + j * SV_BK] = v; });
        __syncthreads();
        // X_bc = -W_b S
        mk_zero(acc);
        const MkOps<false, true> op2{X0 + inv_blk(b, b) * SV_BK * SV_BK, SV_BK, Sb, SV_BK};
        mk_accum(op2, SV_BK, SV_BK, 0, 0, 0, SV_BK, acc, sm);  // ends with a barrier: S is read
        mk_store(acc, [&](int i, int j, double v) { Sb[i + j * SV_BK] = -v; });
        __syncthreads();
    }
}

// ---- the pass ---------------------------------------------------------------

// Values that pass between workgroups are written and read past the L1 and the
// XCD's L2 (agent scope); a counter follows them once every store of the
// workgroup has completed.
__device__ __forceinline__ double sf_ld(const double *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void sf_st(double *p, double v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ int sf_cnt(const int *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void sf_publish(int *cnt)
{
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(cnt, 1);
}

// a[c][j] = F(r, cb + c), r = tid + 512 j, for the columns below c1, else 0; F
// (NB rows) held in type pr.  The resource ends with column c1 - 1.
template <int CC, int RT>
__device__ __forceinline__ void sf_cols(double (&a)[CC][RT], const void *F, int pr, int NB, int tid, int cb, int c1)
{
    const int es = pr == LR_F64 ? 8 : (pr == LR_F32 ? 4 : 2);
    const wv_rsrc rs = wv_col_rsrc((const double *)F, c1 * NB * es);
    int off[RT];
#pragma unroll
    for (int j = 0; j < RT; j++) off[j] = tid + SF_T * j < NB ? (tid + SF_T * j) * es : (int)WV_OOB;
    if (pr == LR_F64) {
#pragma unroll
        for (int c = 0; c < CC; c++)
#pragma unroll
            for (int j = 0; j < RT; j++) a[c][j] = wv_lds(rs, off[j], (cb + c) * NB * 8);
    } else if (pr == LR_F32) {
#pragma unroll
        for (int c = 0; c < CC; c++)
#pragma unroll
            for (int j = 0; j < RT; j++) a[c][j] = (double)wv_lds32(rs, off[j], (cb + c) * NB * 4);
    } else {
#pragma unroll
        for (int c = 0; c < CC; c++)
#pragma unroll
            for (int j = 0; j < RT; j++) a[c][j] = (double)lr_bf16{wv_lds16(rs, off[j], (cb + c) * NB * 2)};
    }
}

// wave totals of N = 4, 8 or 16 values: lane l gets that of value l / (64 / N)
__device__ __forceinline__ double sf_scatter(double (&p)[4]) { return wrs4(p[0], p[1], p[2], p[3]); }
__device__ __forceinline__ double sf_scatter(double (&p)[8]) { return wrs8(p); }
__device__ __forceinline__ double sf_scatter(double (&p)[16]) { return wrs16(p); }

// columns of a low-rank share held in registers (a wider share takes several rounds)
template <int RT>
struct SfCfg {
    static constexpr int CC = RT <= 2 ? 4 : 2;
};

// update tasks of a tile row: a dense tile needs more of them than a low-rank
// one (sixteen against eight: 4.6 and 5.6 ms for eight right-hand sides at N=30011
// band 16, 2.2 and 2.0 ms for one at N=90000 band 1)
__host__ __device__ __forceinline__ int sf_shares(const TLR &t) { return t.band_size > 1 ? SF_GMAX : 8; }

// Q right-hand sides of one pass over the rows r of the tiles, RT rows per
// thread (r = tid + 512 j).  Position p of the order is tile row p (forward) or
// NT-1-p (backward).  Task order: position, group of right-hand sides, then the
// updates and the diagonal tasks.  cnt: [0] task counter, then per (position,
// group) the finished update and diagonal tasks.  Pw: the shares' sums, NB x Q per
// (position, group, share).  LDS: x or y (64 nb x Q), partial sums.
template <int Q, int RT>
__global__ void __launch_bounds__(SF_T, 4)
k_solve_flow(TLR t, const double *Xinv, double *B, long ldb, int nrhs, int trans, double *Pw, int *cnt, int *stall)
{
    constexpr int CC = SfCfg<RT>::CC, NV = CC * Q <= 4 ? 4 : CC * Q;  // values of a reduction: 4, 8 or 16
    extern __shared__ double sm[];
    __shared__ int s_task, s_ready;
    const int NB = t.NB, NT = t.NT, nb = (NB + SV_BK - 1) / SV_BK, ngrp = (nrhs + Q - 1) / Q;
    const int G = sf_shares(t), nd = (NB + SF_RB - 1) / SF_RB, per = G + nd, ntask = NT * ngrp * per;
    double *xs = sm;                          // xs[i * Q + q]
    double *pt = sm + (size_t)nb * SV_BK * Q;  // 16 x 32 x Q
    for (;;) {
        // opaque, so that no address of one kind of task is kept through the other
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        const int lane = tid & 63, w = uni(tid >> 6);
        __syncthreads();  // s_task and the LDS are free
        if (tid == 0) s_task = atomicAdd(cnt, 1);
        __syncthreads();
        const int task = uni(s_task);
        if (task >= ntask) break;
        const int row = task / per, sub = task - row * per, p = row / ngrp, grp = row - p * ngrp;
        const int m = trans ? NT - 1 - p : p, q0 = grp * Q, nq = min(Q, nrhs - q0);
        int *uc = cnt + 16 + 2 * row, *dc = uc + 1;
        double *Pm = Pw + (size_t)row * G * NB * Q;
        const int rows_m = tdim(t, m);
        // thread 0 waits until *c reaches n
        auto wait = [&](const int *c, int n) {
            if (tid == 0) {
                int k = 0;
                while (sf_cnt(c) < n) {
                    __builtin_amdgcn_s_sleep(1);
                    if (++k > SF_SPIN_LIMIT) {
                        __hip_atomic_store(stall, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                        break;
                    }
                }
            }
            __syncthreads();
        };
        if (sub < G) {
            // ---- update: acc = b_m (share 0) - sum over earlier rows of its share
            const int g = sub;
            double acc[RT][Q];
#pragma unroll
            for (int j = 0; j < RT; j++)
#pragma unroll
                for (int q = 0; q < Q; q++) {
                    const int r = tid + SF_T * j;
                    acc[j][q] = (g == 0 && r < rows_m && q < nq) ? B[(size_t)m * NB + r + (q0 + q) * ldb] : 0.0;
                }
            double v[CC][RT], u[CC][RT], x[RT][Q];
            int ready = 0;
            bool have = false, xhave = false;  // v and u hold the first round of the tile, x its x
            // the share's columns c0 .. c1 of the tile at position pk, its factors
            struct Sh {
                const void *F, *G;  // w = F^T x, acc -= G w
                size_t off;
                int c0, c1, pr;
                bool dense;
            };
            auto share = [&](int pk) {
                const int k = trans ? NT - 1 - pk : pk, hi = trans ? k : m, lo = trans ? m : k;
                Sh s;
                s.dense = hi - lo < t.band_size;
                s.c0 = s.c1 = 0;
                s.F = s.G = nullptr;
                s.pr = LR_F64;
                if (!s.dense) {
                    const int r = uni(max(*rank_at(t, hi, lo), 0)), cs = (r + G - 1) / G;
                    s.c0 = min(r, g * cs);
                    s.c1 = min(r, s.c0 + cs);
                    s.pr = uni(lr_prec(t, hi, lo));
                    const char *T = (const char *)lr_tile(t, hi, lo);
                    const size_t vo = (size_t)NB * r * (s.pr == LR_F64 ? 8 : (s.pr == LR_F32 ? 4 : 2));
                    s.F = trans ? T : T + vo;
                    s.G = trans ? T + vo : T;
                } else {
                    s.F = band_tile(t, hi, lo);
                }
                return s;
            };
            auto load_x = [&](int pk) {
                const int k = trans ? NT - 1 - pk : pk, rk = tdim(t, k);
#pragma unroll
                for (int q = 0; q < Q; q++) {
                    const wv_rsrc rs = wv_col_rsrc(B + (size_t)k * NB + (q0 + (q < nq ? q : 0)) * ldb, q < nq ? rk * 8 : 0);
#pragma unroll
                    for (int j = 0; j < RT; j++) x[j][q] = wv_lds<true>(rs, (tid + SF_T * j) * 8, 0);
                }
            };
            Sh cur = share(0);
            for (int pk = 0; pk < p; pk++) {
                if (!have && cur.c0 < cur.c1) {
                    sf_cols(v, cur.F, cur.pr, NB, tid, cur.c0, cur.c1);
                    sf_cols(u, cur.G, cur.pr, NB, tid, cur.c0, cur.c1);
                }
                if (pk >= ready) {  // how many rows from pk on are solved
                    if (w == 0) {
                        const int *c = cnt + 16 + 2 * ((pk + lane) * ngrp + grp) + 1;
                        int n = 0, k = 0;
                        for (;;) {
                            const bool done = pk + lane < p && sf_cnt(c) >= nd;
                            const unsigned long long open = ~__ballot(done);
                            n = open ? __builtin_ctzll(open) : 64;
                            if (n > 0) break;
                            __builtin_amdgcn_s_sleep(1);
                            if (++k > SF_SPIN_LIMIT) {
                                if (lane == 0) __hip_atomic_store(stall, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                                n = 1;
                                break;
                            }
                        }
                        if (lane == 0) s_ready = pk + n;
                    }
                    __syncthreads();
                    ready = uni(s_ready);
                    __syncthreads();
                }
                if (cur.dense) {
                    const wv_rsrc T = wv_col_rsrc((const double *)cur.F, NB * NB * 8);
                    const int k = trans ? NT - 1 - pk : pk, rk = tdim(t, k);
                    // share g of the columns of T
                    const int cs = (NB + G - 1) / G, l0 = min(NB, g * cs), l1 = min(NB, l0 + cs);
                    const int i0 = trans ? 0 : l0, i1 = trans ? NB : l1;  // rows of x_k it needs
                    for (int e = tid; e < (i1 - i0) * Q; e += SF_T) {
                        const int q = e / (i1 - i0), i = i0 + e - q * (i1 - i0);
                        xs[i * Q + q] = (i < rk && q < nq) ? sf_ld(B + (size_t)k * NB + i + (q0 + q) * ldb) : 0.0;
                    }
                    __syncthreads();
                    if (!trans) {  // acc(r) -= sum over the share's columns T(r, l) x(l)
#pragma unroll
                        for (int j = 0; j < RT; j++) {
                            const int r = tid + SF_T * j;
                            if (r < NB) {
#pragma unroll 8
                                for (int l = l0; l < l1; l++) {
                                    const double tv = wv_lds(T, r * 8, l * NB * 8);
#pragma unroll
                                    for (int q = 0; q < Q; q++) acc[j][q] = fma(-tv, xs[l * Q + q], acc[j][q]);
                                }
                            }
                        }
                    } else {  // acc(l) -= T(:, l)^T x for the share's columns l, one wave each in turn
                        double *ob = pt;
                        for (int l = l0 + w; l < l1; l += SF_W) {
                            double d[Q];
#pragma unroll
                            for (int q = 0; q < Q; q++) d[q] = 0.0;
#pragma unroll 8
                            for (int i = lane; i < NB; i += 64) {
                                const double tv = wv_lds(T, i * 8, uni(l) * NB * 8);
#pragma unroll
                                for (int q = 0; q < Q; q++) d[q] = fma(tv, xs[i * Q + q], d[q]);
                            }
#pragma unroll
                            for (int q = 0; q < Q; q++) {
                                const double sv = wsum(d[q]);
                                if (lane == 0) ob[(l - l0) * Q + q] = sv;
                            }
                        }
                        __syncthreads();
#pragma unroll
                        for (int j = 0; j < RT; j++) {
                            const int r = tid + SF_T * j;
                            if (r >= l0 && r < l1) {
#pragma unroll
                                for (int q = 0; q < Q; q++) acc[j][q] -= ob[(r - l0) * Q + q];
                            }
                        }
                    }
                    __syncthreads();
                }
                const Sh now = cur;
                if (now.c0 < now.c1 && !xhave) load_x(pk);
                if (pk + 1 < p) cur = share(pk + 1);
                have = xhave = false;
                for (int cb = now.c0; cb < now.c1; cb += CC) {
                    // w = F^T x: the products summed over the rows of all waves
                    double pr[NV];
#pragma unroll
                    for (int e = 0; e < NV; e++) pr[e] = 0.0;
#pragma unroll
                    for (int c = 0; c < CC; c++)
#pragma unroll
                        for (int q = 0; q < Q; q++)
#pragma unroll
                            for (int j = 0; j < RT; j++) pr[c * Q + q] = fma(v[c][j], x[j][q], pr[c * Q + q]);
                    const double part = sf_scatter(pr);
                    if (lane % (64 / NV) == 0) pt[w * 16 + lane / (64 / NV)] = part;
                    // v is free: the next round, or the next tile's first one (and its x,
                    // if that row is solved), loads while this one goes on
                    const bool last = cb + CC >= now.c1, next = last && pk + 1 < p && cur.c0 < cur.c1;
                    if (!last) sf_cols(v, now.F, now.pr, NB, tid, cb + CC, now.c1);
                    if (next) {
                        sf_cols(v, cur.F, cur.pr, NB, tid, cur.c0, cur.c1);
                        if (pk + 1 < ready) {
                            load_x(pk + 1);
                            xhave = true;
                        }
                    }
                    __syncthreads();
                    // lanes 4e .. 4e+3 add value e's eight parts
                    double tot = pt[(2 * (lane & 3)) * 16 + (lane >> 2)] + pt[(2 * (lane & 3) + 1) * 16 + (lane >> 2)];
                    tot += dppd<DPP_XOR1>(tot);
                    tot += dppd<DPP_XOR2>(tot);
#pragma unroll
                    for (int c = 0; c < CC; c++)
#pragma unroll
                        for (int q = 0; q < Q; q++) {
                            const double wv = rdlane(tot, 4 * (c * Q + q));
#pragma unroll
                            for (int j = 0; j < RT; j++) acc[j][q] = fma(-u[c][j], wv, acc[j][q]);
                        }
                    if (!last) sf_cols(u, now.G, now.pr, NB, tid, cb + CC, now.c1);
                    if (next) {
                        sf_cols(u, cur.G, cur.pr, NB, tid, cur.c0, cur.c1);
                        have = true;
                    }
                    __syncthreads();  // pt is free
                }
            }
#pragma unroll
            for (int j = 0; j < RT; j++)
#pragma unroll
                for (int q = 0; q < Q; q++) {
                    const int r = tid + SF_T * j;
                    if (r < NB) sf_st(Pm + ((size_t)g * Q + q) * NB + r, acc[j][q]);
                }
            sf_publish(uc);
            continue;
        }
        // ---- diagonal: 32 rows of L_mm^-1 y or L_mm^-T y
        const int h = sub - G, b = h >> 1;
        const double *X0 = Xinv + (size_t)m * inv_tile(nb);
        // forward: thread (row i, column group cg): columns cg + 16 e of block (b, c), c <= b;
        // backward: wave w takes columns 4 w .. 4 w + 3 of the 32, lanes run down the rows of
        // block (c, b), c >= b
        const int i32 = tid & 31, cg = tid >> 5, ro = 32 * (h & 1);
        const wv_rsrc xr = wv_col_rsrc(X0, (int)inv_tile(nb) * 8);
        const int eo = trans ? (lane + SV_BK * (ro + 4 * w)) * 8 : (ro + i32 + SV_BK * cg) * 8;
        auto elem = [&](int cc, int e) -> double {  // cc-th block of the product
            const int blk = (int)(trans ? inv_blk(b + cc, b) : inv_blk(b, cc)) * SV_BK * SV_BK * 8;
            return wv_lds(xr, eo + (trans ? SV_BK * 8 : 16 * SV_BK * 8) * e, blk);
        };
        const int nblk = trans ? nb - b : b + 1;
        double pf[SF_PF][4];
#pragma unroll
        for (int cc = 0; cc < SF_PF; cc++)
            if (cc < nblk) {
#pragma unroll
                for (int e = 0; e < 4; e++) pf[cc][e] = elem(cc, e);
            }
        wait(uc, G);
        for (int e = tid; e < nb * SV_BK * Q; e += SF_T) {
            const int q = e / (nb * SV_BK), i = e - q * (nb * SV_BK);
            double s = 0.0;
            if (i < NB) {
                for (int g0 = 0; g0 < G; g0 += 8) {
                    double pv[8];
#pragma unroll
                    for (int g = 0; g < 8; g++) pv[g] = sf_ld(Pm + (unsigned)(((g0 + g) * Q + q) * NB + i));
#pragma unroll
                    for (int g = 0; g < 8; g++) s += pv[g];
                }
            }
            xs[i * Q + q] = s;
        }
        __syncthreads();
        double a[4 * Q];
#pragma unroll
        for (int e = 0; e < 4 * Q; e++) a[e] = 0.0;
        if (!trans) {
#pragma unroll
            for (int cc = 0; cc < SF_PF; cc++)
                if (cc < nblk) {
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const int i = SV_BK * cc + cg + 16 * e;
#pragma unroll
                        for (int q = 0; q < Q; q++) a[q] = fma(pf[cc][e], xs[i * Q + q], a[q]);
                    }
                }
#pragma unroll 2
            for (int cc = SF_PF; cc < nblk; cc++) {
                double f[4];
#pragma unroll
                for (int e = 0; e < 4; e++) f[e] = elem(cc, e);
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int i = SV_BK * cc + cg + 16 * e;
#pragma unroll
                    for (int q = 0; q < Q; q++) a[q] = fma(f[e], xs[i * Q + q], a[q]);
                }
            }
#pragma unroll
            for (int q = 0; q < Q; q++) pt[(cg * 32 + i32) * Q + q] = a[q];
            __syncthreads();
            for (int e = tid; e < 32 * nq; e += SF_T) {
                const int q = e >> 5, i = e & 31, r = SF_RB * h + i;
                double s = 0.0;
#pragma unroll
                for (int c = 0; c < 16; c++) s += pt[(c * 32 + i) * Q + q];
                if (r < rows_m) sf_st(B + (size_t)m * NB + r + (q0 + q) * ldb, s);
            }
        } else {
#pragma unroll
            for (int cc = 0; cc < SF_PF; cc++)
                if (cc < nblk) {
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const int i = SV_BK * (b + cc) + lane;
#pragma unroll
                        for (int q = 0; q < Q; q++) a[e * Q + q] = fma(pf[cc][e], xs[i * Q + q], a[e * Q + q]);
                    }
                }
#pragma unroll 2
            for (int cc = SF_PF; cc < nblk; cc++) {
                double f[4];
#pragma unroll
                for (int e = 0; e < 4; e++) f[e] = elem(cc, e);
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int i = SV_BK * (b + cc) + lane;
#pragma unroll
                    for (int q = 0; q < Q; q++) a[e * Q + q] = fma(f[e], xs[i * Q + q], a[e * Q + q]);
                }
            }
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int q = 0; q < Q; q++) {
                    const double s = wsum(a[e * Q + q]);
                    const int r = SF_RB * h + 4 * w + e;
                    if (lane == 0 && q < nq && r < rows_m) sf_st(B + (size_t)m * NB + r + (q0 + q) * ldb, s);
                }
        }
        sf_publish(dc);
    }
}

__global__ void k_sf_zero(int *p, int n)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e < n) p[e] = 0;
}

// sum of squares of x(0 : n), per-block parts, and their fixed-order total
__global__ void __launch_bounds__(256) k_sumsq_parts(const double *x, int n, double *part)
{
    __shared__ double red[4];
    const int i = blockIdx.x * 256 + threadIdx.x;
    double v = (i < n) ? x[i] * x[i] : 0.0;
    v = wsum(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

__global__ void __launch_bounds__(256) k_sum_seq(const double *part, int n, double *out)
{
    __shared__ double red[4];
    double s = 0.0;
    for (int q = threadIdx.x; q < n; q += 256) s += part[q];
    s = wsum(s);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) *out = (red[0] + red[1]) + (red[2] + red[3]);
}

// ---------------------------------------------------------------------------
// host side

// right-hand sides per group (groups of eight spill: 7.9 instead of 4.6 ms for
// eight right-hand sides at N=30011 band 16)
static int solve_q(int nrhs) { return nrhs >= 3 ? 4 : nrhs; }

// doubles of workspace a solve needs: every L_kk^-1 (unless the descriptor
// has them), the shares' sums, the counters, reduction parts (of the sum of
// squares, then of the log-det), eight scalars
static size_t solve_pw(const TLR &t, int nrhs)
{
    const size_t Q = solve_q(nrhs), ngrp = (nrhs + Q - 1) / Q;
    return (size_t)t.NT * ngrp * sf_shares(t) * t.NB * Q;
}
static size_t solve_cnt(const TLR &t, int nrhs)
{
    const size_t Q = solve_q(nrhs), ngrp = (nrhs + Q - 1) / Q;
    return 16 + 2 * (size_t)t.NT * ngrp;
}
size_t solve_ws_doubles(const TLR &t, int nrhs, bool have_inv)
{
    const int nbk = (t.NB + SV_BK - 1) / SV_BK;
    const size_t Np = (size_t)t.NT * t.NB;
    return (have_inv ? 0 : (size_t)t.NT * inv_tile(nbk)) + solve_pw(t, nrhs) + solve_cnt(t, nrhs) / 2 + 1 +
           std::max((Np + 255) / 256, (size_t)t.NT) + 8;
}

size_t hicma_solve_bytes(int N, int NB)
{
    TLR t{};
    t.N = N;
    t.NB = NB;
    t.NT = (N + NB - 1) / NB;
    return sizeof(double) * solve_ws_doubles(t, 1, true);
}

// LDS the solve kernels of four right-hand sides may take (the limit of the
// tile and rank sizes)
static size_t diag_lds(const TLR &t)
{
    const size_t nbk = (size_t)(t.NB + SV_BK - 1) / SV_BK;
    return sizeof(double) * (nbk * SV_BK * 4 + 4096);
}
static size_t update_lds(const TLR &t) { return sizeof(double) * (((size_t)t.NB + (size_t)t.cap) * 4 + 4096); }

template <int Q, int RT>
static int flow_launch_qr(hicma_ctx *ctx, const TLR &t, const double *Xinv, double *B, long ldb, int nrhs, int trans,
                          double *Pw, int *cnt)
{
    const int nb = (t.NB + SV_BK - 1) / SV_BK, ngrp = (nrhs + Q - 1) / Q;
    const int per = sf_shares(t) + (t.NB + SF_RB - 1) / SF_RB;
    // a transposed dense share of up to NB / 8 columns, or 16 x 32 partial sums
    const size_t part = std::max<size_t>(512, (size_t)t.NB / 8 + 1);
    const size_t lds = sizeof(double) * ((size_t)nb * SV_BK + part) * Q;
    const auto kern = k_solve_flow<Q, RT>;
    HIPCHK(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    const int ncnt = (int)solve_cnt(t, nrhs);
    hipLaunchKernelGGL(k_sf_zero, dim3((unsigned)((ncnt + 255) / 256)), dim3(256), 0, ctx->stream, cnt, ncnt);
    // two workgroups per CU
    const long ntask = (long)t.NT * ngrp * per;
    hipLaunchKernelGGL(kern, dim3((unsigned)std::min<long>(2L * ctx->ncu, ntask)), dim3(SF_T), lds, ctx->stream, t,
                       Xinv, B, ldb, nrhs, trans, Pw, cnt, ctx->d_stall);
    return 0;
}
template <int Q>
static int flow_launch_q(hicma_ctx *ctx, const TLR &t, const double *Xinv, double *B, long ldb, int nrhs, int trans,
                         double *Pw, int *cnt)
{
    // rows per thread
    if (t.NB <= SF_T) return flow_launch_qr<Q, 1>(ctx, t, Xinv, B, ldb, nrhs, trans, Pw, cnt);
    if (t.NB <= 2 * SF_T) return flow_launch_qr<Q, 2>(ctx, t, Xinv, B, ldb, nrhs, trans, Pw, cnt);
    if (t.NB <= 4 * SF_T) return flow_launch_qr<Q, 4>(ctx, t, Xinv, B, ldb, nrhs, trans, Pw, cnt);
    return flow_launch_qr<Q, 8>(ctx, t, Xinv, B, ldb, nrhs, trans, Pw, cnt);
}

// dirs: 1 forward, 2 backward, 3 both.  B: device, N x nrhs, ld ldb.
// quad (if not null): ||L^-1 B(:, 0)||^2 after the forward pass.  ws: device
// workspace of solve_ws_doubles() doubles.  Asynchronous on the context stream.
int solve_launch(hicma_ctx *ctx, hicma_tlr_desc *A, int dirs, int nrhs, double *B, long ldb, double *ws,
                 double *d_quad, double *d_logdet)
{
    const TLR &t = A->t;
    const int NT = t.NT, NB = t.NB, nbk = (NB + SV_BK - 1) / SV_BK;
    hipStream_t st = ctx->stream;
    const double *Xinv = A->linv;
    double *Pw = ws;
    if (!A->linv_ok) {
        hipLaunchKernelGGL(k_tri_inv, dim3((unsigned)(NT * nbk)), dim3(64), 0, st, t, ws);
        if (nbk > 1) hipLaunchKernelGGL(k_tile_inv, dim3((unsigned)(NT * nbk)), dim3(256), 0, st, t, ws);
        Xinv = ws;
        Pw = ws + (size_t)NT * inv_tile(nbk);
    }
    int *cnt = (int *)(Pw + solve_pw(t, nrhs));
    double *parts = (double *)cnt + solve_cnt(t, nrhs) / 2 + 1;
    *ctx->h_stall = 0;
    auto pass = [&](int trans) {
        const int Q = solve_q(nrhs);
        if (Q == 1) return flow_launch_q<1>(ctx, t, Xinv, B, ldb, nrhs, trans, Pw, cnt);
        if (Q == 2) return flow_launch_q<2>(ctx, t, Xinv, B, ldb, nrhs, trans, Pw, cnt);
        return flow_launch_q<4>(ctx, t, Xinv, B, ldb, nrhs, trans, Pw, cnt);
    };
    if (dirs & 1) {
        RCHK(pass(0));
        if (d_quad) {
            const int nb = (int)((t.N + 255) / 256);
            hipLaunchKernelGGL(k_sumsq_parts, dim3(nb), dim3(256), 0, st, (const double *)B, t.N, parts);
            hipLaunchKernelGGL(k_sum_seq, dim3(1), dim3(256), 0, st, (const double *)parts, nb, d_quad);
        }
    }
    if (dirs & 2) RCHK(pass(1));
    if (d_logdet) logdet_launch(t, parts, d_logdet, st);
    HIPCHK(hipGetLastError());
    return 0;
}

// after the stream has been waited for: whether a bounded device wait ran out
int solve_stalled(hicma_ctx *ctx)
{
    if (!*(volatile int *)ctx->h_stall) return 0;
    fprintf(stderr, "hicma_tlr: a wait of the solve's schedule ran out; the result is not valid\n");
    return HICMA_ERR_HIP;
}

int check_solve_args(hicma_ctx *ctx, hicma_tlr_desc *A, int nrhs, const double *B, long ldb)
{
    if (!ctx || !A || !B || nrhs < 1 || ldb < A->t.N) return HICMA_ERR_ARG;
    if (update_lds(A->t) > ctx->lds_max || diag_lds(A->t) > ctx->lds_max) return HICMA_ERR_ARG;
    return 0;
}

extern "C" int hicma_tlr_trsm(hicma_ctx *ctx, hicma_tlr_desc *A, int trans, int nrhs, double *B, int ldb)
{
    RCHK(check_solve_args(ctx, A, nrhs, B, ldb));
    if (trans != 0 && trans != 1) return HICMA_ERR_ARG;
    HIPCHK(hipSetDevice(ctx->device));
    RCHK(hicma_ensure_ws(ctx, sizeof(double) * solve_ws_doubles(A->t, nrhs, A->linv_ok)));
    RCHK(solve_launch(ctx, A, trans ? 2 : 1, nrhs, B, ldb, ctx->ws, nullptr, nullptr));
    HIPCHK(hipStreamSynchronize(ctx->stream));
    return solve_stalled(ctx);
}

extern "C" int hicma_tlr_potrs(hicma_ctx *ctx, hicma_tlr_desc *A, int nrhs, double *B, int ldb)
{
    RCHK(check_solve_args(ctx, A, nrhs, B, ldb));
    HIPCHK(hipSetDevice(ctx->device));
    RCHK(hicma_ensure_ws(ctx, sizeof(double) * solve_ws_doubles(A->t, nrhs, A->linv_ok)));
    RCHK(solve_launch(ctx, A, 3, nrhs, B, ldb, ctx->ws, nullptr, nullptr));
    HIPCHK(hipStreamSynchronize(ctx->stream));
    return solve_stalled(ctx);
}

// log-likelihood of one vector z (device, N entries; overwritten by L^-1 z)
int loglik_finish(hicma_ctx *ctx, const TLR &t, double *d_vals, double *logdet, double *quad, double *loglik)
{
    double h[2];
    // wait for the stream first, then copy: a copy into pageable memory that
    // waits for its stream holds the runtime's staging path meanwhile, and
    // other threads' copies queue behind it
    HIPCHK(hipStreamSynchronize(ctx->stream));
    RCHK(solve_stalled(ctx));
    HIPCHK(hipMemcpy(h, d_vals, 2 * sizeof(double), hipMemcpyDeviceToHost));
    if (quad) *quad = h[0];
    if (logdet) *logdet = h[1];
    if (loglik) *loglik = -0.5 * (h[0] + h[1] + (double)t.N * log(2.0 * 3.14159265358979323846));
    return 0;
}

extern "C" int hicma_tlr_loglik(hicma_ctx *ctx, hicma_tlr_desc *A, double *z, double *logdet, double *quad,
                                double *loglik)
{
    RCHK(check_solve_args(ctx, A, 1, z, A ? A->t.N : 0));
    HIPCHK(hipSetDevice(ctx->device));
    const size_t need = solve_ws_doubles(A->t, 1, A->linv_ok);
    RCHK(hicma_ensure_ws(ctx, sizeof(double) * need));
    double *vals = ctx->ws + need - 8;
    RCHK(solve_launch(ctx, A, 1, 1, z, A->t.N, ctx->ws, vals, vals + 1));
    return loglik_finish(ctx, A->t, vals, logdet, quad, loglik);
}

// ---- device memory plumbing for callers without a GPU runtime of their own ----
extern "C" int hicma_dev_malloc(hicma_ctx *ctx, size_t bytes, void **p)
{
    if (!ctx || !p) return HICMA_ERR_ARG;
    HIPCHK(hipSetDevice(ctx->device));
    HIPCHK(ctx_malloc(ctx, p, bytes ? bytes : 1));
    return 0;
}

extern "C" int hicma_dev_free(hicma_ctx *ctx, void *p)
{
    if (!ctx) return HICMA_ERR_ARG;
    HIPCHK(hipSetDevice(ctx->device));
    if (p) HIPCHK(ctx_free(ctx, p));
    return 0;
}

extern "C" int hicma_memcpy(hicma_ctx *ctx, void *dst, const void *src, size_t bytes, int to_device)
{
    if (!ctx || (!dst && bytes) || (!src && bytes)) return HICMA_ERR_ARG;
    HIPCHK(hipSetDevice(ctx->device));
    HIPCHK(hipStreamSynchronize(ctx->stream));
    HIPCHK(hipMemcpy(dst, src, bytes, to_device ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost));
    return 0;
}
