// rc_task.hpp -- sizes, thresholds and counts that the recompression kernels
// (rc_wave.hpp, rc_big.hpp) and their launches share.
#pragma once
#include "tlr.hpp"

#define WV_SMAX 64   // largest stack width s = rc + ra, and largest rb
#define WV_KMAX 16   // most rows per lane: NB <= 64 * WV_KMAX
#define WV_PW 4      // Householder panel width
#define WV_S2MAX 60  // widest stack of list 2; wider stacks go to k_rc_big

// one wave per SIMD (the full register file), four per workgroup: one workgroup per CU
#define WV_WPB 4

// per-wave HBM workspace: W (QR copy), Qn, Out (2 blocks), Rp, Rq, Ku
__host__ __device__ inline size_t wv_slot_doubles(int NB)
{
    return (size_t)NB * 4 * WV_SMAX + 4 * (size_t)WV_SMAX * WV_SMAX;
}

// Accepted error of the V' = Q (Rq^-1 Vs_r) back-substitution of the fast
// kernels, absolute in the tile: a fraction of the truncation threshold,
// never below rounding of M (fro = ||M||_F).
__device__ __forceinline__ double rc_solve_tol(double acc, int fixed_rk, double fro)
{
    const double floor_ = 1e-13 * fro;
    return (fixed_rk > 0 || !(acc > 0.0)) ? floor_ : fmax(1e-3 * acc, floor_);
}

// Squared-norm floor below which a Jacobi pair is not rotated: rounding noise
// of M, or, when truncating at acc, (1e-3 acc)^2 (see k_rc_wave).
__device__ __forceinline__ double wv_skip_floor(double f2, int s, double acc, int fixed_rk)
{
    const double nz = (2.3e-16 * s) * (2.3e-16 * s) * f2;
    const double tz = (fixed_rk > 0 || !(acc > 0.0)) ? 0.0 : (1e-3 * acc) * (1e-3 * acc);
    return fmax(nz, tz);
}

// op counts of one recompression (the reference's formulas) and its totals:
// op count, tasks, algorithmic bytes (8 * (inputs A, B, C + output) words, B
// dense in case iv)
__device__ __forceinline__ void rc_oplog(const OpLog &o, const TLR &t, int m, int n, int ra, int rb, int rc, int nr,
                                         bool bdense)
{
    const unsigned long long mm = tdim(t, m), ss = rc + ra;  // the reference counts with tile m's rows
    const unsigned long long qa = opc('q', mm, ss, 0, 0);
    // case iv (dense B) counts the product B Av, case v the products with B's factors
    const unsigned long long qb = bdense ? opc('q', mm, ss, 0, 0) + opc('m', ra, mm, mm, 0)
                                         : opc('m', ra, rb, mm, 0) + opc('m', ra, mm, rb, 0) + opc('q', mm, ss, 0, 0);
    const unsigned long long sv = opc('r', ss, ss, 2, 0) + opc('s', ss, 0, 0, 0) + ss * nr;
    const unsigned long long nu = opc('o', mm, nr, ss, 1), nv = opc('o', nr, mm, ss, 2);
    const unsigned long long ops = qa + qb + sv + nu + nv;
    oplog(o, t.NT, ops, m, n, false, false);
    atomicAdd(o.stat + 4, ops);
    atomicAdd(o.stat + 5, 1ULL);
    const unsigned long long words =
        2ULL * t.NB * (ra + rc + nr) + (bdense ? (unsigned long long)t.NB * t.NB : 2ULL * t.NB * rb);
    atomicAdd(o.stat + 6, 8ULL * words);
}

// Dense-B tasks (case iv: tile (n, k) in the band, (m, k) and (m, n) low
// rank) get Qn = -B Av precomputed by k_qn_dense into a slot of QN_COLS
// columns: slot (n - k - 1) T + (m - k - 1), T = NT - 1 - k.
#define QN_COLS 128
__host__ __device__ inline size_t qn_slot(int NT, int NB, int k, int m, int n)
{
    const int T = NT - 1 - k;
    return ((size_t)(n - k - 1) * T + (size_t)(m - k - 1)) * NB * QN_COLS;
}
