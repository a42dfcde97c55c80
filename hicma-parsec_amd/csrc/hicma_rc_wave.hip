// hicma_rc_wave.hip -- the one-wave recompressions of a step (rc_wave.hpp).
#include "internal.hpp"
#include "rc_wave.hpp"

// Every task of lists 2, 1 and 0, in this order: a wave takes the next one from
// the shared counter *wnext whatever its class, so the long tasks start first and
// the short ones fill the tail.  (One kernel per class on two streams left CUs idle
// behind the longest class and needed a stream more: with them a pass took 423 ms
// for N=90000 tile 900 band 1, 66.4 ms for N=16384 tile 512 band 3 with its
// generation, 10.0 ms for N=2600 tile 270 band 3; now 386, 61.5 and 9.1 ms, the
// last two also by KR = 8.)
template <int KR>
__global__ void __launch_bounds__(64 * WV_WPB, 1)
k_rc_wave(TLR t, int k, const int *wlist, int cap, const int *wcount, int *wnext, int *redo, int *nredo, double *ws,
          double acc, int fixed_rk, int maxrank, OpLog o, int *ovf, const double *qn_dense)
{
    extern __shared__ double smem[];
    const int lane = threadIdx.x & 63;
    const int wv = uni(threadIdx.x >> 6);
    double *L = smem + (size_t)wv * WV_LDS;
    double *Wq = ws + (size_t)(blockIdx.x * WV_WPB + wv) * wv_slot_doubles(t.NB);
    const int c2 = uni(wcount[2]), c1 = c2 + uni(wcount[1]), c0 = c1 + uni(wcount[0]);
    for (;;) {
        int idx = 0;
        if (lane == 0) idx = atomicAdd(wnext, 1);
        idx = uni(idx);
        if (idx >= c0) break;
        if (idx < c2)
            rc_wave_task<64, KR>(t, k, uni(wlist[2 * (size_t)cap + idx]), Wq, L, redo, nredo, acc, fixed_rk, maxrank,
                                 o, ovf, qn_dense);
        else if (idx < c1)
            rc_wave_task<48, KR>(t, k, uni(wlist[(size_t)cap + idx - c2]), Wq, L, redo, nredo, acc, fixed_rk, maxrank,
                                 o, ovf, qn_dense);
        else
            rc_wave_task<32, KR>(t, k, uni(wlist[idx - c1]), Wq, L, redo, nredo, acc, fixed_rk, maxrank, o, ovf,
                                 qn_dense);
    }
}

// wlist, wcount, redo: k_classify_wave's lists (cap entries each) and counters
int rc_wave_launch(hipStream_t st, int grid, const TLR &t, int k, const int *wlist, int cap, int *wcount, int *redo,
                   double *ws, double acc, int fixed_rk, int maxrank, const OpLog &o, int *ovf, const double *qn_dense)
{
    // tiles of up to 512 rows: 8 rows per lane in the panels (with 16 the two QR of a
    // tile of 270 rows took 0.28 of the 0.79 ms of the widest class)
    const auto f = t.NB <= 512 ? k_rc_wave<8> : k_rc_wave<WV_KMAX>;
    const size_t lds = sizeof(double) * WV_LDS * WV_WPB;
    HIPCHK(hipFuncSetAttribute((const void *)f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(f, dim3(grid), dim3(64 * WV_WPB), lds, st, t, k, wlist, cap, (const int *)wcount, wcount + 4, redo,
                       wcount + 8, ws, acc, fixed_rk, maxrank, o, ovf, qn_dense);
    return 0;
}
