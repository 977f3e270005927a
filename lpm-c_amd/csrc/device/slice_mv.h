// The block SpMV of a sliced-ELL matrix (64 rows per slice, slot-major), shared by the
// CG and the AMG smoother: the row sums (A x)_i, handed to the caller's epilogue.
#pragma once

#include "common.h"

// One slot of a row: the BR x BC block times the gathered entries of x.  The matrix
// streams through once and is read nontemporally, so that it does not evict the
// gathered vector window from L2.
template <int BR, int BC, typename TV, typename TX>
__device__ __forceinline__ void slice_mac(const TV *__restrict__ kb, const TX *__restrict__ x, int m, TX *acc)
{
    TX xm[BC];
#pragma unroll
    for (int c = 0; c < BC; c++)
        xm[c] = x[(int64_t)m * BC + c];
#pragma unroll
    for (int r = 0; r < BR; r++)
#pragma unroll
        for (int c = 0; c < BC; c++)
            acc[r] += (TX)__builtin_nontemporal_load(kb + (r * BC + c) * 64) * xm[c];
}

// Wavefronts per slice: wavefront w takes the slots w, w + W, ..., and the first one adds
// the partial sums in wavefront order.  With one wavefront per slice a launch takes the
// time of one row's chain of slots however small the matrix, and keeps fewer loads in
// flight at any size.  The CG's SpMV on SC lattices, us (FP64 / FP32; W = 1 with its
// four FP32 slots loaded ahead):
//   rows       512       8,000      27,000      79,507     216,000    405,224   1,000,000
//   W = 1   21 / 9    58 / 21     61 / 23     80 / 39    186 / 87   349 / 166   839 / 412
//   W = 4  7.5 / 4.6  16 / 10     23 / 14     59 / 31    169 / 83   337 / 158   830 / 411
//   W = 16 7.6 / 4.2  12 / 7.1    23 / 13     58 / 30    166 / 80   329 / 153   804 / 388
// (5.7 and 6.3 TB/s at 1M.)  Short rows leave 16 wavefronts one slot each: the
// prolongator of 1M (13 slots a row) takes 159, 140, 138 and 167 us at W = 1, 4, 8 and
// 16, the 2x2 tangent of 55,000 rows (19 slots) 12.4, 8.7, 8.9 and 9.3 us.
static inline bool slice_wide(int64_t nslots, int nslices) { return nslots >= 32 * (int64_t)nslices; } // W = 16, else 4

// acc = (A x)_i of the thread's row position i; true on the threads that hold one (the
// first wavefront of the W that share the slice, a work-group).  s: the slice; sh: W *
// BR * 64 entries of LDS.  Every thread of the work-group must call it.
template <int BR, int BC, typename TV, typename TX, int W>
__device__ __forceinline__ bool slice_rows(int nr, int s, const int *__restrict__ sptr, const int *__restrict__ col,
                                           const TV *__restrict__ val, const TX *__restrict__ x, int &i, TX *acc,
                                           TX *sh)
{
    constexpr int U = 2; // slots loaded ahead per step
    const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
    i = s * 64 + l;
#pragma unroll
    for (int r = 0; r < BR; r++)
        acc[r] = 0;
    if (i < nr) // the positions beyond nr hold no slots to add
    {
        const int k1 = sptr[s + 1];
        int k = sptr[s] + w;
        for (; k + (U - 1) * W < k1; k += U * W)
        {
            int m[U];
#pragma unroll
            for (int u = 0; u < U; u++)
                m[u] = __builtin_nontemporal_load(col + (int64_t)(k + u * W) * 64 + l);
#pragma unroll
            for (int u = 0; u < U; u++)
                slice_mac<BR, BC, TV, TX>(val + (int64_t)(k + u * W) * BR * BC * 64 + l, x, m[u], acc);
        }
        for (; k < k1; k += W)
            slice_mac<BR, BC, TV, TX>(val + (int64_t)k * BR * BC * 64 + l, x,
                                      __builtin_nontemporal_load(col + (int64_t)k * 64 + l), acc);
    }
#pragma unroll
    for (int r = 0; r < BR; r++)
        sh[(w * BR + r) * 64 + l] = acc[r];
    __syncthreads();
    if (w != 0)
        return false;
#pragma unroll
    for (int r = 0; r < BR; r++)
    {
        TX t = sh[r * 64 + l];
#pragma unroll
        for (int k = 1; k < W; k++)
            t += sh[(k * BR + r) * 64 + l];
        acc[r] = t;
    }
    return i < nr;
}
