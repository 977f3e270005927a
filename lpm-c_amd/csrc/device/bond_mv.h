// The finest operator's product over the bonds (tangent.hip, k_bond_form), shared by the AMG
// smoother and the CG.
#pragma once

#include "common.h"

// K x from the bond form (tangent.hip, k_bond_form) in two passes: the shell sums of every
// particle, then the bonds' terms with the partners' sums.  BF_W wavefronts share 64
// particles, each every BF_W-th bond, their partial sums added in order through LDS, as in
// slice_mv.h.  It reads D + 4 words a bond and pass (18 bonds) for the D * D + 1 of each of
// 59 stored blocks.  (FP32 at 1M, us: stored 388, sums 83 and product 138; at 216k 80, 15
// and 18; FP64 at 79k 58, 11.5 and 18.  3 wavefronts the same, 9 slower, with nontemporal
// loads 1% faster at 1M and 2-4% slower where the bonds fit the last-level cache.)  A step:
// 27k mixed 11.7 -> 11.1 ms, 79k FP64 39.8 -> 33.8, 1M mixed 249 -> 214.
#define BF_W 6
static_assert(BF_W >= 4, "a thread per entry of the sums and of the product");

// delta and the partner's entries of bond code cd.
template <int D, typename TX>
__device__ __forceinline__ TX bond_delta(int cd, const TX *a, const TX *xi, const TX *__restrict__ x, TX *dx)
{
    const int64_t j = cd >> 4;
    TX s = 0;
#pragma unroll
    for (int c = 0; c < D; c++)
    {
        const TX xj = x[j * D + c];
        dx[c] = xi[c] - (cd >> c & 1 ? (TX)0 : xj);
        s += a[c] * dx[c];
    }
    return s;
}

template <int NB, int D, typename TX>
__global__ __launch_bounds__(64 * BF_W) void k_bond_sums(int n, int nb_, const int *__restrict__ code,
                                                         const int *__restrict__ mask, const TX *__restrict__ v,
                                                         const TX *__restrict__ x, TX *__restrict__ ab, const int *done)
{
    if (done && *done)
        return;
    static_assert(NB % BF_W == 0, "whole trips");
    const int nb = NB ? NB : nb_;
    __shared__ TX sh[BF_W][4][64];
    const int l = threadIdx.x & 63, w = threadIdx.x >> 6, i = xcd_block() * 64 + l;
    const int trips = NB ? NB / BF_W : (nb - w + BF_W - 1) / BF_W;
    const int64_t plane = (int64_t)n * nb;
    TX A[2] = {0, 0}, B[2] = {0, 0};
    if (i < n)
    {
        TX xi[D];
        const int m = mask[i];
#pragma unroll
        for (int c = 0; c < D; c++)
            xi[c] = m >> c & 1 ? (TX)0 : x[(int64_t)i * D + c];
#pragma unroll 3
        for (int u = 0; u < trips; u++)
        {
            const int e = w + u * BF_W;
            const int64_t b = (int64_t)e * n + i;
            const int cd = code[b];
            TX a[D], dx[D];
#pragma unroll
            for (int c = 0; c < D; c++)
                a[c] = v[c * plane + b];
            const TX tv = v[D * plane + b];
            const TX s = bond_delta<D, TX>(cd, a, xi, x, dx);
            const bool s1 = cd & 8;
            A[0] += s1 ? (TX)0 : s, A[1] += s1 ? s : (TX)0;
            B[0] += s1 ? (TX)0 : tv * s, B[1] += s1 ? tv * s : (TX)0;
        }
    }
    sh[w][0][l] = A[0], sh[w][1][l] = B[0], sh[w][2][l] = A[1], sh[w][3][l] = B[1];
    __syncthreads();
    // thread t: entry t % 4 of particle t / 4 of the 64
    const int t = threadIdx.x, q = t & 3, il = t >> 2, ig = xcd_block() * 64 + il;
    if (t < 256 && ig < n)
    {
        TX s = 0;
#pragma unroll
        for (int k = 0; k < BF_W; k++)
            s += sh[k][q][il];
        ab[(int64_t)ig * 4 + q] = s;
    }
}

// (K x) of the work-group's 64 particles: entry t % D of particle t / D of them in tot[t],
// after a barrier; true on the threads that hold one.  Every thread must call it.
template <int NB, int D, typename TX>
__device__ __forceinline__ bool bond_rows(int n, int nb_, const int *__restrict__ code, const int *__restrict__ mask,
                                          const TX *__restrict__ v, const TX *__restrict__ dd,
                                          const TX *__restrict__ x, const TX *__restrict__ ab, TX nd, TX *tot)
{
    const int nb = NB ? NB : nb_;
    __shared__ TX sh[BF_W][D][64];
    const int l = threadIdx.x & 63, w = threadIdx.x >> 6, i = xcd_block() * 64 + l;
    const int trips = NB ? NB / BF_W : (nb - w + BF_W - 1) / BF_W;
    const int64_t plane = (int64_t)n * nb;
    TX acc[D];
#pragma unroll
    for (int c = 0; c < D; c++)
        acc[c] = 0;
    if (i < n)
    {
        const int m = mask[i];
        TX xi[D], own[4];
#pragma unroll
        for (int q = 0; q < 4; q++)
            own[q] = (TX)0.5 * ab[(int64_t)i * 4 + q];
#pragma unroll
        for (int c = 0; c < D; c++)
            xi[c] = m >> c & 1 ? (TX)0 : x[(int64_t)i * D + c];
#pragma unroll 3
        for (int u = 0; u < trips; u++)
        {
            const int e = w + u * BF_W;
            const int64_t b = (int64_t)e * n + i;
            const int cd = code[b], s1 = cd >> 3 & 1;
            TX a[D], dx[D];
#pragma unroll
            for (int c = 0; c < D; c++)
                a[c] = v[c * plane + b];
            const TX tv = v[D * plane + b], kp = v[(D + 1) * plane + b], gs = v[(D + 2) * plane + b];
            const TX *abj = ab + (int64_t)(cd >> 4) * 4 + 2 * s1;
            const TX Aj = abj[0], Bj = abj[1];
            const TX s = bond_delta<D, TX>(cd, a, xi, x, dx);
            const TX f = kp * s + (s1 ? own[3] : own[1]) + (TX)0.5 * Bj + tv * ((s1 ? own[2] : own[0]) + (TX)0.5 * Aj);
#pragma unroll
            for (int c = 0; c < D; c++)
                acc[c] += a[c] * f + gs * dx[c];
        }
    }
#pragma unroll
    for (int c = 0; c < D; c++)
        sh[w][c][l] = acc[c];
    __syncthreads();
    // thread t: entry t % D of particle t / D of the 64, so that the epilogue's accesses to
    // DOF vectors are contiguous
    const int t = threadIdx.x, c = t % D, il = t / D, ie = xcd_block() * 64 + il;
    const bool mine = t < 64 * D && ie < n;
    if (mine)
    {
        const int me = mask[ie];
        const TX *xe = x + (int64_t)ie * D;
        TX s = 0;
#pragma unroll
        for (int k = 0; k < BF_W; k++)
            s += sh[k][c][il];
#pragma unroll
        for (int k = 0; k < D; k++)
        {
            const int lo = c < k ? c : k, hi = c < k ? k : c; // upper triangle by rows
            s += dd[(int64_t)(lo * D - lo * (lo - 1) / 2 + hi - lo) * n + ie] * (me >> k & 1 ? (TX)0 : xe[k]);
        }
        tot[t] = me >> c & 1 ? nd * xe[c] : s;
    }
    __syncthreads();
    return mine;
}

// Algorithmic HBM bytes of a product with values of sv bytes: both passes' bonds, the shell
// sums written and read, x twice and two more vector streams.
static inline double bond_form_bytes(double sv)
{
    const double nb = (double)g.n * g.nb, D = g.dim;
    return nb * ((D + 1) * sv + 4) + nb * ((D + 3) * sv + 4) + (double)g.n * (8 + (8 + D * (D + 1) / 2 + 4 * D) * sv);
}
