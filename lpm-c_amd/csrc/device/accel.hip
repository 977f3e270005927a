// Anderson acceleration of the modified-Newton iteration of a load step.
//
// The reference's Newton loop (src/lpmc_project.c:424-447) is the fixed-point
// iteration u <- u + d(u) with d(u) = K^-1 R(u), K the elastic tangent assembled once
// per step.  In plastic flow the elastic tangent over-estimates the stiffness by
// E/H and that iteration contracts by nearly 1 per step.  Anderson's method (type
// II, Walker & Ni, SIAM J. Numer. Anal. 49 (2011) 1715-1735) keeps the last m
// differences dU_j = u_j+1 - u_j, dF_j = d_j+1 - d_j and moves to
//     u_k+1 = u_k + d_k - sum_j gamma_j (dU_j + dF_j),
//     gamma = argmin | d_k - sum_j gamma_j dF_j |_2,
// which has the same fixed points (R(u) = 0) as the plain iteration.  Constrained
// DOFs have d = 0 in every iterate, so every difference is 0 there and the
// prescribed displacements are untouched.
//
// The same mixing serves the fixed-point iteration of the adjoint solve on a DOF
// vector (lpmx_aa_*).
//
// All on the device: the history lives in DOF vectors (n*dim doubles); the 2m dot
// products of an iteration are one pass with per-block partials and a fixed-order total,
// so the result is deterministic; one work-group then solves the m x m least-squares
// system, by LDL^T of the Tikhonov-regularised Gram matrix, and leaves the
// coefficients in device memory for the mix, so that an iteration does not wait for the
// host here.
#include <math.h>
#include <string.h>

#include "common.h"

#define AA_MAX 32

// dC_j = dU_j + dF_j (the iterate and correction differences, summed: the mix uses
// only their sum) and dF_j (the Gram matrix and right-hand side use the corrections),
// stored in FP64, or in FP32 for the mixed-precision Newton loop (the iterate, the
// corrections and the dot products stay FP64).
template <typename T>
struct AaPtrsT
{
    T *dC[AA_MAX], *dF[AA_MAX];
};
typedef AaPtrsT<double> AaPtrs;
typedef AaPtrsT<float> AaPtrs32;

// One Anderson history over DOF vectors of n*dim entries.  The iterate itself may
// be strided: entry (i, c) of the iterate is at xs*i + c (xs = 3 for positions,
// xs = dim for a DOF vector).
struct AaHist
{
    int n = 0, dim = 0, depth = 0, cnt = 0, next = 0, have_prev = 0, f32 = 0;
    double *u_prev = nullptr, *f_prev = nullptr, *parts = nullptr;
    double *gram = nullptr, *gam = nullptr; // AA_MAX^2 dot products of the dF, coefficients
    int *flag = nullptr;                    // pinned host: 1 solved, 0 degenerate Gram matrix
    int pending = 0;                        // a solve whose flag has not been looked at
    AaPtrs P{};
    AaPtrs32 P32{};
};

static AaHist A; // the Newton loop's history

// work-groups of the dot pass: three per CU (256 CUs).  At the kernel's 177 VGPRs
// (two waves per SIMD) that is 1.5 resident rounds; two per CU (one round) took 0.082
// against 0.0995 ms at 1M, but its other grouping of the partial sums moved the
// iterates enough that one step of the 216k perturbed-parameter history at Newton
// 1e-10 stalled at its cap, so the grouping stays.
static const int AA_GRID = 768;

static void aa_release(AaHist *a)
{
    for (int j = 0; j < AA_MAX; j++)
    {
        void *ps[] = {a->P.dC[j], a->P.dF[j], a->P32.dC[j], a->P32.dF[j]};
        for (void *p : ps)
            if (p)
                hipFree(p);
    }
    void *ps[] = {a->u_prev, a->f_prev, a->parts, a->gram, a->gam};
    for (void *p : ps)
        if (p)
            hipFree(p);
    if (a->flag)
        hipHostFree(a->flag);
    *a = AaHist();
}

void lpmx_accel_free(void) { aa_release(&A); }

// u = x - d (the iterate the update started from); with a previous iterate the new
// differences go to slot s; then (u, d) become the previous iterate.
template <typename T>
__global__ void k_aa_push(int n, int dim, int xs, const double *__restrict__ x, const double *__restrict__ d,
                          double *__restrict__ u_prev, double *__restrict__ f_prev, T *__restrict__ dC,
                          T *__restrict__ dF, int have_prev)
{
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (t >= (int64_t)n * dim)
        return;
    const int64_t i = t / dim;
    const int c = (int)(t - i * dim);
    const double u = x[xs * i + c] - d[t];
    if (have_prev)
    {
        const double du = u - u_prev[t], df = d[t] - f_prev[t];
        dC[t] = (T)(du + df);
        dF[t] = (T)df;
    }
    u_prev[t] = u;
    f_prev[t] = d[t];
}

// Partials of dF_s . dF_j and dF_j . d for the cnt active slots: parts[b][2*AA_MAX].
// Every slot is read: the host points the slots from cnt on at slot s (cached after
// its first read), so the AA_MAX loads of an element are issued together.  With the
// loads under `j < cnt` each one was waited for before the next was issued.
template <typename T>
__global__ __launch_bounds__(256) void k_aa_dots(int64_t m, AaPtrsT<T> P, int cnt, int s,
                                                 const double *__restrict__ d, double *parts)
{
    double g[AA_MAX], h[AA_MAX];
#pragma unroll
    for (int j = 0; j < AA_MAX; j++)
        g[j] = 0.0, h[j] = 0.0;
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < m; t += (int64_t)gridDim.x * blockDim.x)
    {
        const double fs = (double)P.dF[s][t], dt = d[t];
        double f[AA_MAX];
#pragma unroll
        for (int j = 0; j < AA_MAX; j++)
            f[j] = (double)P.dF[j][t];
#pragma unroll
        for (int j = 0; j < AA_MAX; j++)
        {
            g[j] += fs * f[j];
            h[j] += f[j] * dt;
        }
    }
    // wave sums of the 2 AA_MAX values at once: at each step of the butterfly a lane keeps
    // one half of its values and gives the other half to its partner, so lane q ends with
    // the sum of value q (63 exchanges instead of 6 for each of the 64 values; the sums
    // are those of the full butterfly, bit for bit).  Then the work-group totals in wave
    // order through LDS.
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    static_assert(2 * AA_MAX == 64, "a value per lane");
    double v[AA_MAX];
#pragma unroll
    for (int j = 0; j < AA_MAX; j++)
    {
        const bool up = lane & 32;
        v[j] = (up ? h[j] : g[j]) + __shfl_xor(up ? g[j] : h[j], 32, 64);
    }
#pragma unroll
    for (int o = 16; o >= 1; o >>= 1)
    {
        const bool up = lane & o;
#pragma unroll
        for (int j = 0; j < AA_MAX / 2; j++)
            if (j < o)
                v[j] = (up ? v[j + o] : v[j]) + __shfl_xor(up ? v[j] : v[j + o], o, 64);
    }
    __shared__ double wsum[4][2 * AA_MAX];
    wsum[w][lane] = v[0];
    __syncthreads();
    const int q = threadIdx.x;
    if (q < 2 * AA_MAX)
    {
        double t = 0.0;
        for (int k = 0; k < (int)(blockDim.x >> 6); k++)
            t += wsum[k][q];
        parts[(int64_t)blockIdx.x * 2 * AA_MAX + q] = t;
    }
}

// 1 / d of a positive finite d by two Newton steps from the hardware's estimate (error
// below 2 ulp): the factorisation is a chain of them, and a division is four times as long.
__device__ __forceinline__ double reciprocal(double d)
{
    double r = __builtin_amdgcn_rcp(d);
    r = fma(fma(-d, r, 1.0), r, r);
    return fma(fma(-d, r, 1.0), r, r);
}

// The totals of the np partials, row and column s of the Gram matrix, and gamma =
// (G + lam I)^-1 h by an LDL^T factorisation of the cnt x cnt system; one work-group, a
// thread per entry of the lower triangle, with the right-hand side as its row AA_MAX.  A
// step publishes one column in LDS (each its own, so one barrier per step) and updates
// the entries right of it; the back substitution is one wavefront's.  *flag gets 0 and
// gamma zeros when the matrix is not positive definite.  A chain of barriers, LDS reads
// and reciprocals bounds it.  (Averages over a step of 8,000 particles: Cholesky with a
// thread per entry of the square and three barriers per step 17 us, this with one partial
// at a time and divisions 12, as it is 10; over the brittle shear of 58,000 particles, with
// 455 partials, 25 and 16.  Two columns per barrier and a back substitution from
// registers were no faster.)
#define AA_ENTRIES ((AA_MAX + 1) * (AA_MAX + 2) / 2)
#define AA_SOLVE_T 576
#define AA_BATCH 16 // partials a thread has in flight: one memory latency per batch
static_assert(AA_SOLVE_T >= AA_ENTRIES && AA_SOLVE_T % 64 == 0, "a thread per entry, whole wavefronts");
__global__ __launch_bounds__(AA_SOLVE_T) void k_aa_solve(const double *parts, int np, int cnt, int s,
                                                         double *__restrict__ gram, double *__restrict__ gam,
                                                         int *flag)
{
    __shared__ double T[AA_SOLVE_T / 64][2 * AA_MAX], col[AA_MAX][AA_MAX + 2], tot[2 * AA_MAX], diag[AA_MAX];
    const int t = threadIdx.x;
    // entry (i, k) of the triangle
    int i = (int)((sqrtf(8.0f * t + 1.0f) - 1.0f) * 0.5f);
    i += (i + 1) * (i + 2) / 2 <= t;
    i -= i * (i + 1) / 2 > t;
    const int k = t - i * (i + 1) / 2;
    const bool gramian = i < cnt; // k <= i
    double a = gramian ? gram[i * AA_MAX + k] : 0.0;
    {
        const int q = t & 63, c = t >> 6;
        double sum = 0.0;
        for (int b0 = c; b0 < np; b0 += AA_BATCH * (AA_SOLVE_T / 64))
        {
            double p[AA_BATCH];
#pragma unroll
            for (int u = 0; u < AA_BATCH; u++)
            {
                const int b = b0 + u * (AA_SOLVE_T / 64);
                p[u] = parts[(int64_t)(b < np ? b : np - 1) * 2 * AA_MAX + q];
            }
#pragma unroll
            for (int u = 0; u < AA_BATCH; u++)
                if (b0 + u * (AA_SOLVE_T / 64) < np)
                    sum += p[u];
        }
        T[c][q] = sum;
    }
    __syncthreads();
    if (t < 2 * AA_MAX)
    {
        double sum = 0.0;
        for (int c = 0; c < AA_SOLVE_T / 64; c++)
            sum += T[c][t];
        tot[t] = sum;
    }
    __syncthreads();
    if (gramian && (i == s || k == s))
    {
        a = tot[i == s ? k : i];
        gram[i * AA_MAX + k] = a;
    }
    else if (i == AA_MAX && k < cnt)
        a = tot[AA_MAX + k];
    if (gramian && i == k)
        diag[i] = a;
    __syncthreads();
    double dmax = 0.0;
    for (int j = 0; j < cnt; j++)
        dmax = fmax(dmax, diag[j]);
    bool ok = dmax > 0.0 && isfinite(dmax);
    if (gramian && i == k)
        a += 1e-12 * dmax;
    for (int j = 0; j < cnt; j++)
    {
        if (k == j && i <= AA_MAX)
            col[j][i] = a;
        __syncthreads();
        const double d = col[j][j];
        ok = ok && d > 0.0 && isfinite(d);
        if (k > j && i <= AA_MAX)
            a -= col[j][i] * (col[j][k] * reciprocal(d));
    }
    __syncthreads();
    if (t >= 64)
        return;
    // lane j: x_j = (y_j - sum over i > j of col[j][i] x_i) / d_j
    const int l = t < AA_MAX ? t : 0;
    double x = l < cnt ? col[l][AA_MAX] / col[l][l] : 0.0;
    const double r = l < cnt ? 1.0 / col[l][l] : 0.0;
    for (int j = cnt - 1; j > 0; j--)
    {
        const double xj = __shfl(x, j, 64);
        if (t < j)
            x -= col[t][j] * r * xj;
    }
    if (__any(t < cnt && !isfinite(x)))
        ok = false;
    if (t < AA_MAX)
        gam[t] = ok && t < cnt ? x : 0.0;
    if (t == 0)
        *flag = ok;
}

// x -= sum_j gamma_j dC_j.  Every slot is read, as in k_aa_dots: the host points the
// slots from cnt on at slot s, with gamma_j = +0 there (everywhere when the Gram matrix
// was degenerate: x stays the plain iterate), so their terms are +-0 and leave the sum's
// bits as they are, and the AA_MAX loads of an element are issued
// together.
template <typename T>
__global__ void k_aa_mix(int n, int dim, int xs, double *__restrict__ x, AaPtrsT<T> P,
                         const double *__restrict__ gam)
{
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (t >= (int64_t)n * dim)
        return;
    double s = 0.0;
#pragma unroll
    for (int j = 0; j < AA_MAX; j++)
        s += gam[j] * (double)P.dC[j][t];
    const int64_t i = t / dim;
    const int c = (int)(t - i * dim);
    x[xs * i + c] -= s;
}

// x = u_prev + f_prev: the plain iterate of the last update.
__global__ void k_aa_plain(int n, int dim, int xs, double *__restrict__ x, const double *__restrict__ u_prev,
                           const double *__restrict__ f_prev)
{
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (t >= (int64_t)n * dim)
        return;
    const int64_t i = t / dim;
    const int c = (int)(t - i * dim);
    x[xs * i + c] = u_prev[t] + f_prev[t];
}

// Start a new history (a new load step, or a re-solve after bond breakage: the
// tangent, and with it the map, has changed).
static int aa_begin(AaHist *a, int depth, int f32 = 0)
{
    if (depth < 0 || depth > AA_MAX)
        return lpmx_fail(LPMX_ERR_ARG, "acceleration depth %d outside 0..%d", depth, AA_MAX);
    if (a->n != g.n || a->dim != g.dim)
        aa_release(a);
    const int64_t m = (int64_t)g.n * g.dim;
    for (int j = 0; j < depth; j++)
    {
        if (f32)
        {
            if (!a->P32.dC[j])
                HIPCHK(dev_malloc(&a->P32.dC[j], sizeof(float) * m));
            if (!a->P32.dF[j])
                HIPCHK(dev_malloc(&a->P32.dF[j], sizeof(float) * m));
        }
        else
        {
            if (!a->P.dC[j])
                HIPCHK(dev_malloc(&a->P.dC[j], sizeof(double) * m));
            if (!a->P.dF[j])
                HIPCHK(dev_malloc(&a->P.dF[j], sizeof(double) * m));
        }
    }
    a->f32 = f32;
    if (depth > 0 && !a->u_prev)
    {
        HIPCHK(dev_malloc(&a->u_prev, sizeof(double) * m));
        HIPCHK(dev_malloc(&a->f_prev, sizeof(double) * m));
        HIPCHK(dev_malloc(&a->parts, sizeof(double) * AA_GRID * 2 * AA_MAX));
        HIPCHK(dev_malloc(&a->gram, sizeof(double) * AA_MAX * AA_MAX));
        HIPCHK(dev_malloc(&a->gam, sizeof(double) * AA_MAX));
        HIPCHK(hipHostMalloc(&a->flag, sizeof(int)));
    }
    a->n = g.n, a->dim = g.dim;
    a->depth = depth;
    a->cnt = a->next = a->have_prev = a->pending = 0;
    return LPMX_OK;
}

static void aa_forget(AaHist *a) { a->cnt = a->next = 0; }

static int aa_revert(AaHist *a, double *x, int xs)
{
    if (a->depth == 0 || !a->have_prev)
        return LPMX_OK;
    hipLaunchKernelGGL(k_aa_plain, dim3(nblocks((int64_t)g.n * g.dim)), dim3(LPMX_BLOCK), 0, g_stream, g.n, g.dim, xs,
                       x, a->u_prev, a->f_prev);
    LAUNCHCHK();
    aa_forget(a);
    return LPMX_OK;
}

// After a synchronisation with the stream: whether the last mix took place.  A degenerate
// history kept the plain iterate, and its differences start afresh.
static int aa_check(AaHist *a)
{
    if (!a->pending)
        return 0;
    a->pending = 0;
    if (*(volatile int *)a->flag)
        return 1;
    aa_forget(a);
    return 0;
}

// The point that the iterate after this update records: the previous iterate and
// correction, and the slot of its differences.  The caller has synchronised with the
// stream since the last mix (for its residual norm).
static void aa_point(AaHist *a, AaPush *p)
{
    aa_check(a);
    const int s = a->next;
    p->on = a->depth > 0;
    p->u_prev = a->u_prev, p->f_prev = a->f_prev, p->f32 = a->f32, p->have_prev = a->have_prev;
    p->dC = a->f32 ? (void *)a->P32.dC[s] : (void *)a->P.dC[s];
    p->dF = a->f32 ? (void *)a->P32.dF[s] : (void *)a->P.dF[s];
}

// With the point recorded (aa_point): move x to the accelerated iterate.  *mixed = 1 when
// a mix is queued.
static int aa_mix(AaHist *a, double *x, int xs, const double *d, int *mixed)
{
    *mixed = 0;
    if (a->depth == 0)
        return LPMX_OK;
    const int n = g.n, dim = g.dim;
    const int64_t m = (int64_t)n * dim;
    const int nb = nblocks(m);
    const int s = a->next;
    if (!a->have_prev)
    {
        a->have_prev = 1;
        return LPMX_OK;
    }
    if (a->cnt < a->depth)
        a->cnt++;
    a->next = (a->next + 1) % a->depth;
    const int cnt = a->cnt;
    // the unused slots read slot s (written just now, so finite and cached)
    AaPtrs32 Q32 = a->P32;
    AaPtrs Q64 = a->P;
    for (int j = cnt; j < AA_MAX; j++)
    {
        Q32.dF[j] = a->P32.dF[s], Q32.dC[j] = a->P32.dC[s];
        Q64.dF[j] = a->P.dF[s], Q64.dC[j] = a->P.dC[s];
    }
    const int np = nb < AA_GRID ? nb : AA_GRID; // no work-group without an entry
    if (a->f32)
        hipLaunchKernelGGL(k_aa_dots<float>, dim3(np), dim3(256), 0, g_stream, m, Q32, cnt, s, d, a->parts);
    else
        hipLaunchKernelGGL(k_aa_dots<double>, dim3(np), dim3(256), 0, g_stream, m, Q64, cnt, s, d, a->parts);
    hipLaunchKernelGGL(k_aa_solve, dim3(1), dim3(AA_SOLVE_T), 0, g_stream, a->parts, np, cnt, s, a->gram, a->gam,
                       a->flag);
    if (a->f32)
        hipLaunchKernelGGL(k_aa_mix<float>, dim3(nb), dim3(LPMX_BLOCK), 0, g_stream, n, dim, xs, x, Q32, a->gam);
    else
        hipLaunchKernelGGL(k_aa_mix<double>, dim3(nb), dim3(LPMX_BLOCK), 0, g_stream, n, dim, xs, x, Q64, a->gam);
    LAUNCHCHK();
    a->pending = 1;
    *mixed = 1;
    return LPMX_OK;
}

// After an update has set x = u_k + d_k: record the iterate and, with a history,
// move x to the accelerated iterate.
static int aa_step(AaHist *a, double *x, int xs, const double *d, int *mixed)
{
    AaPush p;
    aa_point(a, &p);
    if (p.on)
    {
        const int nb = nblocks((int64_t)g.n * g.dim);
        if (p.f32)
            hipLaunchKernelGGL(k_aa_push<float>, dim3(nb), dim3(LPMX_BLOCK), 0, g_stream, g.n, g.dim, xs, x, d,
                               p.u_prev, p.f_prev, (float *)p.dC, (float *)p.dF, p.have_prev);
        else
            hipLaunchKernelGGL(k_aa_push<double>, dim3(nb), dim3(LPMX_BLOCK), 0, g_stream, g.n, g.dim, xs, x, d,
                               p.u_prev, p.f_prev, (double *)p.dC, (double *)p.dF, p.have_prev);
        LAUNCHCHK();
    }
    return aa_mix(a, x, xs, d, mixed);
}

// --------------------------------------------------------- the Newton loop's -----
// precision LPMX_MIXED keeps the differences in FP32
int lpmx_accel_begin(int depth, int precision) { return aa_begin(&A, depth, precision == LPMX_MIXED); }
// Keep the history's differences and drop only its last point: the next step records
// a new point without a difference across it (a re-solve of the same load step after
// bond breakage, whose map differs from the last one by the broken bonds).
void lpmx_accel_rebase(void) { A.have_prev = 0; }
void lpmx_accel_forget(void) { aa_forget(&A); }
// Revert xyz to the plain iterate of the last solve and forget the history.
int lpmx_accel_revert(void) { return aa_revert(&A, g.x, 3); }
// After a solve has set xyz = u_k + d_k (d_k in g.disp).
int lpmx_accel_step(int *mixed) { return aa_step(&A, g.x, 3, g.disp, mixed); }
int lpmx_accel_push(AaPush *p)
{
    aa_point(&A, p);
    return LPMX_OK;
}
int lpmx_accel_mix(int *mixed) { return aa_mix(&A, g.x, 3, g.disp, mixed); }
// After the next synchronisation: whether the mix that lpmx_accel_step queued took place.
int lpmx_accel_check(void) { return aa_check(&A); }

// ------------------------------------------------------------ other histories ----
AaHist *lpmx_aa_create(void) { return new AaHist(); }
void lpmx_aa_destroy(AaHist *a)
{
    if (a)
    {
        aa_release(a);
        delete a;
    }
}
int lpmx_aa_begin(AaHist *a, int depth) { return aa_begin(a, depth); }
int lpmx_aa_step(AaHist *a, double *x, const double *d, int *mixed) { return aa_step(a, x, g.dim, d, mixed); }
