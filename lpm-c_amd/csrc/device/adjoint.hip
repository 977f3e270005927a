// Reverse mode of the J2 load path on the device: vector-Jacobian products of one
// force evaluation (the J2 law of src/constitutive.c:466-686 as evaluated by
// k_j2_particle / k_j2_force), and the discrete adjoint of a load history built on
// them (lpmx_adjoint_run).
//
// A force evaluation maps positions x, the slot-0 state s = (dLp, beta, alpha) and
// the parameters (per-particle modulus factor e, yield stress sigmay, H) to the
// internal force Pin and the slot-2 state.  Its reverse sweep, for seeds on Pin and
// the slot-2 state, runs in two kernels of a thread per bond, both deterministic
// (gathers, no atomics; sums over a particle's bonds in slot order through LDS, as in
// bondforce.hip):
//   k_vjp_bonds   adjoint of F_ij (= Pbar_i . cs_ij), the geometric term of Pin = sum cs
//                 F and the bond-constant adjoints of F; the adjoints of the second-pass
//                 stretches and sums from both ends' forces; then the second stretch
//                 pass, radial return, trial stress and first stretch pass in reverse,
//                 recomputed in the forward's order (so every yield decision is the
//                 forward's);
//   k_vjp_gather  positions from the bond-vector adjoints (x_i - x_q), modulus factor
//                 from the bond constants (SC averages both ends).
#include <math.h>
#include <string.h>

#include <vector>

#include "common.h"

#define BI(j, i) ((int64_t)(j) * v.n + (i))


struct AdjWork
{
    double *gb = nullptr, *Knb = nullptr, *Tvb = nullptr, *c44b = nullptr;
    int64_t cap = 0;
};
static AdjWork AW;

void lpmx_adjoint_free_work(void)
{
    void *ps[] = {AW.gb, AW.Knb, AW.Tvb, AW.c44b};
    for (void *p : ps)
        if (p)
            hipFree(p);
    AW = AdjWork();
}

static int adj_work(void)
{
    const int64_t nbn = (int64_t)g.n * g.nb;
    if (AW.cap == nbn && AW.gb)
        return LPMX_OK;
    lpmx_adjoint_free_work();
    HIPCHK(dev_malloc(&AW.gb, sizeof(double) * 3 * nbn));
    HIPCHK(dev_malloc(&AW.Knb, sizeof(double) * nbn));
    HIPCHK(dev_malloc(&AW.Tvb, sizeof(double) * nbn));
    HIPCHK(dev_malloc(&AW.c44b, sizeof(double) * g.n));
    AW.cap = nbn;
    return LPMX_OK;
}

__device__ __forceinline__ double vjp_opp(const DV &v, int i, int j)
{
    if (v.nbcur[i] == v.nb)
        return 0.5;
    const int o = v.opp[BI(j, i)];
    if (o < 0)
        return 1.0;
    return v.db[BI(o, i)] <= LPMX_EPS ? 1.0 : 0.5;
}

__device__ __forceinline__ void cc6(double cx, double cy, double cz, double *o)
{
    o[0] = cx * cx, o[1] = cy * cy, o[2] = cz * cz, o[3] = cy * cz, o[4] = cx * cz, o[5] = cx * cy;
}

__device__ __forceinline__ void cc6_bar(double cx, double cy, double cz, const double *ob, double *cb)
{
    cb[0] += 2 * cx * ob[0] + cz * ob[4] + cy * ob[5];
    cb[1] += 2 * cy * ob[1] + cz * ob[3] + cx * ob[5];
    cb[2] += 2 * cz * ob[2] + cy * ob[3] + cx * ob[4];
}

// Position adjoint of a bond from the adjoints of its distance (disb) and unit vector
// (cb): d(dis)/dx_i = c, dc/dx_i = (I - c c^T)/dis.  Linear in (disb, cb), so each
// reverse pass adds its own part.
__device__ __forceinline__ void vjp_geom(double *gb, const double *c, double dis, double disb, const double *cb)
{
    const double dot = c[0] * cb[0] + c[1] * cb[1] + c[2] * cb[2];
    gb[0] += disb * c[0] + (cb[0] - dot * c[0]) / dis;
    gb[1] += disb * c[1] + (cb[1] - dot * c[1]) / dis;
    gb[2] += disb * c[2] + (cb[2] - dot * c[2]) / dis;
}

#define VT 32 // particles per work-group

// Sum over the slots of particle p's terms.
template <int NB>
__device__ __forceinline__ double vjp_sum(const double (*t)[VT], int nb, int p)
{
    double s = 0.0;
    if (NB)
    {
#pragma unroll
        for (int j = 0; j < NB; j++)
            s += t[j][p];
    }
    else
        for (int j = 0; j < nb; j++)
            s += t[j][p];
    return s;
}

// The same over the bonds of one shell, each bond's own term and then its partner's
// (null: none).
template <int NB>
__device__ __forceinline__ double vjp_shell_sum(const double (*t)[VT], const double (*u)[VT],
                                                const unsigned char (*sh)[VT], int shell, int nb, int p)
{
    double s = 0.0;
#pragma unroll NB ? NB : 1
    for (int j = 0; j < (NB ? NB : nb); j++)
    {
        const bool in = sh[j][p] == shell;
        s += in ? t[j][p] : 0.0;
        if (u)
            s += in ? u[j][p] : 0.0;
    }
    return s;
}

// Everything per bond and per particle up to the gather of both ends.  The bond's
// geometry, stretches and constants are read or formed once and stay in the thread's
// registers through the four reverse passes, and the partner's force adjoint is
// recomputed from its seed; one thread per particle walked its bonds six times (its
// three kernels took 173, 27 and 23 us for 8,000 particles of 18 bonds, this one takes 16).
template <int NB>
__global__ __launch_bounds__(VT *(NB ? NB : LPMX_MAXNB)) void k_vjp_bonds(DV v, VjpIO io, AdjWork a)
{
    const int nb = NB ? NB : v.nb;
    __shared__ double T[6][NB ? NB : LPMX_MAXNB][VT];
    __shared__ unsigned char sh[NB ? NB : LPMX_MAXNB][VT];
    __shared__ double AB[8][VT], D[6][VT];
    const int p = threadIdx.x % VT, j = threadIdx.x / VT, n = v.n, i = blockIdx.x * VT + p, nt = VT * nb;
    const int64_t b = (int64_t)j * n + i, NBn = (int64_t)n * v.nb;
    bool bond = false, rev = false;
    int s = 0;
    double c[3] = {0, 0, 0}, gb[3] = {0, 0, 0}, dis = 1, L0 = 0, tv = 0, kn = 0, dw = 0, db = 0, dl = 0, w = 0;
    double t = 0, tr = 0, tvr = 0, knr = 0, Knb = 0, Tvb = 0, d2b = 0;
    if (i < n)
    {
        db = v.db[b], d2b = io.dLp2b[b];
        bond = j < v.nb0[i];
    }
    if (bond)
    {
        const int q = v.nbr[b], r = v.rev[b];
        s = v.nsign[b];
        rev = r >= 0;
        L0 = v.L0[b], tv = v.Tv[b], kn = v.Kn[b], dw = v.dw[b];
        const double dx = v.x[3 * i] - v.x[3 * q], dy = v.x[3 * i + 1] - v.x[3 * q + 1],
                     dz = v.x[3 * i + 2] - v.x[3 * q + 2];
        dis = sqrt(dx * dx + dy * dy + dz * dz);
        c[0] = dx / dis, c[1] = dy / dis, c[2] = dz / dis;
        dl = dis - L0;
        dl -= v.dLp0[b];
        dl *= db;
        w = vjp_opp(v, i, j) / v.volume * L0;
        // force F_ij of the evaluation (v.F, v.dLave, v.A, v.Bt hold it)
        const double p0 = io.Pb[3 * i], p1 = io.Pb[3 * i + 1], p2 = io.Pb[3 * i + 2], F = v.F[b];
        const double fb = p0 * c[0] + p1 * c[1] + p2 * c[2];
        const double bx = p0 * F, by = p1 * F, bz = p2 * F;
        const double dot = c[0] * bx + c[1] * by + c[2] * bz;
        gb[0] = (bx - dot * c[0]) / dis, gb[1] = (by - dot * c[1]) / dis, gb[2] = (bz - dot * c[2]) / dis;
        t = fb * dw;
        Knb = t * 2.0 * v.dLave[b];
        Tvb = t * 0.5 * (v.A[(int64_t)s * n + i] + v.A[(int64_t)s * n + q]);
        if (rev)
        {
            const int64_t br = (int64_t)r * n + q;
            const double fr = -(io.Pb[3 * q] * c[0] + io.Pb[3 * q + 1] * c[1] + io.Pb[3 * q + 2] * c[2]);
            tr = fr * v.dw[br], tvr = v.Tv[br], knr = v.Kn[br];
        }
    }
    sh[j][p] = (unsigned char)s;
    T[0][j][p] = t * 0.5 * tv, T[1][j][p] = tr * 0.5 * tvr;
    T[2][j][p] = t * 0.5, T[3][j][p] = tr * 0.5;
    T[4][j][p] = dl, T[5][j][p] = tv * dl;
    __syncthreads();
    // sums of the adjoints of the second-pass stretches, from both ends' forces (A2b,
    // B2b), and the forward's first-pass sums (A1, B1)
    for (int k = threadIdx.x; k < 8 * VT; k += nt)
    {
        const int kind = k / VT, shell = kind & 1, pp = k % VT;
        const double(*own)[VT] = kind < 2 ? T[0] : kind < 4 ? T[2] : kind < 6 ? T[4] : T[5];
        const double(*par)[VT] = kind < 2 ? T[1] : kind < 4 ? T[3] : nullptr;
        AB[kind][pp] = vjp_shell_sum<NB>(own, par, sh, shell, nb, pp);
    }
    __syncthreads();
    const double A2b = AB[s][p], B2b = AB[2 + s][p], A1 = AB[4 + s][p], B1 = AB[6 + s][p];
    double Ftr = 2.0 * kn * dl + B1 + tv * A1;
    Ftr *= dw;
    {
        const double f = w * Ftr;
        T[0][j][p] = f * c[0] * c[0], T[1][j][p] = f * c[1] * c[1], T[2][j][p] = f * c[2] * c[2];
        T[3][j][p] = f * c[1] * c[2], T[4][j][p] = f * c[0] * c[2], T[5][j][p] = f * c[0] * c[1];
    }
    __syncthreads();
    for (int k = threadIdx.x; k < 6 * VT; k += nt)
        D[k / VT][k % VT] = vjp_sum<NB>(T[k / VT], nb, k % VT);
    __syncthreads();
    // the particle's radial return, by its slot-0 thread
    double sl[6] = {0, 0, 0, 0, 0, 0}, dep[6] = {0, 0, 0, 0, 0, 0}, seq = 0, alpha0 = 0, c44 = 0, yf = 0, dlam = 0;
    const double H = v.H, xi = v.xi;
    bool plastic = false;
    const bool lead = j == 0 && i < n;
    if (lead)
    {
        for (int k = 0; k < 6; k++)
            sl[k] = D[k][p];
        const double tmp = 1.0 / 3.0 * (sl[0] + sl[1] + sl[2]);
        for (int k = 0; k < 3; k++)
            sl[k] -= tmp;
        for (int k = 0; k < 6; k++)
            sl[k] -= v.beta0[(int64_t)k * n + i];
        for (int k = 0; k < 6; k++)
            seq += k < 3 ? sl[k] * sl[k] : 2.0 * sl[k] * sl[k];
        seq = sqrt(3.0 / 2.0 * seq);
        alpha0 = v.alpha0[i], c44 = v.c44[i];
        yf = seq - (v.sigmay[i] + (1.0 - xi) * H * alpha0);
        plastic = yf > 0.0;
        dlam = plastic ? yf / (3 * c44 + H) : 0.0;
        if (fabs(seq) > LPMX_EPS)
            for (int k = 0; k < 6; k++)
                dep[k] = dlam * 1.5 * sl[k] / seq;
        for (int k = 0; k < 6; k++)
            D[k][p] = dep[k];
    }
    __syncthreads();
    // second pass in reverse (dL2 of the evaluation is in v.dL)
    double xpb = d2b * db, cc[6];
    cc6(c[0], c[1], c[2], cc);
    if (bond)
    {
        double dL2b = rev ? t * kn : 0.0;
        if (rev)
            dL2b += tr * knr;
        const double tot = dL2b + A2b + B2b * tv;
        Tvb += B2b * v.dL[b];
        xpb = -tot * db + d2b * db;
        double ccb[6], cb[3] = {0.0, 0.0, 0.0};
        for (int k = 0; k < 6; k++)
            ccb[k] = xpb * L0 * db * (k < 3 ? 1.0 : 2.0) * D[k][p];
        cc6_bar(c[0], c[1], c[2], ccb, cb);
        vjp_geom(gb, c, dis, tot * db, cb);
    }
    for (int k = 0; k < 6; k++)
        T[k][j][p] = bond ? xpb * L0 * db * (k < 3 ? 1.0 : 2.0) * cc[k] : 0.0;
    __syncthreads();
    for (int k = threadIdx.x; k < 6 * VT; k += nt)
        D[k / VT][k % VT] = vjp_sum<NB>(T[k / VT], nb, k % VT);
    __syncthreads();
    if (lead)
    {
        // slot-2 state
        double depb[6], dlamb = io.alpha2b[i], Hb = 0.0, alpha0b = io.alpha2b[i], beta0b[6];
        for (int k = 0; k < 6; k++)
        {
            const double bb = io.beta2b[(int64_t)k * n + i];
            beta0b[k] = bb;
            depb[k] = D[k][p] + 2. / 3. * xi * H * bb;
            Hb += 2. / 3. * xi * dep[k] * bb;
        }
        double sdevb[6] = {0, 0, 0, 0, 0, 0}, seqb = 0.0;
        if (fabs(seq) > LPMX_EPS)
            for (int k = 0; k < 6; k++)
            {
                dlamb += depb[k] * 1.5 * sl[k] / seq;
                sdevb[k] += depb[k] * 1.5 * dlam / seq;
                seqb -= depb[k] * 1.5 * dlam * sl[k] / (seq * seq);
            }
        double c44b = 0.0, syb = 0.0;
        if (plastic)
        {
            const double den = 3 * c44 + H;
            const double yfb = dlamb / den;
            c44b -= dlamb * yf * 3.0 / (den * den);
            Hb -= dlamb * yf / (den * den);
            seqb += yfb;
            syb -= yfb;
            Hb -= yfb * (1.0 - xi) * alpha0;
            alpha0b -= yfb * (1.0 - xi) * H;
        }
        if (seq > 0.0)
            for (int k = 0; k < 6; k++)
                sdevb[k] += seqb * 1.5 * (k < 3 ? 1.0 : 2.0) * sl[k] / seq;
        const double mb = (sdevb[0] + sdevb[1] + sdevb[2]) / 3.0;
        for (int k = 0; k < 6; k++)
        {
            io.beta0b[(int64_t)k * n + i] = beta0b[k] - sdevb[k];
            D[k][p] = k < 3 ? sdevb[k] - mb : sdevb[k];
        }
        io.alpha0b[i] = alpha0b;
        io.syb[i] = syb;
        io.Hb[i] = Hb;
        a.c44b[i] = c44b;
    }
    __syncthreads();
    // trial stress, trial force: adjoint of the trial force and the part of the
    // unit-vector adjoint that comes through the trial stress
    double tb = 0.0;
    if (bond)
    {
        double Ftrb = 0.0, ccb[6], cb[3] = {0.0, 0.0, 0.0};
        for (int k = 0; k < 6; k++)
            Ftrb += D[k][p] * w * cc[k], ccb[k] = D[k][p] * w * Ftr;
        cc6_bar(c[0], c[1], c[2], ccb, cb);
        tb = Ftrb * dw;
        Knb += tb * 2.0 * dl;
        Tvb += tb * A1;
        vjp_geom(gb, c, dis, 0.0, cb);
    }
    T[0][j][p] = tb, T[1][j][p] = tb * tv;
    __syncthreads();
    for (int k = threadIdx.x; k < 4 * VT; k += nt)
        AB[k / VT][k % VT] = vjp_shell_sum<NB>(T[k / VT < 2 ? 1 : 0], nullptr, sh, (k / VT) & 1, nb, k % VT);
    __syncthreads();
    // first pass and geometry
    if (bond)
    {
        const double A1b = AB[s][p], B1b = AB[2 + s][p];
        const double dL1b = tb * 2.0 * kn;
        const double tot = dL1b + A1b + B1b * tv;
        Tvb += B1b * dl;
        xpb -= tot * db;
        const double zero[3] = {0.0, 0.0, 0.0};
        vjp_geom(gb, c, dis, tot * db, zero);
        a.gb[b] = gb[0], a.gb[NBn + b] = gb[1], a.gb[2 * NBn + b] = gb[2];
        a.Knb[b] = Knb, a.Tvb[b] = Tvb;
    }
    if (i < n)
        io.dLp0b[b] = xpb;
}

// Positions from the bond vectors; the modulus factor from the bond constants.
template <int NB>
__global__ __launch_bounds__(VT *(NB ? NB : LPMX_MAXNB)) void k_vjp_gather(DV v, VjpIO io, AdjWork a)
{
    const int nb = NB ? NB : v.nb;
    __shared__ double T[7][NB ? NB : LPMX_MAXNB][VT];
    const int p = threadIdx.x % VT, j = threadIdx.x / VT, n = v.n, g0 = blockIdx.x * VT, i = g0 + p, nt = VT * nb;
    const int64_t b = (int64_t)j * n + i, NBn = (int64_t)n * v.nb;
    double x[3] = {0, 0, 0}, y[3] = {0, 0, 0}, e = 0;
    if (i < n && j < v.nb0[i])
    {
        const int q = v.nbr[b], s = v.nsign[b], r = v.rev[b], ti = v.type[i];
        const double kn = v.lattice == 1 ? v.ktype_t[3 * ti] : v.ktype_t[3 * ti + s];
        const double tv = v.lattice == 1 ? v.ktype_t[3 * ti + 1] : v.ktype_t[3 * ti + 2];
        const double own = a.Knb[b] * kn + a.Tvb[b] * tv;
        for (int k = 0; k < 3; k++)
            x[k] = a.gb[k * NBn + b];
        e = v.lattice == 2 ? 0.5 * own : own;
        if (r >= 0)
        {
            const int64_t br = (int64_t)r * n + q;
            for (int k = 0; k < 3; k++)
                y[k] = a.gb[k * NBn + br];
            if (v.lattice == 2)
                e = 0.5 * own + 0.5 * (a.Knb[br] * kn + a.Tvb[br] * tv);
        }
    }
    for (int k = 0; k < 3; k++)
        T[k][j][p] = x[k], T[3 + k][j][p] = y[k];
    T[6][j][p] = e;
    __syncthreads();
    for (int k = threadIdx.x; k < 4 * VT; k += nt)
    {
        const int c = k / VT, pp = k % VT, m = g0 + pp;
        if (m >= n)
            continue;
        if (c == 3)
        {
            io.eb[m] = vjp_sum<NB>(T[6], nb, pp) + a.c44b[m] * v.ce_t[3 * v.type[m] + 2];
            continue;
        }
        double t = 0.0;
#pragma unroll NB ? NB : 1
        for (int q = 0; q < (NB ? NB : nb); q++)
        {
            t += T[c][q][pp];
            t -= T[3 + c][q][pp];
        }
        io.xb[3 * (int64_t)m + c] = t;
    }
}

// The reverse sweep on device buffers, at the forward values left by the last
// lpmx_eval_j2 (positions and slot-0 state unchanged since).
int lpmx_vjp_device(const VjpIO &io)
{
    RETCHK(adj_work());
    const dim3 G(nblocks(g.n, VT)), B(VT * g.nb);
    if (g.nb == 18) // SC, FCC
    {
        hipLaunchKernelGGL(k_vjp_bonds<18>, G, B, 0, g_stream, g, io, AW);
        hipLaunchKernelGGL(k_vjp_gather<18>, G, B, 0, g_stream, g, io, AW);
    }
    else
    {
        hipLaunchKernelGGL(k_vjp_bonds<0>, G, B, 0, g_stream, g, io, AW);
        hipLaunchKernelGGL(k_vjp_gather<0>, G, B, 0, g_stream, g, io, AW);
    }
    LAUNCHCHK();
    return LPMX_OK;
}

// rows [n][w] <-> planes [w][n]
__global__ void k_adj_transpose(const double *src, double *dst, int n, int w, int to_planes)
{
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (t >= (int64_t)n * w)
        return;
    const int64_t i = t / w, c = t - i * w;
    if (to_planes)
        dst[c * n + i] = src[t];
    else
        dst[t] = src[c * n + i];
}

// One J2 evaluation at the current state, then its reverse sweep, host arrays in
// the reference layouts (Pbar [3n], dLp2bar [n][nb], beta2bar [n][6], alpha2bar [n];
// outputs likewise, Hbar a scalar).
extern "C" int lpmx_vjp(const double *Pb, const double *dLp2b, const double *beta2b, const double *alpha2b,
                        double *xb, double *dLp0b, double *beta0b, double *alpha0b, double *eb, double *syb,
                        double *Hb)
{
    RETCHK(lpmx_require_model());
    if (!Pb || !dLp2b || !beta2b || !alpha2b || !xb || !dLp0b || !beta0b || !alpha0b || !eb || !syb || !Hb)
        return lpmx_fail(LPMX_ERR_ARG, "lpmx_vjp: null argument");
    const int n = g.n, nb = g.nb;
    const int64_t NB = (int64_t)n * nb;
    // device scratch: seeds and outputs
    std::vector<double *> bufs;
    auto alloc = [&](int64_t c) -> double * {
        double *p = nullptr;
        if (dev_malloc(&p, sizeof(double) * c) != hipSuccess)
            return nullptr;
        bufs.push_back(p);
        return p;
    };
    double *dPb = alloc(3 * (int64_t)n), *tmp = alloc(NB > 6 * (int64_t)n ? NB : 6 * (int64_t)n);
    double *ddLp2b = alloc(NB), *dbeta2b = alloc(6 * (int64_t)n), *dalpha2b = alloc(n);
    double *dxb = alloc(3 * (int64_t)n), *ddLp0b = alloc(NB), *dbeta0b = alloc(6 * (int64_t)n);
    double *dalpha0b = alloc(n), *deb = alloc(n), *dsyb = alloc(n), *dHb = alloc(n);
    int rc = LPMX_OK;
    for (double *p : bufs)
        if (!p)
            rc = lpmx_fail(LPMX_ERR_HIP, "lpmx_vjp: allocation");
    if (rc == LPMX_OK)
        do
        {
            const dim3 B(LPMX_BLOCK);
            if ((rc = lpmx_eval_j2()) != LPMX_OK)
                break;
            hipMemcpyAsync(dPb, Pb, sizeof(double) * 3 * n, hipMemcpyHostToDevice, g_stream);
            hipMemcpyAsync(tmp, dLp2b, sizeof(double) * NB, hipMemcpyHostToDevice, g_stream);
            hipLaunchKernelGGL(k_adj_transpose, dim3(nblocks(NB)), B, 0, g_stream, tmp, ddLp2b, n, nb, 1);
            hipMemcpyAsync(tmp, beta2b, sizeof(double) * 6 * n, hipMemcpyHostToDevice, g_stream);
            hipLaunchKernelGGL(k_adj_transpose, dim3(nblocks(6 * (int64_t)n)), B, 0, g_stream, tmp, dbeta2b, n, 6, 1);
            hipMemcpyAsync(dalpha2b, alpha2b, sizeof(double) * n, hipMemcpyHostToDevice, g_stream);
            VjpIO io = {dPb, ddLp2b, dbeta2b, dalpha2b, dxb, ddLp0b, dbeta0b, dalpha0b, deb, dsyb, dHb};
            if ((rc = lpmx_vjp_device(io)) != LPMX_OK)
                break;
            hipMemcpyAsync(xb, dxb, sizeof(double) * 3 * n, hipMemcpyDeviceToHost, g_stream);
            hipLaunchKernelGGL(k_adj_transpose, dim3(nblocks(NB)), B, 0, g_stream, ddLp0b, tmp, n, nb, 0);
            hipMemcpyAsync(dLp0b, tmp, sizeof(double) * NB, hipMemcpyDeviceToHost, g_stream);
            hipStreamSynchronize(g_stream);
            hipLaunchKernelGGL(k_adj_transpose, dim3(nblocks(6 * (int64_t)n)), B, 0, g_stream, dbeta0b, tmp, n, 6, 0);
            hipMemcpyAsync(beta0b, tmp, sizeof(double) * 6 * n, hipMemcpyDeviceToHost, g_stream);
            hipMemcpyAsync(alpha0b, dalpha0b, sizeof(double) * n, hipMemcpyDeviceToHost, g_stream);
            hipMemcpyAsync(eb, deb, sizeof(double) * n, hipMemcpyDeviceToHost, g_stream);
            hipMemcpyAsync(syb, dsyb, sizeof(double) * n, hipMemcpyDeviceToHost, g_stream);
            double hsum = 0.0;
            if ((rc = lpmx_dev_sum(dHb, n, &hsum)) != LPMX_OK)
                break;
            *Hb = hsum;
            if (hipStreamSynchronize(g_stream) != hipSuccess || hipGetLastError() != hipSuccess)
                rc = lpmx_fail(LPMX_ERR_HIP, "lpmx_vjp: device error");
        } while (0);
    for (double *p : bufs)
        if (p)
            hipFree(p);
    return rc;
}

void lpmx_adjoint_free(void)
{
    lpmx_adjoint_free_work();
    lpmx_history_free();
}
