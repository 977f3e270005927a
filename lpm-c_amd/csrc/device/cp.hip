// Crystal plasticity of the reference (plmode 1, src/constitutive.c:866-1396): per
// particle, trial resolved shear stresses on the Schmid tensors, an active-set search
// with an inner Newton iteration on the slips (dense LU with partial pivoting on the
// nslip x nslip slip Jacobian), the plastic bond stretch, then the same final force
// pass as the J2 law.  Half a wavefront per particle: lane j owns bond slot j, lane s
// slip system s and its row of the slip Jacobian; every per-particle array is a plane
// [entry][particle].
//
// The reference factorises the full nslip x nslip slip Jacobian in place
// (LAPACKE_dgesv), with zeros in every row and column of an inactive system but its
// unit diagonal.  Partial pivoting never picks such a row (its entries in the active
// columns are zero), its multipliers are zero and its right-hand side entry is
// zero, so every elimination step on it subtracts zero products: the active
// systems' solution is the LU solve of the active submatrix, rows and columns kept
// in ascending system order, with the same operations in the same order.  This
// kernel factorises only that submatrix (na x na, na active systems) and sums the
// hardening matrix over the active systems only; the results are the same values,
// and the work per inner iteration drops from nslip^3 to na^3.
//
// Compiled without floating-point contraction, in the reference's evaluation order.
#include <math.h>
#include <string.h>

#include "common.h"

#define BI(j, i) ((int64_t)(j) * v.n + (i))
#define CPI(e, i) ((int64_t)(e) * v.n + (i))
#define CP_TOLITER 1e-4 // the reference's TOLITER (include/lpm.h:41)
#define CP_MAXSMALL 20  // the reference's MAXSMALL (include/lpm.h:38)

// pow() of the hardening and rate terms: the exponents 1, 2 and 0 that the
// linear-hardening, linear-rate settings produce are exact, as in a correctly
// rounded pow; other exponents go to the device pow.
__device__ __forceinline__ double cp_pow(double x, double y)
{
    if (y == 1.0)
        return x;
    if (y == 2.0)
        return x * x;
    if (y == 0.0)
        return 1.0;
    return pow(x, y);
}

__device__ __forceinline__ double proj(double cx, double cy, double cz, const double *t)
{
    return cx * cx * t[0] + cy * cy * t[1] + cz * cz * t[2] + cy * cz * t[3] + cx * cz * t[4] + cx * cy * t[5];
}

__device__ __forceinline__ double cp_opp(const DV &v, int i, int j)
{
    if (v.nbcur[i] == v.nb)
        return 0.5;
    const int o = v.opp[BI(j, i)];
    if (o < 0)
        return 1.0;
    return v.db[BI(o, i)] <= LPMX_EPS ? 1.0 : 0.5;
}

// computeCab (constitutive.c:1864-1917): C_ab of every particle at the current
// geometry (distance, cs), C[(a*ns+b)][i].  One thread per particle and system b
// (blockIdx.y), whose shell sums serve all a.
__global__ void k_cp_cab(DV v)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= v.n)
        return;
    const int ns = v.nslip, nbi = v.nb0[i], b = blockIdx.y;
    const double *tb = v.schmid + 6 * b;
    double Ls[2] = {0, 0};
    for (int j = 0; j < nbi; j++)
    {
        const int64_t q = BI(j, i);
        const double t = v.Tv[q] * v.dist[q] * proj(v.csx[q], v.csy[q], v.csz[q], tb);
        if (v.nsign[q] == 0)
            Ls[0] += t;
        else
            Ls[1] += t;
    }
    for (int a = 0; a < ns; a++)
    {
        const double *ta = v.schmid + 6 * a;
        double c = 0.;
        for (int j = 0; j < nbi; j++)
        {
            const int64_t q = BI(j, i);
            const double cx = v.csx[q], cy = v.csy[q], cz = v.csz[q];
            const double dF = -2.0 * v.Kn[q] * v.dist[q] * proj(cx, cy, cz, tb) - 2.0 * (v.nsign[q] == 0 ? Ls[0] : Ls[1]);
            c += -cp_opp(v, i, j) / v.volume * v.dist[q] * dF * proj(cx, cy, cz, ta);
        }
        v.cp_Cab[CPI(a * ns + b, i)] = c;
    }
}

// BLAS dnrm2 (scaled sum of squares), as the reference's cblas_dnrm2, over the entries
// of the active systems (the others are zero, which dnrm2 skips).
__device__ double cp_nrm2(int n, const double *x)
{
    double scale = 0.0, ssq = 1.0;
    for (int k = 0; k < n; k++)
        if (x[k] != 0.0)
        {
            const double ax = fabs(x[k]);
            if (scale < ax)
            {
                ssq = 1.0 + ssq * (scale / ax) * (scale / ax);
                scale = ax;
            }
            else
                ssq += (ax / scale) * (ax / scale);
        }
    return scale * sqrt(ssq);
}

#define CPL 32       // lanes per particle: at least LPMX_MAXNB and LPMX_MAXSLIP
#define CP_PER_WG 4  // particles per work-group (two wavefronts)
#define CP_NREG 8    // active systems whose Jacobian row a lane keeps in registers
static_assert(CPL >= LPMX_MAXNB && CPL >= LPMX_MAXSLIP, "a lane per bond slot and per slip system");

// What a particle's lanes exchange.
struct CpShared
{
    double t[6][CPL + 1]; // bond terms of an ordered sum, one row per sum
    // by active position (ascending systems): slip, yield stress, residual, correction;
    // ga, ra are zero from the number of active systems on
    double ga[LPMX_MAXSLIP], xg[LPMX_MAXSLIP], ra[LPMX_MAXSLIP], xs[LPMX_MAXSLIP];
    int act[LPMX_MAXSLIP]; // the active systems (0 beyond their number)
};

// Orders the LDS accesses of one wavefront's lanes (the lanes of a particle share one).
__device__ __forceinline__ void cp_wave_sync(void)
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Shell sums in slot order of the lanes' x and tx (two shells each), by four lanes; a
// lane without a bond holds zeros, which leave the sums' bits as they are.
template <int NB>
__device__ __forceinline__ void cp_shell_sums(CpShared &S, int lane, unsigned shell1, double x, double tx, double *a,
                                              double *b)
{
    S.t[0][lane] = x;
    S.t[1][lane] = tx;
    cp_wave_sync();
    const double *src = S.t[(lane >> 1) & 1];
    const unsigned want = (lane & 1) ? shell1 : ~shell1;
    double s = 0.0;
#pragma unroll
    for (int j = 0; j < NB; j++)
        s += (want >> j) & 1u ? src[j] : 0.0;
    a[0] = __shfl(s, 0, CPL), a[1] = __shfl(s, 1, CPL);
    b[0] = __shfl(s, 2, CPL), b[1] = __shfl(s, 3, CPL);
    cp_wave_sync();
}

// Local stress (constitutive.c:963-998): lane j's bond adds w F cs cs (w = opposite-bond
// factor / volume * L0); six lanes sum the slots in order.
template <int NB>
__device__ __forceinline__ void cp_stress(CpShared &S, int lane, bool s1, double w, double kn, double tv, double dw,
                                          double cx, double cy, double cz, double x, const double *a,
                                          const double *b, double *sl)
{
    double F = 2.0 * kn * x + (s1 ? b[1] : b[0]) + tv * (s1 ? a[1] : a[0]);
    F *= dw;
    const double f = w * F;
    S.t[0][lane] = f * cx * cx;
    S.t[1][lane] = f * cy * cy;
    S.t[2][lane] = f * cz * cz;
    S.t[3][lane] = f * cy * cz;
    S.t[4][lane] = f * cx * cz;
    S.t[5][lane] = f * cx * cy;
    cp_wave_sync();
    const double *src = S.t[lane < 6 ? lane : 0];
    double s = 0.0;
#pragma unroll
    for (int j = 0; j < NB; j++)
        s += src[j];
#pragma unroll
    for (int c = 0; c < 6; c++)
        sl[c] = __shfl(s, c, CPL);
    cp_wave_sync();
}

__device__ __forceinline__ double cp_rss(const double *sl, const double *t)
{
    return sl[0] * t[0] + sl[1] * t[1] + sl[2] * t[2] + sl[3] * t[3] + sl[4] * t[4] + sl[5] * t[5];
}

// x of another lane of the same eight (DPP control word CTRL).
template <int CTRL>
__device__ __forceinline__ double cp_dpp(double x)
{
    int lo = __double2loint(x), hi = __double2hiint(x);
    lo = __builtin_amdgcn_update_dpp(lo, lo, CTRL, 0xf, 0xf, false);
    hi = __builtin_amdgcn_update_dpp(hi, hi, CTRL, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}

// The largest of the group's lanes (8 or CPL lanes): lane ^ 1, lane ^ 2, the mirror of
// each eight, then across the eights.
template <int G>
__device__ __forceinline__ double cp_group_max(double m)
{
    m = fmax(m, cp_dpp<0xB1>(m));
    m = fmax(m, cp_dpp<0x4E>(m));
    m = fmax(m, cp_dpp<0x141>(m));
    if (G > 8)
    {
        m = fmax(m, __shfl_xor(m, 8, CPL));
        m = fmax(m, __shfl_xor(m, 16, CPL));
    }
    return m;
}

// Row p of the active slip Jacobian, on lane p, and the solution by column: in
// registers for up to CP_NREG active systems (compile-time indices; C and sc hold the
// row of C_ab and, on lanes c < 6, component c of the active Schmid tensors), or, for
// larger active sets, the row in the particle's plane of cp_D and the rest re-read.
struct CpRowReg
{
    static constexpr int N = CP_NREG, U = CP_NREG, G = 8;
    double C[N], sc[N], d[N], x[N];
    __device__ __forceinline__ void load(const DV &v, const CpShared &S, const double (*sch)[6], int i, int lane)
    {
        const int ns = v.nslip, m = lane < N ? S.act[lane] : 0, c6 = lane < 6 ? lane : 0;
#pragma unroll
        for (int e = 0; e < N; e++)
        {
            C[e] = lane < N ? v.cp_Cab[CPI(m * ns + S.act[e], i)] : 0.0;
            sc[e] = sch[S.act[e]][c6];
        }
    }
    __device__ __forceinline__ double cab(const DV &, const CpShared &, int, int, int e) const { return C[e]; }
    __device__ __forceinline__ double schmid(const CpShared &, const double (*)[6], int, int e) const { return sc[e]; }
    __device__ __forceinline__ double get(int e) const { return d[e]; }
    __device__ __forceinline__ void set(int e, double y) { d[e] = y; }
    __device__ __forceinline__ double getx(const CpShared &, int e) const { return x[e]; }
    __device__ __forceinline__ void setx(CpShared &S, int lane, int e, double y)
    {
        x[e] = y;
        if (lane == 0)
            S.xs[e] = y;
    }
};
struct CpRowMem
{
    static constexpr int N = LPMX_MAXSLIP, U = 1, G = CPL;
    double *d;
    int64_t stride;
    __device__ __forceinline__ void load(const DV &v, const CpShared &, const double (*)[6], int i, int lane)
    {
        d = v.cp_D + CPI((lane < v.nslip ? lane : 0) * v.nslip, i), stride = v.n;
    }
    __device__ __forceinline__ double cab(const DV &v, const CpShared &S, int i, int lane, int e) const
    {
        return v.cp_Cab[CPI(S.act[lane] * v.nslip + S.act[e], i)];
    }
    __device__ __forceinline__ double schmid(const CpShared &S, const double (*sch)[6], int lane, int e) const
    {
        return sch[S.act[e]][lane < 6 ? lane : 0];
    }
    __device__ __forceinline__ double get(int e) const { return d[e * stride]; }
    __device__ __forceinline__ void set(int e, double y) { d[e * stride] = y; }
    __device__ __forceinline__ double getx(const CpShared &S, int e) const { return S.xs[e]; }
    __device__ __forceinline__ void setx(CpShared &S, int lane, int e, double y)
    {
        if (lane == 0)
            S.xs[e] = y;
        cp_wave_sync();
    }
};

// Row `lane` (< na) of the active submatrix of the slip Jacobian.  Its hardening sum
// runs over the active systems in order (the inactive ones add Jact * hd = 0): hd(m, u,
// d) is q hp gam_d but at d = m (h + hp gam_m when m = u, else hp gam_m) and at d = u !=
// m (q (h + hp gam_u)); the same expressions as the reference's four cases.  Entry e of
// the row differs from the others only in the term of position e, so the partial sum
// before it is shared.
template <class Row>
__device__ __forceinline__ void cp_jacobian_row(const DV &v, CpShared &S, Row &D, int i, int lane, int na, double h,
                                                double hp)
{
    constexpr int N = Row::N, U = Row::U;
    const double gam = S.ga[lane], xgy = S.xg[lane];
    const double t1 = xgy * (v.cp_eta / v.cp_p / v.dtime *
                             cp_pow(1. + v.cp_eta * gam / v.dtime, (1. - v.cp_p) / v.cp_p));
    const double pw = cp_pow(1. + v.cp_eta * gam / v.dtime, (1. / v.cp_p));
    const double qhp = v.cp_q * hp, hpg = hp * gam, hd = h + hpg;
    double before = 0.0;
#pragma unroll U
    for (int e = 0; e < N; e++)
        if (e < na)
        {
            const double ge = S.ga[e];
            double hs = before + (e == lane ? hd : v.cp_q * (h + hp * ge));
#pragma unroll U
            for (int c = 0; c < N; c++)
                if (c > e && c < na)
                    hs += c == lane ? hpg : qhp * S.ga[c];
            before += e == lane ? hpg : qhp * ge;
            const double t2 = hs * pw, cab = D.cab(v, S, i, lane, e);
            D.set(e, e == lane ? cab + t1 + t2 : cab + t2);
        }
}

// Solve D x = r for the na active rows (row p on lane p, x by position to S.xs):
// Gaussian elimination with partial pivoting (first largest |d_ik| on or below the
// diagonal).  A row swap only exchanges two places; the operations on every entry are
// those of the in-place LU with whole-row swaps, in its order.  False on an exact zero
// pivot.
template <class Row>
__device__ __forceinline__ bool cp_lu_solve(CpShared &S, Row &D, int lane, int na, double r)
{
    constexpr int N = Row::N, U = Row::U;
    const int half = threadIdx.x & 32;
    const bool row = lane < na;
    int place = row ? lane : CPL; // of the lane's row in the permuted matrix
    int at = 0;                   // lane k: the lane whose row is at place k
#pragma unroll U
    for (int k = 0; k < N; k++)
        if (k < na)
        {
            const bool on = row && place >= k;
            const double dk = on ? D.get(k) : 0.0;
            const double a = on ? fabs(dk) : -1.0;
            const double m = cp_group_max<Row::G>(a);
            // the rows' group decides for all lanes of the particle (a group without rows
            // has m = -1)
            if ((unsigned)(__ballot(m == 0.0) >> half))
                return false;
            // of equal entries the first in the order of the permuted rows
            unsigned hit = (unsigned)(__ballot(on && a == m) >> half);
            if (!hit) // a NaN column: the row in place
                hit = (unsigned)(__ballot(place == k) >> half);
            int ml = __ffs(hit) - 1;
            if (hit & (hit - 1))
            {
                int best = on && a == m ? place : CPL;
#pragma unroll
                for (int o = CPL / 2; o >= 1; o >>= 1)
                    best = min(best, __shfl_xor(best, o, CPL));
                ml = __ffs((unsigned)(__ballot(place == best) >> half)) - 1;
            }
            const int old = __shfl(place, ml, CPL);
            if (lane == ml)
                place = k;
            else if (place == k)
                place = old;
            at = lane == k ? ml : at;
            const double dkk = __shfl(dk, ml, CPL);
            const bool below = row && place > k;
            double l = 0.0;
            if (below)
            {
                l = dk / dkk;
                D.set(k, l);
            }
#pragma unroll U
            for (int j = 0; j < N; j++)
                if (j > k && j < na)
                {
                    const double dj = row ? D.get(j) : 0.0;
                    const double y = __shfl(dj, ml, CPL);
                    if (below)
                        D.set(j, dj - l * y);
                }
            // the right-hand side: each row subtracts in column order, as the forward
            // substitution does after the swaps
            const double rk = __shfl(r, ml, CPL);
            if (below)
                r -= l * rk;
        }
#pragma unroll U
    for (int a = N - 1; a >= 0; a--)
        if (a < na)
        {
            double t = 0.0;
            if (place == a)
            {
                t = r;
#pragma unroll U
                for (int j = 0; j < N; j++)
                    if (j > a && j < na)
                        t -= D.get(j) * D.getx(S, j);
                t /= D.get(a);
            }
            D.setx(S, lane, a, __shfl(t, __shfl(at, a, CPL), CPL));
        }
    return true;
}

// The plastic strain of the slips (six components by lanes, sums in system order) and
// their sum.
template <class Row>
__device__ __forceinline__ void cp_slip_sums(const CpShared &S, const Row &D, const double (*sch)[6], int lane, int na,
                                             double *dpl, double *dA)
{
    constexpr int N = Row::N, U = Row::U;
    double p = 0.0, sum = 0.0;
#pragma unroll U
    for (int c = 0; c < N; c++)
        if (N == CP_NREG || c < na)
        {
            const double gc = S.ga[c];
            p += gc * D.schmid(S, sch, lane, c);
            sum += gc;
        }
#pragma unroll
    for (int c = 0; c < 6; c++)
        dpl[c] = __shfl(p, c, CPL);
    *dA = sum;
}

// The return map of each particle (constitutive.c:944-1320), then its second
// stretch pass with the updated plastic stretch and slot 2 of its state.  Sums over
// bonds and systems run in the reference's order: the lanes put the terms in LDS and
// one lane per sum adds them in slot order, so the bits are those of the serial map.
//
// A launch lasts as long as its slowest particles (up to 22 active-set passes and 84
// inner iterations at 256k particles), and at two waves per SIMD (240 VGPRs) the chain
// of one inner iteration is what it waits for.  Hence the lanes per particle, the
// Jacobian rows in registers, the loads of C_ab once per pass, the pivot search over
// eight lanes, and one loop over the inner iterations of all passes, so that the two
// particles of a wavefront wait for each other only at the end.  Against one thread per
// particle with its arrays in scratch memory: 256,000 particles 40.2 -> 20.4 ms, 32,000
// 15.8 -> 2.9 ms, 500 10.2 -> 0.62 ms a force evaluation, transfers included, with the
// same bits.  Three waves per SIMD (168 VGPRs, 123 spilled) took 20.7, 3.0 and 0.70 ms;
// rows of up to 24 systems in registers one wave per SIMD.
template <int NB>
__global__ __launch_bounds__(CPL * CP_PER_WG) __attribute__((amdgpu_waves_per_eu(2))) void k_cp_particle(DV v, int first,
                                                                                                      int count)
{
    __shared__ CpShared SH[CP_PER_WG];
    __shared__ double sch[LPMX_MAXSLIP][6];
    const int ns = v.nslip;
    for (int t = threadIdx.x; t < 6 * ns; t += CPL * CP_PER_WG)
        sch[t / 6][t % 6] = v.schmid[t];
    __syncthreads();
    const int lane = threadIdx.x & (CPL - 1), w = threadIdx.x / CPL;
    const int i = first + blockIdx.x * CP_PER_WG + w;
    if (i >= first + count)
        return; // uniform over the particle's lanes; no work-group barrier follows
    CpShared &S = SH[w];
    const int half = threadIdx.x & 32;
    const int nbi = v.nb0[i];
    // lane's bond (zeros on lanes without one)
    const bool bond = lane < nbi;
    const int64_t b = BI(lane < v.nb ? lane : 0, i);
    double cx = 0, cy = 0, cz = 0, dis = 0, L0 = 0, kn = 0, tv = 0, db = 0, dw = 0, wl = 0, dl = 0;
    bool s1 = false;
    if (bond)
    {
        const int q = v.nbr[b];
        const double dx = v.x[3 * i] - v.x[3 * q], dy = v.x[3 * i + 1] - v.x[3 * q + 1],
                     dz = v.x[3 * i + 2] - v.x[3 * q + 2];
        dis = sqrt(dx * dx + dy * dy + dz * dz);
        cx = dx / dis, cy = dy / dis, cz = dz / dis;
        L0 = v.L0[b], kn = v.Kn[b], tv = v.Tv[b], dw = v.dw[b], db = v.db[b];
        s1 = v.nsign[b] != 0;
        wl = cp_opp(v, i, lane) / v.volume * L0;
        dl = dis - L0;
        dl -= v.dLp0[b];
        dl *= db;
    }
    const unsigned shell1 = (unsigned)(__ballot(s1) >> half);
    double xa[2], xb[2], sl[6];
    cp_shell_sums<NB>(S, lane, shell1, dl, tv * dl, xa, xb);
    cp_stress<NB>(S, lane, s1, wl, kn, tv, dw, cx, cy, cz, dl, xa, xb, sl);
    // lane's slip system
    const bool sys = lane < ns;
    const double *ts = sch[sys ? lane : 0];
    const double gy0 = sys ? v.cp_gy0[CPI(lane, i)] : 0.0;
    double rss = cp_rss(sl, ts), gam = 0, dgy = 0, dA = 0.0, dd = 0.0;
    int Jact = 0;
    if ((unsigned)(__ballot(sys && rss - gy0 > LPMX_EPS) >> half))
    {
        if (lane == 0)
            v.pl_flag[i] = 1;
        const double A0 = v.cp_A0[i], tsd = v.cp_taus - v.cp_tau0;
        // the active systems of a pass, ascending; an active lane's position pos
        int nouter = 1, ninner = 0, na = 0, pos = CPL;
        CpRowReg DR;
        CpRowMem DM;
        if (lane < LPMX_MAXSLIP)
            S.act[lane] = 0, S.ga[lane] = 0.0, S.ra[lane] = 0.0;
        cp_wave_sync();
        DR.load(v, S, sch, i, lane);
        DM.load(v, S, sch, i, lane);
        for (;;)
        {
            ninner++;
            if (Jact == 1)
                S.ga[pos] = gam;
            cp_wave_sync();
            // sums over the active systems: an inactive one adds Jact * ... = 0
            double dpl[6];
            if (na <= CP_NREG)
                cp_slip_sums(S, DR, sch, lane, na, dpl, &dA);
            else
                cp_slip_sums(S, DM, sch, lane, na, dpl, &dA);
            dd = L0 * (dpl[0] * cx * cx + dpl[1] * cy * cy + dpl[2] * cz * cz + dpl[3] * cy * cz + dpl[4] * cx * cz +
                       dpl[5] * cx * cy);
            dd *= db;
            const double xdl = dl - dd;
            cp_shell_sums<NB>(S, lane, shell1, xdl, tv * xdl, xa, xb);
            cp_stress<NB>(S, lane, s1, wl, kn, tv, dw, cx, cy, cz, xdl, xa, xb, sl);
            // cosh and tanh round to 1 and to the argument below 1e-9
            const double xA = A0 + dA, ha = v.cp_h0 * xA / tsd;
            const bool flat = fabs(ha) < 1e-9;
            const double ch = flat ? 1.0 : cosh(ha), th = flat ? ha : tanh(ha);
            const double h = v.cp_h0 / cp_pow(ch, 2.0);
            const double hp = -2.0 * v.cp_h0 * v.cp_h0 / tsd * th * h;
            const double qh = v.cp_q * h;
            dgy = 0.0;
            if (Jact == 1)
                for (int c = 0; c < na; c++)
                    dgy += (c == pos ? h : qh) * S.ga[c];
            const double xgy = gy0 + dgy;
            rss = cp_rss(sl, ts);
            if (Jact == 1)
            {
                const double r = rss - xgy * cp_pow(1. + gam * v.cp_eta / v.dtime, 1. / v.cp_p);
                S.xg[pos] = xgy;
                S.ra[pos] = r;
            }
            cp_wave_sync();
            const double rp = lane < na ? S.ra[lane] : 0.0;
            bool ok;
            if (na <= CP_NREG)
            {
                if (lane < na)
                    cp_jacobian_row(v, S, DR, i, lane, na, h, hp);
                ok = cp_lu_solve(S, DR, lane, na, rp);
            }
            else
            {
                if (lane < na)
                    cp_jacobian_row(v, S, DM, i, lane, na, h, hp);
                ok = cp_lu_solve(S, DM, lane, na, rp);
            }
            cp_wave_sync();
            if (!ok)
            {
                if (lane == 0)
                    atomicAdd(v.cp_fail, 1);
                break;
            }
            if (Jact == 1)
                gam += S.xs[pos];
            // |r| > CP_TOLITER with the reference's scaled norm; its value matters only
            // where the plain sum of squares is within rounding of the bound
            double s2 = 0.0;
            if (na <= CP_NREG)
#pragma unroll
                for (int c = 0; c < CP_NREG; c++)
                    s2 += S.ra[c] * S.ra[c];
            else
                for (int c = 0; c < na; c++)
                    s2 += S.ra[c] * S.ra[c];
            const double bound = CP_TOLITER * CP_TOLITER;
            bool more;
            if (s2 > bound * (1.0 + 1e-10) && s2 < 1e300)
                more = true;
            else if (s2 < bound * (1.0 - 1e-10))
                more = false;
            else
                more = cp_nrm2(na, S.ra) > CP_TOLITER;
            if (more && ninner < CP_MAXSMALL)
                continue;
            // end of a pass: the active system with the lowest negative yield function
            // and no slip leaves; else the inactive one with the highest positive one
            // enters (of equal ones the first)
            const double yf = rss - xgy;
            double m = Jact == 1 && gam <= 0.0 && yf < 0.0 ? -yf : 0.0;
            const bool out = (unsigned)(__ballot(m > 0.0) >> half) != 0;
            if (!out)
                m = sys && Jact == 0 && yf > 0.0 ? yf : 0.0;
            const double top = cp_group_max<CPL>(m);
            if (!(top > 0.0))
                break;
            const int ml = __ffs((unsigned)(__ballot(m == top) >> half)) - 1;
            if (lane == ml)
                Jact = out ? 0 : 1;
            if (!out && nouter >= v.cp_maxloop)
                break;
            nouter++, ninner = 0;
            const unsigned amask = (unsigned)(__ballot(Jact == 1) >> half);
            na = __popc(amask);
            pos = Jact == 1 ? __popc(amask & ((1u << lane) - 1u)) : CPL;
            gam = 0.0;
            cp_wave_sync();
            if (lane < LPMX_MAXSLIP)
                S.act[lane] = 0, S.ga[lane] = 0.0, S.ra[lane] = 0.0;
            cp_wave_sync();
            if (Jact == 1)
                S.act[pos] = lane;
            cp_wave_sync();
            DR.load(v, S, sch, i, lane);
        }
    }
    if (sys)
    {
        const double das = Jact * gam;
        v.cp_Jact[CPI(lane, i)] = Jact;
        v.cp_RSS[CPI(lane, i)] = rss;
        v.cp_dgy[CPI(lane, i)] = dgy;
        v.cp_dAs[CPI(lane, i)] = das;
        v.cp_gy2[CPI(lane, i)] = gy0 + dgy;
        v.cp_As2[CPI(lane, i)] = v.cp_As0[CPI(lane, i)] + das;
    }
    if (lane == 0)
        v.cp_dA[i] = dA, v.cp_A2[i] = v.cp_A0[i] + dA;
    // plastic stretch of the step, second stretch pass, slot 2
    double d2 = 0.0;
    if (lane < v.nb)
    {
        double xp = v.dLp0[b];
        if (bond)
        {
            xp += dd;
            d2 = dis - L0;
            d2 -= xp;
            d2 *= db;
            v.ddLp[b] = dd;
            v.dL[b] = d2;
            v.csx[b] = cx, v.csy[b] = cy, v.csz[b] = cz;
        }
        v.dLp2[b] = (bond ? db : v.db[b]) * xp;
    }
    cp_shell_sums<NB>(S, lane, shell1, d2, tv * d2, xa, xb);
    if (lane < 2)
        v.A[(int64_t)lane * v.n + i] = lane ? xa[1] : xa[0], v.Bt[(int64_t)lane * v.n + i] = lane ? xb[1] : xb[0];
}

static double *cp_alloc(int64_t count)
{
    double *p = nullptr;
    if (dev_malloc(&p, sizeof(double) * count) != hipSuccess)
        return nullptr;
    return p;
}

void lpmx_cp_free(void)
{
    void *ps[] = {g.schmid, g.cp_gy0, g.cp_gy1, g.cp_gy2, g.cp_As0, g.cp_As1, g.cp_As2, g.cp_A0, g.cp_A1,
                  g.cp_A2, g.cp_dA, g.cp_dgy, g.cp_dAs, g.cp_RSS, g.cp_Jact, g.cp_Cab, g.cp_D, g.cp_fail};
    for (void *p : ps)
        if (p)
            hipFree(p);
    g.schmid = g.cp_gy0 = g.cp_gy1 = g.cp_gy2 = g.cp_As0 = g.cp_As1 = g.cp_As2 = nullptr;
    g.cp_A0 = g.cp_A1 = g.cp_A2 = g.cp_dA = g.cp_dgy = g.cp_dAs = g.cp_RSS = g.cp_Cab = g.cp_D = nullptr;
    g.cp_Jact = g.cp_fail = nullptr;
    g.nslip = 0;
}

__global__ void k_cp_init(DV v, double tau0)
{
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    const int64_t m = (int64_t)v.nslip * v.n;
    if (t < m)
    {
        v.cp_gy0[t] = v.cp_gy1[t] = v.cp_gy2[t] = tau0;
        v.cp_As0[t] = v.cp_As1[t] = v.cp_As2[t] = 0.0;
        v.cp_dgy[t] = v.cp_dAs[t] = v.cp_RSS[t] = 0.0;
        v.cp_Jact[t] = 0;
    }
    if (t < v.n)
        v.cp_A0[t] = v.cp_A1[t] = v.cp_A2[t] = v.cp_dA[t] = 0.0;
}

extern "C" int lpmx_set_slip_systems(int nslip, const double *schmid, const lpmx_cp_params *p)
{
    RETCHK(lpmx_require_model());
    if (nslip <= 0 || nslip > LPMX_MAXSLIP || !schmid || !p)
        return lpmx_fail(LPMX_ERR_ARG, "slip systems: nslip %d outside 1..%d or null input", nslip, LPMX_MAXSLIP);
    if (!(p->dtime > 0.0) || !(p->cp_p > 0.0) || p->taus == p->tau0)
        return lpmx_fail(LPMX_ERR_ARG, "slip systems: dtime and p must be positive and taus != tau0");
    lpmx_cp_free();
    const int64_t n = g.n, m = (int64_t)nslip * n;
    double **planes[] = {&g.cp_gy0, &g.cp_gy1, &g.cp_gy2, &g.cp_As0, &g.cp_As1, &g.cp_As2, &g.cp_dgy, &g.cp_dAs,
                         &g.cp_RSS};
    for (double **q : planes)
        if (!(*q = cp_alloc(m)))
            return lpmx_fail(LPMX_ERR_HIP, "slip-system state allocation");
    double **vecs[] = {&g.cp_A0, &g.cp_A1, &g.cp_A2, &g.cp_dA};
    for (double **q : vecs)
        if (!(*q = cp_alloc(n)))
            return lpmx_fail(LPMX_ERR_HIP, "slip-system state allocation");
    if (!(g.cp_Cab = cp_alloc(m * nslip)) || !(g.cp_D = cp_alloc(m * nslip)) ||
        !(g.schmid = cp_alloc(6 * nslip)))
        return lpmx_fail(LPMX_ERR_HIP, "slip-system matrix allocation");
    HIPCHK(dev_malloc(&g.cp_Jact, sizeof(int) * m));
    HIPCHK(dev_malloc(&g.cp_fail, sizeof(int)));
    HIPCHK(hipMemsetAsync(g.cp_fail, 0, sizeof(int), g_stream));
    HIPCHK(hipMemsetAsync(g.cp_Cab, 0, sizeof(double) * m * nslip, g_stream));
    HIPCHK(hipMemcpyAsync(g.schmid, schmid, sizeof(double) * 6 * nslip, hipMemcpyHostToDevice, g_stream));
    g.nslip = nslip;
    g.cp_tau0 = p->tau0, g.cp_taus = p->taus, g.cp_h0 = p->h0, g.cp_q = p->q;
    g.cp_eta = p->eta, g.cp_p = p->cp_p, g.dtime = p->dtime, g.cp_maxloop = p->maxloop;
    hipLaunchKernelGGL(k_cp_init, dim3(nblocks(m > n ? m : n)), dim3(LPMX_BLOCK), 0, g_stream, g, p->tau0);
    LAUNCHCHK();
    HIPCHK(hipStreamSynchronize(g_stream));
    return LPMX_OK;
}

extern "C" int lpmx_compute_cab(void)
{
    RETCHK(lpmx_require_model());
    if (g.nslip <= 0)
        return lpmx_fail(LPMX_ERR_STATE, "computeCab before the slip systems are set");
    hipLaunchKernelGGL(k_cp_cab, dim3(nblocks(g.n), g.nslip), dim3(LPMX_BLOCK), 0, g_stream, g);
    LAUNCHCHK();
    return LPMX_OK;
}

// Return maps of all particles (plmode 1); the caller then runs the J2 force pass.
int lpmx_cp_particles(void)
{
    if (g.nslip <= 0)
        return lpmx_fail(LPMX_ERR_STATE, "plmode 1 before the slip systems are set");
    const dim3 G(nblocks(g.n, CP_PER_WG)), B(CPL * CP_PER_WG);
    if (g.nb <= 18)
        hipLaunchKernelGGL(k_cp_particle<18>, G, B, 0, g_stream, g, 0, g.n);
    else
        hipLaunchKernelGGL(k_cp_particle<LPMX_MAXNB>, G, B, 0, g_stream, g, 0, g.n);
    LAUNCHCHK();
    return LPMX_OK;
}

extern "C" int lpmx_cp_failures(int *count)
{
    RETCHK(lpmx_require_model());
    *count = 0;
    if (g.cp_fail)
    {
        HIPCHK(hipMemcpyAsync(count, g.cp_fail, sizeof(int), hipMemcpyDeviceToHost, g_stream));
        HIPCHK(hipStreamSynchronize(g_stream));
    }
    return LPMX_OK;
}
