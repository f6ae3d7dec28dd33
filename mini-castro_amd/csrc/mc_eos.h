// Device Helmholtz EOS for gfx950.
//
// Same thermodynamics and floating-point evaluation order as the reference
// routine `eos` (Source/eos.F90:141-576), organised for a GPU:
//  * the table is node-interleaved: each (i,j) node holds the 13 columns the
//    hydro path consumes in one 128-byte row (f ft ftt fd fdd fdt fddt fdtt
//    fddtt dpdf dpdft dpdfd dpdfdt + 3 pad), so one evaluation reads four
//    128-byte rows instead of 52 scattered words;
//  * the density-side quantities (iat, xd and all density basis weights)
//    depend only on ye*rho, which is fixed during a Newton solve, so they are
//    computed once per call;
//  * Newton iterations evaluate only e and de/dT (eos_energy: the three h5
//    sums that feed them); the rest (eos_pressure: p, dp/drho, dp/dT, gamma_1,
//    ...) is evaluated once, at the temperature the reference's final pass
//    uses, with weights of its own.  Every quantity that is computed is
//    computed with the reference's expression, so results are bit-identical
//    to the reference arithmetic when built without FMA contraction;
//  * table cells are found with a single-precision logarithm except near grid
//    lines, and a convergence test divides only near its tolerance.
// With both halves of an evaluation in one loop a kernel took 256 registers
// and spilled or ran one wavefront per SIMD; apart they take at most 251 with
// a cell's state (256^3: K_prim 3.55 -> 2.95 ms, K_update 4.5 -> 4.1, K_est 2.0 ->
// 1.4; a 64^3 box: estdt 81 -> 25 us, compute_temp on its grown 72^3 31 -> 17;
// 1,000,000 unordered (rho, e) solves 436 -> 342 us).
// The electron chemical potential and number density tables (ef*, xf*) and
// the entropy terms feed nothing on the hydro path and are not evaluated.
#pragma once

#include "mc_common.h"

namespace mc {

constexpr int EOS_IMAX = 541;
constexpr int EOS_JMAX = 201;
constexpr int EOS_NODE = 16;   // doubles per table node
constexpr int EOS_GRID = 8;    // doubles per grid entry
constexpr int EOS_MAX_NEWTON = 100;  // Source/eos.F90:126

// Node column slots.
enum { NF = 0, NFT, NFTT, NFD, NFDD, NFDT, NFDDT, NFDTT, NFDDTT, NDPDF, NDPDFT, NDPDFD, NDPDFDT };
// Grid entry slots: temperature (t dt dt2 dti dt2i), density (d dd dd2 ddi dd2i).
enum { G_X = 0, G_D, G_D2, G_DI, G_D2I };

struct EosTable {
    const double *node;  // IMAX*JMAX nodes, node (i,j) at (i-1) + IMAX*(j-1)
    const double *tg;    // JMAX entries
    const double *dg;    // IMAX entries
    unsigned long long *newton_fail;  // Newton solves that ended unconverged (may be null)
};

// The reference lets a Newton solve that has not converged after
// EOS_MAX_NEWTON iterations pass silently (Source/eos.F90:193,550); the
// result is the same here, and the solve is also counted.
__device__ __forceinline__ void eos_note_newton_failure(const EosTable &tab)
{
    if (tab.newton_fail) atomicAdd(tab.newton_fail, 1ull);
}

// Source/eos.F90:60-74,129-137 (the entropy constant sioncon is unused)
namespace eosc {
constexpr double tlo = 3.0, thi = 13.0, dlo = -12.0, dhi = 15.0;
constexpr double tstp = (thi - tlo) / 200.0;
constexpr double tstpi = 1.0 / tstp;
constexpr double dstp = (dhi - dlo) / 540.0;
constexpr double dstpi = 1.0 / dstp;
constexpr double mintemp = 1000.0;
constexpr double ttol = 1.0e-8;
constexpr double clight = 2.99792458e10;
constexpr double kerg = 1.380650424e-16;
constexpr double avo_eos = 6.0221417930e23;
constexpr double asol = 4.0 * 5.67051e-5 / clight;
constexpr double kergavo = kerg * avo_eos;
constexpr double asoli3 = asol / 3.0;
} // namespace eosc

// Hermite basis, Source/eos.F90:740-1031
__device__ __forceinline__ double psi0(double z) { return (z * z * z) * (z * (-6.0 * z + 15.0) - 10.0) + 1.0; }
__device__ __forceinline__ double dpsi0(double z) { return (z * z) * (z * (-30.0 * z + 60.0) - 30.0); }
__device__ __forceinline__ double ddpsi0(double z) { return z * (z * (-120.0 * z + 180.0) - 60.0); }
__device__ __forceinline__ double psi1(double z) { return z * ((z * z) * (z * (-3.0 * z + 8.0) - 6.0) + 1.0); }
__device__ __forceinline__ double dpsi1(double z) { return z * z * (z * (-15.0 * z + 32.0) - 18.0) + 1.0; }
__device__ __forceinline__ double ddpsi1(double z) { return z * (z * (-60.0 * z + 96.0) - 36.0); }
__device__ __forceinline__ double psi2(double z) { return 0.5 * z * z * (z * (z * (-z + 3.0) - 3.0) + 1.0); }
__device__ __forceinline__ double dpsi2(double z) { return 0.5 * z * (z * (z * (-5.0 * z + 12.0) - 9.0) + 2.0); }
__device__ __forceinline__ double ddpsi2(double z) { return 0.5 * (z * (z * (-20.0 * z + 36.0) - 18.0) + 2.0); }
__device__ __forceinline__ double xpsi0(double z) { return z * z * (2.0 * z - 3.0) + 1.0; }
__device__ __forceinline__ double xpsi1(double z) { return z * (z * (z - 2.0) + 1.0); }

// Six weights of one variable: value at x and at 1-x for orders 0,1,2.
struct W6 {
    double w0, w1, w2, w0m, w1m, w2m;
};

// One column of a biquintic or bicubic sum: the four nodes' values a b c d
// (nodes (i,j) (i+1,j) (i,j+1) (i+1,j+1)) with the density weights (wd, wmd)
// and temperature weights (wt, wmt), added to acc in h5's term order (the
// first column starts the sum).
__device__ __forceinline__ void hcol(double &acc, bool first, double a, double b, double c, double d, double wd,
                                     double wmd, double wt, double wmt)
{
    acc = first ? a * wd * wt : acc + a * wd * wt;
    acc = acc + b * wmd * wt;
    acc = acc + c * wd * wmt;
    acc = acc + d * wmd * wmt;
}

// weight k (0, 1, 2) of a W6, and its m counterpart
__device__ __forceinline__ double wsel(const W6 &w, int k) { return k == 0 ? w.w0 : (k == 1 ? w.w1 : w.w2); }
__device__ __forceinline__ double wselm(const W6 &w, int k) { return k == 0 ? w.w0m : (k == 1 ? w.w1m : w.w2m); }

// Table cell of x on a logarithmic axis: (int)((log10(x) - lo) * stpi) + 1,
// clamped to 1..n (Source/eos.F90:229-244).  Except within 1/2048 of a grid
// line the single-precision logarithm decides it: over the table its error is
// below 8e-5 cells (of up to 541: 3e-5 the last rounding, 4e-5 those of the
// logarithm, its product and difference times 20 cells a decade).  There, and
// for anything but a positive normal number, log10 does; at 1/256 a third of the
// wavefronts ran both.
__device__ __forceinline__ int eos_cell(double x, double lo, double stpi, int n)
{
    const int h = __double2hiint(x);
    const int ex = (h >> 20) - 1023;
    const float m = __int_as_float(0x3f800000 | ((h & 0xfffff) << 3) | (int)((unsigned)__double2loint(x) >> 29));
    const float f = (((float)ex + __builtin_amdgcn_logf(m)) * 0.301029996f - (float)lo) * (float)stpi;
    const float r = f - floorf(f);
    int c = (int)f + 1;
    if (!(r > 0x1p-11f && r < 1.0f - 0x1p-11f && ex > -500 && ex < 500)) c = (int)((log10(x) - lo) * stpi) + 1;
    return c < 1 ? 1 : (c > n ? n : c);
}

// Density-side data of one EOS call (constant through the Newton solve).
struct EosDen {
    double den, deni, ytot1, ye, din, xd;
    int iat;
    W6 D;  // quintic weights (value)
};

__device__ __forceinline__ void eos_density(const EosTable &tab, double rho, double abar, double zbar,
                                            EosDen &s)
{
    s.den = rho;
    s.ytot1 = 1.0 / abar;
    s.ye = zbar / abar;
    s.din = s.ye * s.den;
    s.deni = 1.0 / s.den;
    s.iat = eos_cell(s.din, eosc::dlo, eosc::dstpi, EOS_IMAX - 1);
    const double *g = tab.dg + (long)(s.iat - 1) * EOS_GRID;
    const double dI = g[G_X], dd = g[G_D], dd2 = g[G_D2], ddi = g[G_DI];
    const double xd = fmax((s.din - dI) * ddi, 0.0);
    const double mxd = 1.0 - xd;
    s.xd = xd;
    s.D.w0 = psi0(xd);
    s.D.w1 = psi1(xd) * dd;
    s.D.w2 = psi2(xd) * dd2;
    s.D.w0m = psi0(mxd);
    s.D.w1m = -psi1(mxd) * dd;
    s.D.w2m = psi2(mxd) * dd2;
}

// Thermodynamic output of one evaluation.
struct EosFull {
    double p, e, dpdT, dpdr, dedT, dedr, gam1, dpde, dpdr_e;
};

// The four table rows of a cell, two columns (c2 = 0: columns 0 and 1, ...) at
// a time.
struct EosCols {
    double2 a, b, c, d;  // nodes (i,j) (i+1,j) (i,j+1) (i+1,j+1)
};
struct EosRows {
    const char *base;
    unsigned off;
    __device__ __forceinline__ EosCols load(int c2) const
    {
        const char *q = base + off + 16 * c2;
        return EosCols{*(const double2 *)q, *(const double2 *)(q + 8 * EOS_NODE),
                       *(const double2 *)(q + 8L * EOS_IMAX * EOS_NODE),
                       *(const double2 *)(q + 8L * EOS_IMAX * EOS_NODE + 8 * EOS_NODE)};
    }
};
// Pairs of columns loaded together.  A row is one cache line, and a
// wavefront's rows (4 per lane) can fill the vector L1: where lanes share no
// rows (mc_eos_eval_batch over unordered points) every group fetches the lines
// again.  1,000,000 such (rho, e) solves took 531, 508, 489 and 342 us with
// groups of 1 (one ahead), 2, 3 and 5; cells of a flow are indifferent
// (K_prim 2.9 ms, K_update 3.8 to 4.1 at 256^3), as are three wavefronts per
// SIMD, which groups of 1 allow.
constexpr int EOS_CHUNK = 5;
__device__ __forceinline__ EosRows eos_rows(const EosTable &tab, int iat, int jat)
{
    EosRows r;
    r.base = (const char *)tab.node;
    r.off = ((unsigned)(iat - 1) + (unsigned)EOS_IMAX * (unsigned)(jat - 1)) * (8u * EOS_NODE);
    return r;
}
// The next columns' address waits for the sums so far: without the tie the
// compiler gathers every column of every sum first (104 registers of table
// values, and one wavefront per SIMD or spills).
#define MC_EOS_STEP(r, s0, s1, s2) asm volatile("" : "+v"((r).off), "+v"(s0), "+v"(s1), "+v"(s2))

// columns' weights in the order of the node slots: density weight dsel,
// temperature weight tsel
__device__ constexpr int eos_dsel[9] = {0, 0, 0, 1, 2, 1, 2, 1, 2};
__device__ constexpr int eos_tsel[9] = {0, 1, 2, 0, 0, 1, 1, 2, 2};

// e and de/dT at temperature temp (Source/eos.F90:195-518): what a Newton
// iteration needs.
// The biquintic sums (Source/eos.F90:915-950) of the free energy and its
// derivatives run column by column: every sum adds the reference's terms in
// its order, EOS_CHUNK pairs of columns of the four nodes at a time.
__device__ __forceinline__ void eos_energy(const EosTable &tab, const EosDen &s, double temp, int &jat_out,
                                           EosFull &o)
{
    using namespace eosc;
    const double den = s.den, deni = s.deni, ytot1 = s.ytot1, ye = s.ye;
    const int jat = eos_cell(temp, tlo, tstpi, EOS_JMAX - 1);
    jat_out = jat;
    EosRows rows = eos_rows(tab, s.iat, jat);
    EosCols col[5];
    const double *g = tab.tg + (long)(jat - 1) * EOS_GRID;
    const double tJ = g[G_X], dt = g[G_D], dt2 = g[G_D2], dti = g[G_DI], dt2i = g[G_D2I];

    const double tempi = 1.0 / temp;
    const double prad = asoli3 * temp * temp * temp * temp;
    const double dpraddt = 4.0 * prad * tempi;
    const double erad = 3.0 * prad * deni;
    const double deraddt = 3.0 * dpraddt * deni;
    const double pion = kergavo * ytot1 * den * temp;
    const double dpiondt = kergavo * ytot1 * den;
    const double eion = 1.5 * pion * deni;
    const double deiondt = 1.5 * dpiondt * deni;

    const double xt = fmax((temp - tJ) * dti, 0.0);
    const double mxt = 1.0 - xt;
    W6 T, dT, ddT;
    T.w0 = psi0(xt);
    T.w1 = psi1(xt) * dt;
    T.w2 = psi2(xt) * dt2;
    T.w0m = psi0(mxt);
    T.w1m = -psi1(mxt) * dt;
    T.w2m = psi2(mxt) * dt2;
    dT.w0 = dpsi0(xt) * dti;
    dT.w1 = dpsi1(xt);
    dT.w2 = dpsi2(xt) * dt;
    dT.w0m = -dpsi0(mxt) * dti;
    dT.w1m = dpsi1(mxt);
    dT.w2m = -dpsi2(mxt) * dt;
    ddT.w0 = ddpsi0(xt) * dt2i;
    ddT.w1 = ddpsi1(xt) * dti;
    ddT.w2 = ddpsi2(xt);
    ddT.w0m = ddpsi0(mxt) * dt2i;
    ddT.w1m = -ddpsi1(mxt) * dti;
    ddT.w2m = ddpsi2(mxt);

    double free = 0.0, df_t = 0.0, df_tt = 0.0;
#pragma unroll
    for (int c2 = 0; c2 < 5; ++c2) {
        if (c2 % EOS_CHUNK == 0) {
            if (c2) MC_EOS_STEP(rows, free, df_t, df_tt);
#pragma unroll
            for (int l = c2; l < c2 + EOS_CHUNK && l < 5; ++l) col[l] = rows.load(l);
        }
        const EosCols cur = col[c2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int q = 2 * c2 + h;
            if (q >= 9) break;
            const double a = h ? cur.a.y : cur.a.x, b = h ? cur.b.y : cur.b.x, c = h ? cur.c.y : cur.c.x,
                         d = h ? cur.d.y : cur.d.x;
            const double wd = wsel(s.D, eos_dsel[q]), wmd = wselm(s.D, eos_dsel[q]);
            hcol(free, q == 0, a, b, c, d, wd, wmd, wsel(T, eos_tsel[q]), wselm(T, eos_tsel[q]));
            hcol(df_t, q == 0, a, b, c, d, wd, wmd, wsel(dT, eos_tsel[q]), wselm(dT, eos_tsel[q]));
            hcol(df_tt, q == 0, a, b, c, d, wd, wmd, wsel(ddT, eos_tsel[q]), wselm(ddT, eos_tsel[q]));
        }
    }

    const double sele = -df_t * ye;
    const double dsepdt = -df_tt * ye;
    const double eele = ye * free + temp * sele;
    const double deepdt = temp * dsepdt;
    o.e = erad + eion + eele;
    o.dedT = deraddt + deiondt + deepdt;
}

// The rest of an evaluation whose e and de/dT eos_energy left in o: pressure
// and its derivatives, de/drho, gamma_1.
__device__ __forceinline__ void eos_pressure(const EosTable &tab, const EosDen &s, double temp, int jat, EosFull &o)
{
    using namespace eosc;
    const double den = s.den, deni = s.deni, ytot1 = s.ytot1, ye = s.ye;
    EosRows rows = eos_rows(tab, s.iat, jat);
    EosCols col[7];
    const double *g = tab.tg + (long)(jat - 1) * EOS_GRID;
    const double tJ = g[G_X], dt = g[G_D], dt2 = g[G_D2], dti = g[G_DI];
    const double *gd = tab.dg + (long)(s.iat - 1) * EOS_GRID;
    const double dd = gd[G_D], ddi = gd[G_DI];
    const double xt = fmax((temp - tJ) * dti, 0.0);
    const double mxt = 1.0 - xt, xd = s.xd, mxd = 1.0 - s.xd;

    W6 T, dT, dD;
    T.w0 = psi0(xt);
    T.w1 = psi1(xt) * dt;
    T.w2 = psi2(xt) * dt2;
    T.w0m = psi0(mxt);
    T.w1m = -psi1(mxt) * dt;
    T.w2m = psi2(mxt) * dt2;
    dT.w0 = dpsi0(xt) * dti;
    dT.w1 = dpsi1(xt);
    dT.w2 = dpsi2(xt) * dt;
    dT.w0m = -dpsi0(mxt) * dti;
    dT.w1m = dpsi1(mxt);
    dT.w2m = -dpsi2(mxt) * dt;
    dD.w0 = dpsi0(xd) * ddi;
    dD.w1 = dpsi1(xd);
    dD.w2 = dpsi2(xd) * dd;
    dD.w0m = -dpsi0(mxd) * ddi;
    dD.w1m = dpsi1(mxd);
    dD.w2m = -dpsi2(mxd) * dd;

    // df_d, df_dt over the quintic columns, then the bicubic dpdf sum
    // (Source/eos.F90:1034-1059) over columns 9..12, in its order (d0, t0),
    // (d0, t1), (d1, t0), (d1, t1)
    double df_d = 0.0, df_dt = 0.0, dpepdd = 0.0;
#pragma unroll
    for (int c2 = 0; c2 < 7; ++c2) {
        if (c2 % EOS_CHUNK == 0) {
            if (c2) MC_EOS_STEP(rows, df_d, df_dt, dpepdd);
#pragma unroll
            for (int l = c2; l < c2 + EOS_CHUNK && l < 7; ++l) col[l] = rows.load(l);
        }
        const EosCols cur = col[c2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int q = 2 * c2 + h;
            if (q >= 13) break;
            const double a = h ? cur.a.y : cur.a.x, b = h ? cur.b.y : cur.b.x, c = h ? cur.c.y : cur.c.x,
                         d = h ? cur.d.y : cur.d.x;
            if (q < 9) {
                const double ed = wsel(dD, eos_dsel[q]), emd = wselm(dD, eos_dsel[q]);
                hcol(df_d, q == 0, a, b, c, d, ed, emd, wsel(T, eos_tsel[q]), wselm(T, eos_tsel[q]));
                hcol(df_dt, q == 0, a, b, c, d, ed, emd, wsel(dT, eos_tsel[q]), wselm(dT, eos_tsel[q]));
            } else {
                const bool d1 = q >= 11, t1 = q == 10 || q == 12;
                hcol(dpepdd, q == 9, a, b, c, d, d1 ? xpsi1(xd) * dd : xpsi0(xd), d1 ? -xpsi1(mxd) * dd : xpsi0(mxd),
                     t1 ? xpsi1(xt) * dt : xpsi0(xt), t1 ? -xpsi1(mxt) * dt : xpsi0(mxt));
            }
        }
    }
    dpepdd = fmax(ye * dpepdd, 0.0);

    const double tempi = 1.0 / temp;
    const double prad = asoli3 * temp * temp * temp * temp;
    const double dpraddt = 4.0 * prad * tempi;
    const double erad = 3.0 * prad * deni;
    const double pion = kergavo * ytot1 * den * temp;
    const double dpiondd = kergavo * ytot1 * temp;
    const double dpiondt = kergavo * ytot1 * den;
    const double eion = 1.5 * pion * deni;
    const double deraddd = -erad * deni;
    const double deiondd = (1.5 * dpiondd - eion) * deni;
    double x = s.din * s.din;
    const double pele = x * df_d;
    const double dpepdt = x * df_dt;
    x = ye * ye;
    const double dsepdd = -df_dt * x;
    const double deepdd = x * df_d + temp * dsepdd;

    const double pres = prad + pion + pele;
    const double dpresdd = 0.0 + dpiondd + dpepdd;
    const double dpresdt = dpraddt + dpiondt + dpepdt;
    const double denerdd = deraddd + deiondd + deepdd;
    const double denerdt = o.dedT;

    const double zz = pres * deni;
    const double zzi = den / pres;
    const double chit = temp / pres * dpresdt;
    const double chid = dpresdd * zzi;
    o.gam1 = chit * zz * chit / (temp * denerdt) + chid;
    o.p = pres;
    o.dpdT = dpresdt;
    o.dpdr = dpresdd;
    o.dpde = dpresdt / denerdt;
    o.dpdr_e = dpresdd - dpresdt * denerdd / denerdt;
    o.dedr = denerdd;
}
#undef MC_EOS_STEP

// e and de/dT of one state.  eos_rt_e calls this, not eos_energy, which changes the
// order in which the compiler inlines: the same arithmetic, but K_prim of 256^3 takes
// 3.10 ms with the direct call and 2.96 so.
__device__ __forceinline__ void eos_eval(const EosTable &tab, const EosDen &s, double temp, int &jat, EosFull &o)
{
    eos_energy(tab, s, temp, jat, o);
}

// Result of a (rho, e) solve.
struct EosRE {
    double T, p, gam1, cs, dpde, dpdr_e;
    int iat, jat, niter;
};

// One Newton step on T with the reference's clamps (Source/eos.F90:524-550);
// true when it has converged.  |dT / T| < ttol is decided without the
// division unless it is within rounding of the tolerance.
__device__ __forceinline__ bool eos_newton(double &temp, double f, double want, double dfdT)
{
    const double temp_old = temp;
    temp = temp - (f - want) / dfdT;
    temp = fmax(0.5 * temp_old, fmin(temp, 2.0 * temp_old));
    temp = fmax(eosc::mintemp, temp);
    const double d = fabs(temp - temp_old), t = eosc::ttol * fabs(temp_old);
    bool ok = d < t;
    if (!(d < t * (1.0 - 1.0e-12) || d > t * (1.0 + 1.0e-12))) ok = fabs((temp - temp_old) / temp_old) < eosc::ttol;
    return ok;
}

// eos(eos_input_re, ...): Newton on T for e.  FULL=false when the caller only
// needs T (compute_temp restores e and discards everything else).  As in the
// reference, the evaluation after convergence is the one the outputs come
// from; only that one computes the pressure (the last of a solve that does
// not converge steps on after it).
template <bool FULL>
__device__ __forceinline__ EosRE eos_re(const EosTable &tab, double rho, double T0, double e_want, double abar,
                                        double zbar)
{
    EosDen s;
    eos_density(tab, rho, abar, zbar, s);
    double temp = T0, teval = T0;
    bool converged = false;
    EosFull o;
    int jat = 0, iter;
    for (iter = 1; iter <= EOS_MAX_NEWTON; ++iter) {
        if (!FULL && converged) break;
        teval = temp;
        eos_energy(tab, s, temp, jat, o);
        if (converged) break;
        converged = eos_newton(temp, o.e, e_want, o.dedT);
    }
    if (!converged) eos_note_newton_failure(tab);
    if (FULL) eos_pressure(tab, s, teval, jat, o);
    EosRE r;
    r.niter = iter > EOS_MAX_NEWTON ? EOS_MAX_NEWTON : iter;
    r.T = temp;
    r.iat = s.iat;
    r.jat = jat;
    if (FULL) {
        r.p = o.p;
        r.gam1 = o.gam1;
        r.cs = sqrt(o.gam1 * o.p / rho);
        r.dpde = o.dpde;
        r.dpdr_e = o.dpdr_e;
    }
    return r;
}

// eos(eos_input_rt, ...) for the floors: returns e (Source/eos.F90, converged at entry).
__device__ __forceinline__ double eos_rt_e(const EosTable &tab, double rho, double T, double abar, double zbar)
{
    EosDen s;
    eos_density(tab, rho, abar, zbar, s);
    EosFull o;
    int jat;
    eos_eval(tab, s, T, jat, o);
    return o.e;
}

} // namespace mc
