// EOS evaluations that stand alone, outside the hydro kernels: energy and
// pressure from one reading of the table (batches, the problem set-up).
//
// mc_eos.h takes the two apart for the registers of kernels that hold a cell's
// state, and reads the table for each.  A batch that does not fill the chip waits
// for one reading after another, and a large one of unordered points for the
// lines its rows lie in.  So the grid entries are read ahead of the rows, whose
// weights are formed while the rows come.
// 5419 (rho, p) solves 16.0 us, 1,000,000 232 (in two readings an iteration 19.0 and
// 250; p and dp/dT alone and e once at the end 17.6 and 204); 1,000,000 (rho, T) evaluations
// 95.7 us, in two readings 124.
#pragma once

#include "mc_eos.h"

namespace mc {

// One row's columns after another's: a wavefront's loads of one row meet in its
// lines while the vector L1 has them.  Left to order them, the compiler takes pairs
// of columns in turn, each over all four rows (us, ordered and not: (rho, T)
// evaluations of 1,000,000 points 95.7 and 104, of 60,000 9.7 and 10.2, of 20,000 and
// fewer the same; 5419 (rho, p) solves 16.0 and 16.6).
template <int PAIRS>
__device__ __forceinline__ void eos_load_rows(const EosRows &r, EosCols (&col)[PAIRS])
{
    auto row = [&](auto put, long node) {
#pragma unroll
        for (int l = 0; l < PAIRS; ++l) put(col[l]) = *(const double2 *)(r.base + r.off + 16 * l + node);
        asm volatile("" ::: "memory");
    };
    row([](EosCols &c) -> double2 & { return c.a; }, 0);
    row([](EosCols &c) -> double2 & { return c.b; }, 8 * EOS_NODE);
    row([](EosCols &c) -> double2 & { return c.c; }, 8L * EOS_IMAX * EOS_NODE);
    row([](EosCols &c) -> double2 & { return c.d; }, 8L * EOS_IMAX * EOS_NODE + 8 * EOS_NODE);
}

// At temperature temp (Source/eos.F90:195-518), with eos_energy's and
// eos_pressure's expressions: everything (FULL), or e, p and dp/dT.  dd, ddi: the
// density's grid entry.
template <bool FULL>
__device__ __forceinline__ void eos_once(const EosTable &tab, const EosDen &s, double dd, double ddi, double temp,
                                         int &jat_out, EosFull &o)
{
    using namespace eosc;
    constexpr int PAIRS = FULL ? 7 : 5;
    const double den = s.den, deni = s.deni, ytot1 = s.ytot1, ye = s.ye;
    const int jat = eos_cell(temp, tlo, tstpi, EOS_JMAX - 1);
    jat_out = jat;
    const double *g = tab.tg + (long)(jat - 1) * EOS_GRID;
    const double tJ = g[G_X], dt = g[G_D], dt2 = g[G_D2], dti = g[G_DI], dt2i = g[G_D2I];
    EosCols col[PAIRS];
    eos_load_rows(eos_rows(tab, s.iat, jat), col);

    const double tempi = 1.0 / temp;
    const double prad = asoli3 * temp * temp * temp * temp;
    const double dpraddt = 4.0 * prad * tempi;
    const double erad = 3.0 * prad * deni;
    const double pion = kergavo * ytot1 * den * temp;
    const double dpiondt = kergavo * ytot1 * den;
    const double eion = 1.5 * pion * deni;
    const double xt = fmax((temp - tJ) * dti, 0.0);
    const double mxt = 1.0 - xt, xd = s.xd, mxd = 1.0 - s.xd;
    W6 T, dT, ddT, dD;
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
    dD.w0 = dpsi0(xd) * ddi;
    dD.w1 = dpsi1(xd);
    dD.w2 = dpsi2(xd) * dd;
    dD.w0m = -dpsi0(mxd) * ddi;
    dD.w1m = dpsi1(mxd);
    dD.w2m = -dpsi2(mxd) * dd;

    double free = 0.0, df_t = 0.0, df_tt = 0.0, df_d = 0.0, df_dt = 0.0, dpepdd = 0.0;
#pragma unroll
    for (int q = 0; q < (FULL ? 13 : 9); ++q) {
        const EosCols &v = col[q / 2];
        const double a = q % 2 ? v.a.y : v.a.x, b = q % 2 ? v.b.y : v.b.x, c = q % 2 ? v.c.y : v.c.x,
                     d = q % 2 ? v.d.y : v.d.x;
        if (q < 9) {
            const double wd = wsel(s.D, eos_dsel[q]), wmd = wselm(s.D, eos_dsel[q]);
            const double ed = wsel(dD, eos_dsel[q]), emd = wselm(dD, eos_dsel[q]);
            hcol(free, q == 0, a, b, c, d, wd, wmd, wsel(T, eos_tsel[q]), wselm(T, eos_tsel[q]));
            hcol(df_t, q == 0, a, b, c, d, wd, wmd, wsel(dT, eos_tsel[q]), wselm(dT, eos_tsel[q]));
            if (FULL) hcol(df_tt, q == 0, a, b, c, d, wd, wmd, wsel(ddT, eos_tsel[q]), wselm(ddT, eos_tsel[q]));
            hcol(df_d, q == 0, a, b, c, d, ed, emd, wsel(T, eos_tsel[q]), wselm(T, eos_tsel[q]));
            hcol(df_dt, q == 0, a, b, c, d, ed, emd, wsel(dT, eos_tsel[q]), wselm(dT, eos_tsel[q]));
        } else {
            const bool d1 = q >= 11, t1 = q == 10 || q == 12;
            hcol(dpepdd, q == 9, a, b, c, d, d1 ? xpsi1(xd) * dd : xpsi0(xd), d1 ? -xpsi1(mxd) * dd : xpsi0(mxd),
                 t1 ? xpsi1(xt) * dt : xpsi0(xt), t1 ? -xpsi1(mxt) * dt : xpsi0(mxt));
        }
    }

    const double sele = -df_t * ye;
    o.e = erad + eion + (ye * free + temp * sele);
    double x = s.din * s.din;
    const double pele = x * df_d;
    const double dpepdt = x * df_dt;
    o.p = prad + pion + pele;
    o.dpdT = dpraddt + dpiondt + dpepdt;
    if (!FULL) return;

    const double dsepdt = -df_tt * ye;
    const double deraddt = 3.0 * dpraddt * deni;
    const double deiondt = 1.5 * dpiondt * deni;
    o.dedT = deraddt + deiondt + temp * dsepdt;
    dpepdd = fmax(ye * dpepdd, 0.0);
    const double dpiondd = kergavo * ytot1 * temp;
    const double deraddd = -erad * deni;
    const double deiondd = (1.5 * dpiondd - eion) * deni;
    x = ye * ye;
    const double dsepdd = -df_dt * x;
    const double deepdd = x * df_d + temp * dsepdd;
    o.dpdr = 0.0 + dpiondd + dpepdd;
    o.dedr = deraddd + deiondd + deepdd;
    const double zz = o.p * deni;
    const double zzi = den / o.p;
    const double chit = temp / o.p * o.dpdT;
    const double chid = o.dpdr * zzi;
    o.gam1 = chit * zz * chit / (temp * o.dedT) + chid;
    o.dpde = o.dpdT / o.dedT;
    o.dpdr_e = o.dpdr - o.dpdT * o.dedr / o.dedT;
}

// eos(eos_input_rt, ...) with every output
__device__ __forceinline__ void eos_rt(const EosTable &tab, const EosDen &s, double temp, int &jat, EosFull &o)
{
    const double *gd = tab.dg + (long)(s.iat - 1) * EOS_GRID;
    eos_once<true>(tab, s, gd[G_D], gd[G_DI], temp, jat, o);
}

// eos(eos_input_rp, ...): Newton on T for a target pressure; returns e.
__device__ __forceinline__ double eos_rp_e(const EosTable &tab, double rho, double T0, double p_want, double abar,
                                           double zbar, double *T_out)
{
    EosDen s;
    eos_density(tab, rho, abar, zbar, s);
    const double *gd = tab.dg + (long)(s.iat - 1) * EOS_GRID;
    const double dd = gd[G_D], ddi = gd[G_DI];
    double temp = T0;
    bool converged = false;
    EosFull o;
    int jat;
    for (int iter = 1; iter <= EOS_MAX_NEWTON; ++iter) {
        eos_once<false>(tab, s, dd, ddi, temp, jat, o);
        if (converged) break;
        converged = eos_newton(temp, o.p, p_want, o.dpdT);
    }
    if (!converged) eos_note_newton_failure(tab);
    if (T_out) *T_out = temp;
    return o.e;
}

} // namespace mc
