// Discrete adjoint of the fused CTU step (one instance) on gfx950.
//
// Forward pass: the fused engine advances the state with a given dt
// sequence, storing the state at the start of every step (checkpoints).
// Reverse pass, step n = N-1 .. 0: the step is recomputed from its
// checkpoint (every stage's outputs are then resident in the engine's
// arrays), and the stages are reversed in the opposite order:
//
//   A_update  cells   clean_state x2, S_new = S_old + dt src, clean(S_old)
//   A_final   faces   apply_av, final Riemann, trans2
//   A_trans1  faces   Riemann of the trans1 states, trans1
//   A_flux1   faces   Riemann of the PPM states
//   A_trace   cells+1 characteristic projection, PPM integrals, PPM edges
//   A_flat    cells+1 flattening, node-centred div(u)
//   A_prim    cells   ctoprim, clean_state x2
//
// Each thread re-evaluates its forward stencil point.  What a stage owes the
// fluxes it read is stored zone by zone and gathered by the stage that made
// them, and states and zones are written by their one owner; what is left,
// the zones a trace, the viscosity or the boundary map reaches, is scattered
// with hardware FP64 atomic adds.  The
// adjoint carries the hydro components of the state (rho, rho u, rho v,
// rho w, rho E, rho e); see mc_adjoint.h for why T and the species are
// constants of the differentiated map.
#include <float.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <vector>

#include "../../include/mc_castro.h"
#include "mc_adjoint.h"
#include "mc_cell.h"
#include "mc_common.h"
#include "mc_eos.h"
#include "mc_fused.h"
#include "mc_fused_impl.h"
#include "mc_hydro.h"
#include "mc_internal.h"

namespace mc {

// adjoint component layouts
enum { SB_RHO = 0, SB_U, SB_V, SB_W, SB_P, SB_RE, NSB };            // interface states
enum { ZB_PGP = UEDEN + 1, ZB_PGM, ZB_UGP, ZB_UGM, NZB };  // fluxes across a zone
enum { NB_RHO = 0, NB_MX, NB_MY, NB_MZ, NB_E, NB_EI, NB_GP, NB_GU, NNB };  // final fluxes

struct ACtx {
    const double *Uold;  // checkpoint of the step (NVAR, cell layout)
    double *Ub;          // adjoint of the step's output state (NHB, cell layout)
    double *Ubo;         // adjoint of the step's input state (NHB, cell layout)
    double *Sb;          // adjoint of the update's sources, dt times (NHB, cell layout)
    double *U1b, *Qb, *DVb;
    double *QD[3];       // the primitives' share of direction d's traces (NQB, cell layout)
    double *FLb[3], *SMb[3], *SPb[3];
    double *ZF[6], *ZT[6];  // of F^{t|d} and of F^d (pair t, d), by the zone between the two faces
    double *CG[3];          // c and Gamma_1, by the zone, from the states of direction d ..
    double *CGF[3];         // .. and from F^d's faces: left c, Gamma_1, right c, Gamma_1
};

// device-scope FP64 atomic add (the hardware global_atomic_add_f64)
__device__ __forceinline__ void aadd(gdouble *p, double v)
{
    if (v != 0.0) {
        [[clang::atomic(ignore_denormal_mode)]] {
            (void)__hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}
__device__ __forceinline__ gdouble *EAp(double *a, const FInst &I, int C, int c, idx_t idx)
{
    return &at(a + ((long)C * I.offE + (long)c * I.nE), idx);
}
__device__ __forceinline__ gdouble *CAp(double *a, const FInst &I, int C, int c, idx_t idx)
{
    return &at(a + ((long)C * I.offD + (long)c * I.nD), idx);
}

// ------------------------------------------------------------------ A_update
__global__ __launch_bounds__(256) void A_update(Plan p, Ctx x, ACtx a)
{
    int m, i, j, k;
    if (!plan_cell(p, m, i, j, k)) return;
    const FInst &I = p.inst[m];
    const idx_t c = cidx(I, i, j, k);
    const double dx0 = I.dx[0], dx1 = I.dx[1], dx2 = I.dx[2];
    const double a0 = dx1 * dx2, a1 = dx0 * dx2, a2 = dx0 * dx1;
    const double volinv = 1.0 / (dx0 * dx1 * dx2);
    const idx_t e = eidx(I, i, j, k);
    const idx_t ex = eidx(I, i + 1, j, k), ey = eidx(I, i, j + 1, k), ez = eidx(I, i, j, k + 1);
    double *F0 = x.FN[0], *F1 = x.FN[1], *F2 = x.FN[2];
    const double dt = x.dt_cur[m];
    double u0[NVAR], ua[NVAR], u1[NVAR], u2[NVAR];
#pragma unroll
    for (int n = 0; n < NVAR; ++n) u0[n] = a.Uold[(long)NVAR * I.offD + (long)n * I.nD + c];
#pragma unroll
    for (int n = 0; n < NVAR; ++n) ua[n] = u0[n];
    clean_hydro(ua, x.tab);
    const SpeciesPairs P0 = species_pairs(F0, I, NFN, FN_X), P1 = species_pairs(F1, I, NFN, FN_X),
                       P2 = species_pairs(F2, I, NFN, FN_X);
    const double c0 = species_fac(P0, e, EF(F0, I, NFN, URHO, e)), c0x = species_fac(P0, ex, EF(F0, I, NFN, URHO, ex)),
                 c1 = species_fac(P1, e, EF(F1, I, NFN, URHO, e)), c1y = species_fac(P1, ey, EF(F1, I, NFN, URHO, ey)),
                 c2 = species_fac(P2, e, EF(F2, I, NFN, URHO, e)), c2z = species_fac(P2, ez, EF(F2, I, NFN, URHO, ez));
#pragma unroll
    for (int pr = 0; pr < NSPEC_PAIRS; ++pr) {
        const dbl2 f0 = SP2(P0, pr, e) * c0, f0x = SP2(P0, pr, ex) * c0x, f1 = SP2(P1, pr, e) * c1,
                   f1y = SP2(P1, pr, ey) * c1y, f2 = SP2(P2, pr, e) * c2, f2z = SP2(P2, pr, ez) * c2z;
        const int n = UFS + 2 * pr;
        u1[n] = ua[n] + dt * flux_div(f0.x, f0x.x, f1.x, f1y.x, f2.x, f2z.x, a0, a1, a2, volinv);
        if (n + 1 < NVAR) u1[n + 1] = ua[n + 1] + dt * flux_div(f0.y, f0x.y, f1.y, f1y.y, f2.y, f2z.y, a0, a1, a2, volinv);
    }
    u1[UTEMP] = ua[UTEMP];  // no flux
#pragma unroll
    for (int n = 0; n < UTEMP; ++n) {
        double s = flux_div(EF(F0, I, NFN, n, e), EF(F0, I, NFN, n, ex), EF(F1, I, NFN, n, e), EF(F1, I, NFN, n, ey),
                            EF(F2, I, NFN, n, e), EF(F2, I, NFN, n, ez), a0, a1, a2, volinv);
        if (n == UEINT) {
            const double pdivu = HALF * (EF(F0, I, NFN, FN_GP, ex) + EF(F0, I, NFN, FN_GP, e)) *
                                     (EF(F0, I, NFN, FN_GU, ex) - EF(F0, I, NFN, FN_GU, e)) / dx0 +
                                 HALF * (EF(F1, I, NFN, FN_GP, ey) + EF(F1, I, NFN, FN_GP, e)) *
                                     (EF(F1, I, NFN, FN_GU, ey) - EF(F1, I, NFN, FN_GU, e)) / dx1 +
                                 HALF * (EF(F2, I, NFN, FN_GP, ez) + EF(F2, I, NFN, FN_GP, e)) *
                                     (EF(F2, I, NFN, FN_GU, ez) - EF(F2, I, NFN, FN_GU, e)) / dx2;
            s = s - pdivu;
        }
        u1[n] = ua[n] + dt * s;
    }
#pragma unroll
    for (int n = 0; n < NVAR; ++n) u2[n] = u1[n];
    clean_hydro(u2, x.tab);

    double ub[NHB];
#pragma unroll
    for (int h = 0; h < NHB; ++h) ub[h] = CA(a.Ub, I, NHB, h, c);
    clean_cell_b(u2, x.tab, ub);  // post_timestep clean
    clean_cell_b(u1, x.tab, ub);  // clean after the update
    // u1 = ua + dt s
    double sb[NHB];
#pragma unroll
    for (int h = 0; h < NHB; ++h) sb[h] = dt * ub[h];
    clean_cell_b(u0, x.tab, ub);  // S_old clean
#pragma unroll
    for (int h = 0; h < NHB; ++h) CA(a.Ubo, I, NHB, h, c) = ub[h];

#pragma unroll
    for (int h = 0; h < NHB; ++h) CA(a.Sb, I, NHB, h, c) = sb[h];
}

// ------------------------------------------------------------------ helpers
// Riemann adjoint at face (i,j,k) of direction d; the c / gamma_c adjoints of
// its two cells in cg: left c, right c, left gamma_c, right gamma_c.
__device__ __forceinline__ void face_riemann_hb(const Ctx &x, const FInst &I, int d, int i, int j, int k,
                                                const FaceH &L, const FaceH &R, const RiemannHB &rb, FaceHB &Lb,
                                                FaceHB &Rb, double *cg)
{
    const idx_t cr = cidx(I, i, j, k);
    const idx_t cl = cidx(I, i - (d == 0), j - (d == 1), k - (d == 2));
    Lb = Rb = FaceHB{0, 0, 0, 0, 0, 0};
    cg[0] = cg[1] = cg[2] = cg[3] = 0.0;
    riemann_hydro_b(L, R, CA(x.Q, I, NFQ, FQ_C, cl), CA(x.Q, I, NFQ, FQ_C, cr), CA(x.Q, I, NFQ, FQ_G, cl),
                    CA(x.Q, I, NFQ, FQ_G, cr), rb, Lb, Rb, cg[0], cg[1], cg[2], cg[3]);
}

// a value by direction (of values: a choice between members would keep their
// structure in memory)
__device__ __forceinline__ double pick(int d, double x, double y, double z) { return d == 0 ? +x : (d == 1 ? +y : +z); }

// FaceHB (velocities permuted to direction d) -> absolute-order state adjoint
__device__ __forceinline__ QStateHB from_faceb(const FaceHB &f, int d)
{
    QStateHB o;
    o.rho = f.rho;
    o.p = f.p;
    o.rhoe = f.rhoe;
    // to_face: un = (u,v,w)[d]; ut = d==0 ? v : u; utt = d==2 ? v : w
    o.u = pick(d, f.un, f.ut, f.ut);
    o.v = pick(d, f.ut, f.un, f.utt);
    o.w = pick(d, f.utt, f.utt, f.un);
    return o;
}

// The adjoints of states and of zones' fluxes lie in pairs as the face arrays
// do (EF2): one access moves two components (A_flux1 at 64^3: 133 us, by single
// components 168).
__device__ __forceinline__ void load_stateb(double *S, const FInst &I, idx_t e, QInHB &b)
{
    const dbl2 ru = EF2(S, I, NSB, SB_RHO, e), vw = EF2(S, I, NSB, SB_V, e), pe = EF2(S, I, NSB, SB_P, e);
    b = QInHB{ru.x, ru.y, vw.x, vw.y, pe.x, pe.y};
}
__device__ __forceinline__ void store_stateb(double *S, const FInst &I, idx_t e, const QInHB &b)
{
    EF2(S, I, NSB, SB_RHO, e) = dbl2{b.rho, b.u};
    EF2(S, I, NSB, SB_V, e) = dbl2{b.v, b.w};
    EF2(S, I, NSB, SB_P, e) = dbl2{b.p, b.rhoe};
}

// into a d-face state that this thread alone has in the launch
__device__ __forceinline__ void add_faceb(double *S, const FInst &I, idx_t e, int d, const FaceHB &f)
{
    const QStateHB o = from_faceb(f, d);
    QInHB b;
    load_stateb(S, I, e, b);
    store_stateb(S, I, e, QInHB{b.rho + o.rho, b.u + o.u, b.v + o.v, b.w + o.w, b.p + o.p, b.rhoe + o.rhoe});
}

// Adjoint of the fluxes across a zone (ZB_*): the conserved fluxes enter as
// right less left, so one set serves both faces; Godunov p and u each side.
// (in pairs: two of momenta and rho, p and u of the high face, of the low; E)
__device__ __forceinline__ void store_zoneb(double *Z, const FInst &I, idx_t e, const double (&v)[NZB])
{
    EF2(Z, I, NZB, 0, e) = dbl2{v[URHO], v[UMX]};
    EF2(Z, I, NZB, 2, e) = dbl2{v[UMY], v[UMZ]};
    EA(Z, I, NZB, 8, e) = v[UEDEN];
    EF2(Z, I, NZB, 4, e) = dbl2{v[ZB_PGP], v[ZB_UGP]};
    EF2(Z, I, NZB, 6, e) = dbl2{v[ZB_PGM], v[ZB_UGM]};
}
struct FluxB {
    double rho, mx, my, mz, E, gp, gu;
};
// added to v: what face e owes the zones on its two sides, el and e; has_l,
// has_r: which of them had it
__device__ __forceinline__ void gather_zoneb(double *Z, const FInst &I, idx_t el, idx_t e, bool has_l, bool has_r,
                                             FluxB &v)
{
    if (has_l) {
        const dbl2 f = EF2(Z, I, NZB, 0, el), g = EF2(Z, I, NZB, 2, el), h = EF2(Z, I, NZB, 4, el);
        v.rho += f.x;
        v.mx += f.y;
        v.my += g.x;
        v.mz += g.y;
        v.E += EA(Z, I, NZB, 8, el);
        v.gp += h.x;
        v.gu += h.y;
    }
    if (has_r) {
        const dbl2 f = EF2(Z, I, NZB, 0, e), g = EF2(Z, I, NZB, 2, e), h = EF2(Z, I, NZB, 6, e);
        v.rho -= f.x;
        v.mx -= f.y;
        v.my -= g.x;
        v.mz -= g.y;
        v.E -= EA(Z, I, NZB, 8, e);
        v.gp += h.x;
        v.gu += h.y;
    }
}
// as the adjoint of a Riemann problem's outputs on a d-face
__device__ __forceinline__ RiemannHB riemannb_of(const FluxB &v, int d)
{
    RiemannHB r;
    r.f_rho = v.rho;
    r.f_mn = pick(d, v.mx, v.my, v.mz);
    r.f_mt = pick(d, v.my, v.mx, v.mx);
    r.f_mtt = pick(d, v.mz, v.mz, v.my);
    r.f_E = v.E;
    r.f_e = 0.0;
    r.g_p = v.gp;
    r.g_un = v.gu;
    return r;
}

// What follows is addressed through e, which waits for f: the forward values
// are read again behind the Riemann problem instead of being kept across it.
__device__ __forceinline__ void behind(idx_t &e, FaceHB &f)
{
    asm volatile("" : "+v"(e), "+v"(f.rho), "+v"(f.un), "+v"(f.ut), "+v"(f.utt), "+v"(f.p), "+v"(f.rhoe));
}
__device__ __forceinline__ void behind(idx_t &e, QInHB &f)
{
    asm volatile("" : "+v"(e), "+v"(f.rho), "+v"(f.u), "+v"(f.v), "+v"(f.w), "+v"(f.p), "+v"(f.rhoe));
}

// Bricks of L zones along a direction d, W across (256 threads: (L, W, 1) for
// x, (W, L, 1) for y, (W, 1, L) for z), over the zones -1..n along d and
// -ring..n-1+ring across; consecutive bricks share ovl zones along d.
struct Lines {
    int ring, ovl;
    int L[3], W[3], nb0[3], nb1[3], nb[3];
};
__device__ __forceinline__ bool line_cell(const Lines &q, int d, int lb, const FInst &I, int &i, int &j, int &k, int &l)
{
    const int L = q.L[d], W = q.W[d], t = threadIdx.x, r = q.ring;
    const int b0 = lb % q.nb0[d], b1 = (lb / q.nb0[d]) % q.nb1[d], b2 = lb / (q.nb0[d] * q.nb1[d]);
    const int s = L - q.ovl;
    if (d == 0) {
        l = t % L;
        i = b0 * s + l - 1;
        j = b1 * W + t / L - r;
        k = b2 - r;
    } else {
        l = t / W;
        i = b0 * W + t % W - r;
        j = d == 1 ? b1 * s + l - 1 : b1 - r;
        k = d == 1 ? b2 - r : b2 * s + l - 1;
    }
    const int h0 = I.n[0] + (d == 0 ? 1 : r), h1 = I.n[1] + (d == 1 ? 1 : r), h2 = I.n[2] + (d == 2 ? 1 : r);
    return i < h0 && j < h1 && k < h2;
}

// ------------------------------------------------------------------ A_final
// Final fluxes of direction d: apply_av, the Riemann problem, trans2.  The
// thread of zone c re-evaluates its two d-states (the plus state of d-face c,
// the minus state of d-face c + 1) from the zone's transverse fluxes, read
// once; the minus side goes up through LDS, the thread of a face reverses its
// Riemann problem and its viscosity, and the minus side's share comes back
// down.  Bricks share two zones along d, so that one thread has both faces of
// every zone and owns what the zone gives.  64^3: 250 us; by faces, with an
// atomic add for each of the 74 adjoints a face gives, 603 (atomics come at 92
// to 97 a nanosecond).  Two waves a SIMD wait for memory now: without the
// stores it takes 181, without the Riemann problem 216.
__global__ __launch_bounds__(256) void A_final(Lines q, const FInst *inst, Ctx x, ACtx a)
{
    __shared__ double ls[6][256], lr[14][256];
    int lb = logical_block();
    const int d = lb % 3;
    lb /= 3;
    if (lb >= q.nb[d]) return;  // the whole block
    const FInst &I = inst[0];
    int i, j, k, l;
    const bool ok = line_cell(q, d, lb, I, i, j, k, l);
    const int tid = threadIdx.x, st = d == 0 ? 1 : q.W[d], top = q.L[d] - 1, nd = I.n[d];
    const int t1 = d == 0 ? 1 : 0, t2 = d == 2 ? 1 : 2;
    const int cd = d == 0 ? i : (d == 1 ? j : k);
    const int ei = d == 0, ej = d == 1, ek = d == 2;
    const bool has_p = ok && cd >= 0, has_m = ok && cd + 1 <= nd;  // the zone's plus and minus states
    const idx_t ep = eidx(I, i, j, k), em = eidx(I, i + ei, j + ej, k + ek);
    const idx_t r2 = eidx(I, i + (t1 == 0), j + (t1 == 1), k), r3 = eidx(I, i, j + (t2 == 1), k + (t2 == 2));
    const double dt = x.dt_cur[0];
    const double h2 = 0.5 * dt / I.dx[t1], h3 = 0.5 * dt / I.dx[t2];
    const int p2 = pair_index(t1, t2), p3 = pair_index(t2, t1);
    double f2r[UEDEN + 1], f2l[UEDEN + 1], f3r[UEDEN + 1], f3l[UEDEN + 1], pg2p, ug2p, pg2m, ug2m, pg3p, ug3p, pg3m,
        ug3m, gamc = 0.0;
    QInH qm, qp;
    FaceH side_p{};
    if (ok) {
        load_tflux_h(x.FT[p2], I, r2, f2r, pg2p, ug2p);
        load_tflux_h(x.FT[p2], I, ep, f2l, pg2m, ug2m);
        load_tflux_h(x.FT[p3], I, r3, f3r, pg3p, ug3p);
        load_tflux_h(x.FT[p3], I, ep, f3l, pg3m, ug3m);
        gamc = CA(x.Q, I, NFQ, FQ_G, cidx(I, i, j, k));
        if (has_m) {
            load_qin_h(x.SM[d], I, em, qm);
            const FaceH f = to_face(trans2_hydro(qm, f2r, f2l, f3r, f3l, pg2p, pg2m, ug2p, ug2m, pg3p, pg3m, ug3p,
                                                 ug3m, gamc, h2, h3), d);
            ls[0][tid] = f.rho;
            ls[1][tid] = f.un;
            ls[2][tid] = f.ut;
            ls[3][tid] = f.utt;
            ls[4][tid] = f.p;
            ls[5][tid] = f.rhoe;
        }
        if (has_p) {
            load_qin_h(x.SP[d], I, ep, qp);
            side_p = to_face(trans2_hydro(qp, f2r, f2l, f3r, f3l, pg2p, pg2m, ug2p, ug2m, pg3p, pg3m, ug3p, ug3m,
                                          gamc, h2, h3), d);
        }
    }
    __syncthreads();
    FaceHB Lb{}, Rb{};
    double cg[4] = {0.0, 0.0, 0.0, 0.0}, g[NHB] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    if (has_p && l > 0) {
        const int tb = tid - st;
        const FaceH side_m{ls[0][tb], ls[1][tb], ls[2][tb], ls[3][tb], ls[4][tb], ls[5][tb]};
        // the update: a face is the low face of zone cd, the high face of cd - 1
        const idx_t cr = cidx(I, i, j, k), cl = cidx(I, i - ei, j - ej, k - ek);
        const bool in_r = cd < nd, in_l = cd > 0;
        const double dx0 = I.dx[0], dx1 = I.dx[1], dx2 = I.dx[2], dxd = I.dx[d];
        const double av = (d == 0 ? dx1 * dx2 : (d == 1 ? dx0 * dx2 : dx0 * dx1)) * (1.0 / (dx0 * dx1 * dx2));
        double fnb[NNB];
#pragma unroll
        for (int h = 0; h < NHB; ++h) {
            double v = 0.0;
            if (in_r) v += CA(a.Sb, I, NHB, h, cr) * av;
            if (in_l) v -= CA(a.Sb, I, NHB, h, cl) * av;
            fnb[h] = v;
        }
        // pdivu term of rho e: s -= 0.5 (GP+ + GP-) (GU+ - GU-) / dx_d
        double *F = x.FN[d];
        const dbl2 g0 = EF2(F, I, NFN, FN_GP, ep);
        fnb[NB_GP] = fnb[NB_GU] = 0.0;
        if (in_r) {
            const dbl2 gp = EF2(F, I, NFN, FN_GP, em);
            const double b = -CA(a.Sb, I, NHB, HB_EI, cr) / dxd;
            fnb[NB_GP] += b * HALF * (gp.y - g0.y);
            fnb[NB_GU] -= b * HALF * (gp.x + g0.x);
        }
        if (in_l) {
            const dbl2 gm = EF2(F, I, NFN, FN_GP, eidx(I, i - ei, j - ej, k - ek));
            const double b = -CA(a.Sb, I, NHB, HB_EI, cl) / dxd;
            fnb[NB_GP] += b * HALF * (g0.y - gm.y);
            fnb[NB_GU] += b * HALF * (g0.x + gm.x);
        }
        // artificial viscosity (forward: Source/Castro_hydro_nd.F90:174-245)
        const idx_t na = eidx(I, i + (d != 0), j + (d == 0), k);
        const idx_t nb = d == 2 ? eidx(I, i, j + 1, k) : eidx(I, i, j, k + 1);
        const idx_t nc = d == 2 ? eidx(I, i + 1, j + 1, k) : na;
        const double draw = FOURTH * (EA(x.DV, I, 1, 0, ep) + EA(x.DV, I, 1, 0, na) + EA(x.DV, I, 1, 0, nb) +
                                      EA(x.DV, I, 1, 0, nc));
        const double div1 = 0.1 * fmin(0.0, draw);
        double div1_b = 0.0;
#pragma unroll
        for (int h = 0; h < NHB; ++h) {
            const int n = hb_comp(h);
            div1_b += fnb[h] * dxd * (CA(x.U1, I, NU1, n, cr) - CA(x.U1, I, NU1, n, cl));
            g[h] = fnb[h] * dxd * div1;
        }
        // a face that two bricks have is counted in the upper one
        if (draw < 0.0 && (l < top || cd == nd)) {
            const double v = 0.1 * FOURTH * div1_b;
            aadd(EAp(a.DVb, I, 1, 0, ep), v);
            aadd(EAp(a.DVb, I, 1, 0, na), v);
            aadd(EAp(a.DVb, I, 1, 0, nb), v);
            aadd(EAp(a.DVb, I, 1, 0, nc), v);
        }
        RiemannHB rb;
        rb.f_rho = fnb[NB_RHO];
        rb.f_mn = pick(d, fnb[NB_MX], fnb[NB_MY], fnb[NB_MZ]);
        rb.f_mt = pick(d, fnb[NB_MY], fnb[NB_MX], fnb[NB_MX]);
        rb.f_mtt = pick(d, fnb[NB_MZ], fnb[NB_MZ], fnb[NB_MY]);
        rb.f_E = fnb[NB_E];
        rb.f_e = fnb[NB_EI];
        rb.g_p = fnb[NB_GP];
        rb.g_un = fnb[NB_GU];
        face_riemann_hb(x, I, d, i, j, k, side_m, side_p, rb, Lb, Rb, cg);
    }
    lr[0][tid] = Lb.rho;
    lr[1][tid] = Lb.un;
    lr[2][tid] = Lb.ut;
    lr[3][tid] = Lb.utt;
    lr[4][tid] = Lb.p;
    lr[5][tid] = Lb.rhoe;
    lr[6][tid] = cg[0];
    lr[7][tid] = cg[2];
#pragma unroll
    for (int h = 0; h < NHB; ++h) lr[8 + h][tid] = g[h];
    __syncthreads();
    // the zone's owner has both its faces (its one face at the domain's ends)
    if (!ok || !(l > 0 || cd < 0) || !(l < top || cd == nd)) return;
    double z2[NZB] = {0, 0, 0, 0, 0, 0, 0, 0, 0}, z3[NZB] = {0, 0, 0, 0, 0, 0, 0, 0, 0}, dummy[UEDEN + 1] = {0, 0, 0, 0, 0};
    double gb[8] = {0, 0, 0, 0, 0, 0, 0, 0}, gamcb = has_p ? cg[3] : 0.0, cb = has_p ? cg[1] : 0.0;
    double f2b[5] = {0, 0, 0, 0, 0}, f3b[5] = {0, 0, 0, 0, 0};
    const idx_t c = cidx(I, i, j, k);
    if (has_p) {
        QInHB o{0, 0, 0, 0, 0, 0};
        trans2_hydro_b(qp, f2r, f2l, f3r, f3l, pg2p, pg2m, ug2p, ug2m, pg3p, pg3m, ug3p, ug3m, gamc, h2, h3,
                       from_faceb(Rb, d), o, f2b, dummy, f3b, dummy, gb, gamcb);
        store_stateb(a.SPb[d], I, ep, o);
    }
    if (has_m) {
        const int ta = tid + st;
        QInHB o{0, 0, 0, 0, 0, 0};
        const FaceHB m{lr[0][ta], lr[1][ta], lr[2][ta], lr[3][ta], lr[4][ta], lr[5][ta]};
        trans2_hydro_b(qm, f2r, f2l, f3r, f3l, pg2p, pg2m, ug2p, ug2m, pg3p, pg3m, ug3p, ug3m, gamc, h2, h3,
                       from_faceb(m, d), o, f2b, dummy, f3b, dummy, gb, gamcb);
        store_stateb(a.SMb[d], I, em, o);
        cb += lr[6][ta];
        gamcb += lr[7][ta];
#pragma unroll
        for (int h = 0; h < NHB; ++h) g[h] -= lr[8 + h][ta];
    }
#pragma unroll
    for (int n = 0; n <= UEDEN; ++n) {
        z2[n] = f2b[n];
        z3[n] = f3b[n];
    }
#pragma unroll
    for (int n = 0; n < 4; ++n) {
        z2[ZB_PGP + n] = gb[n];
        z3[ZB_PGP + n] = gb[4 + n];
    }
    store_zoneb(a.ZF[p2], I, ep, z2);
    store_zoneb(a.ZF[p3], I, ep, z3);
    EF2(a.CG[d], I, 2, 0, ep) = dbl2{cb, gamcb};
#pragma unroll
    for (int h = 0; h < NHB; ++h) aadd(CAp(a.U1b, I, NHB, h, c), g[h]);
}

// ------------------------------------------------------------------ A_trans1
// F^{t|d} of both d: the Riemann problem and trans1, by zones along t as in
// A_final; the fluxes' adjoints are gathered from the zones of the third
// direction's A_final.  64^3: 352 us; by faces with atomic adds 787, with the
// forward values kept across the Riemann problem (spilled) 370.
__global__ __launch_bounds__(256) void A_trans1(Lines q, const FInst *inst, Ctx x, ACtx a)
{
    __shared__ double ls[6][256], lr[8][256];
    int lb = logical_block();
    const int t = lb % 3;
    lb /= 3;
    if (lb >= q.nb[t]) return;  // the whole block
    const FInst &I = inst[0];
    int i, j, k, l;
    const bool ok = line_cell(q, t, lb, I, i, j, k, l);
    const int tid = threadIdx.x, st = t == 0 ? 1 : q.W[t], top = q.L[t] - 1, nt = I.n[t];
    const int ct = t == 0 ? i : (t == 1 ? j : k);
    const int ei = t == 0, ej = t == 1, ek = t == 2;
    const bool has_p = ok && ct >= 0, has_m = ok && ct + 1 <= nt;
    const bool own = ok && (l > 0 || ct < 0) && (l < top || ct == nt);
    const idx_t ep = eidx(I, i, j, k), em = eidx(I, i + ei, j + ej, k + ek);
    // where A_final has been: across t the zones of the domain
    const bool in0 = i >= 0 && i < I.n[0], in1 = j >= 0 && j < I.n[1], in2 = k >= 0 && k < I.n[2];
    const bool fin = (t == 0 || in0) && (t == 1 || in1) && (t == 2 || in2);
    QInHB ob_p{0, 0, 0, 0, 0, 0}, ob_m{0, 0, 0, 0, 0, 0};
    double cb = 0.0, gamcb = 0.0, gamc = 0.0;
    if (ok) gamc = CA(x.Q, I, NFQ, FQ_G, cidx(I, i, j, k));
    if (own && fin) {
        if (has_p) load_stateb(a.SPb[t], I, ep, ob_p);
        if (has_m) load_stateb(a.SMb[t], I, em, ob_m);
        const dbl2 v = EF2(a.CG[t], I, 2, 0, ep);
        cb = v.x;
        gamcb = v.y;
    }
    for (int s = 0; s < 2; ++s) {
        const int d = t == 0 ? 1 + s : (t == 1 ? 2 * s : s);
        const bool act = ok && (d == 0 ? in0 : (d == 1 ? in1 : in2));
        const int combo = pair_index(t, d);
        const double cdtdx = x.dt_cur[0] / I.dx[d];
        const double cdt = cdtdx / 3.0;
        double fr[UEDEN + 1], fl[UEDEN + 1], pgp, ugp, pgm, ugm;
        const idx_t dr = eidx(I, i + (d == 0), j + (d == 1), k + (d == 2)) - ep;
        FaceH side_p{};
        idx_t er = ep;
        behind(er, ob_m);
        if (act) {
            load_tflux_h(x.FD[d], I, er + dr, fr, pgp, ugp);
            load_tflux_h(x.FD[d], I, er, fl, pgm, ugm);
            if (has_m) {
                QInH qm;
                load_qin_h(x.SM[t], I, er + (em - ep), qm);
                const FaceH f = to_face(trans1_hydro(qm, fr, fl, pgp, pgm, ugp, ugm, gamc, cdt), t);
                ls[0][tid] = f.rho;
                ls[1][tid] = f.un;
                ls[2][tid] = f.ut;
                ls[3][tid] = f.utt;
                ls[4][tid] = f.p;
                ls[5][tid] = f.rhoe;
            }
            if (has_p) {
                QInH qp;
                load_qin_h(x.SP[t], I, er, qp);
                side_p = to_face(trans1_hydro(qp, fr, fl, pgp, pgm, ugp, ugm, gamc, cdt), t);
            }
        }
        __syncthreads();
        FaceHB Lb{}, Rb{};
        double cg[4] = {0.0, 0.0, 0.0, 0.0};
        if (act && has_p && l > 0) {
            const int tb = tid - st;
            const FaceH side_m{ls[0][tb], ls[1][tb], ls[2][tb], ls[3][tb], ls[4][tb], ls[5][tb]};
            FluxB v{};
            gather_zoneb(a.ZF[combo], I, eidx(I, i - ei, j - ej, k - ek), ep, ct > 0, ct < nt, v);
            face_riemann_hb(x, I, t, i, j, k, side_m, side_p, riemannb_of(v, t), Lb, Rb, cg);
        }
        lr[0][tid] = Lb.rho;
        lr[1][tid] = Lb.un;
        lr[2][tid] = Lb.ut;
        lr[3][tid] = Lb.utt;
        lr[4][tid] = Lb.p;
        lr[5][tid] = Lb.rhoe;
        lr[6][tid] = cg[0];
        lr[7][tid] = cg[2];
        __syncthreads();
        if (!(act && own)) continue;
        er = ep;
        behind(er, Rb);
        load_tflux_h(x.FD[d], I, er + dr, fr, pgp, ugp);
        load_tflux_h(x.FD[d], I, er, fl, pgm, ugm);
        double frb[5] = {0, 0, 0, 0, 0}, dummy[UEDEN + 1] = {0, 0, 0, 0, 0}, z[NZB] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
        if (has_p) {
            QInH qp;
            load_qin_h(x.SP[t], I, er, qp);
            cb += cg[1];
            gamcb += cg[3];
            trans1_hydro_b(qp, fr, fl, pgp, pgm, ugp, ugm, gamc, cdt, from_faceb(Rb, t), ob_p, frb, dummy, z[ZB_PGP],
                           z[ZB_PGM], z[ZB_UGP], z[ZB_UGM], gamcb);
        }
        if (has_m) {
            const int ta = tid + st;
            const FaceHB m{lr[0][ta], lr[1][ta], lr[2][ta], lr[3][ta], lr[4][ta], lr[5][ta]};
            QInH qm;
            load_qin_h(x.SM[t], I, er + (em - ep), qm);
            cb += lr[6][ta];
            gamcb += lr[7][ta];
            trans1_hydro_b(qm, fr, fl, pgp, pgm, ugp, ugm, gamc, cdt, from_faceb(m, t), ob_m, frb, dummy, z[ZB_PGP],
                           z[ZB_PGM], z[ZB_UGP], z[ZB_UGM], gamcb);
        }
#pragma unroll
        for (int n = 0; n <= UEDEN; ++n) z[n] = frb[n];
        store_zoneb(a.ZT[combo], I, ep, z);
    }
    if (!own) return;
    if (has_p) store_stateb(a.SPb[t], I, ep, ob_p);
    if (has_m) store_stateb(a.SMb[t], I, em, ob_m);
    EF2(a.CG[t], I, 2, 0, ep) = dbl2{cb, gamcb};
}

// ------------------------------------------------------------------ A_flux1
__global__ __launch_bounds__(256) void A_flux1(Plan p, Ctx x, ACtx a)
{
    int m, i, j, k;
    int sub_;
    if (!plan_cell_sub(p, 3, sub_, m, i, j, k)) return;
    const int d = sub_;
    const FInst &I = p.inst[m];
    const int pos = d == 0 ? i : (d == 1 ? j : k);
    if (pos < 0) return;
    const idx_t e = eidx(I, i, j, k), el = eidx(I, i - (d == 0), j - (d == 1), k - (d == 2));
    FaceH L, R;
    load_fs_h(x.SM[d], I, e, d, L);
    load_fs_h(x.SP[d], I, e, d, R);
    FluxB v{};
    double cg[4];
    for (int s = 0; s < 2; ++s)  // the two pairs (t, d)
        gather_zoneb(a.ZT[2 * d + s], I, el, e, pos > 0, pos < I.n[d], v);
    FaceHB Lb, Rb;
    face_riemann_hb(x, I, d, i, j, k, L, R, riemannb_of(v, d), Lb, Rb, cg);
    add_faceb(a.SMb[d], I, e, d, Lb);
    add_faceb(a.SPb[d], I, e, d, Rb);
    EF2(a.CGF[d], I, 4, 0, e) = dbl2{cg[0], cg[2]};
    EF2(a.CGF[d], I, 4, 2, e) = dbl2{cg[1], cg[3]};
}

// ------------------------------------------------------------------ A_trace
// The thread of a zone reverses one direction's traces.  What it owes the five
// zones of its stencil is summed along the brick through LDS, a variable at a
// time, and stored; what leaves the brick or the range, or belongs to a zone
// of the ring, is added by itself to the mapped zone.  64^3: 338 us against
// 432 with 38 atomic adds a zone and direction; what is left is arithmetic at
// two waves a SIMD (VALUs 42% busy; three waves spill and gain nothing).
__global__ __launch_bounds__(256) void A_trace(Lines q, const FInst *inst, Ctx x, ACtx a)
{
    __shared__ double ls[2][5][256];
    int lb = logical_block();
    const int d = lb % 3;
    lb /= 3;
    if (lb >= q.nb[d]) return;  // the whole block
    const FInst &I = inst[0];
    int i, j, k, l;
    const bool ok = line_cell(q, d, lb, I, i, j, k, l);
    i = min(i, I.n[0]);  // threads without a zone read the last one
    j = min(j, I.n[1]);
    k = min(k, I.n[2]);
    const int tid = threadIdx.x, st = d == 0 ? 1 : q.W[d], top = q.L[d] - 1, nd = I.n[d];
    const int di = (d == 0), dj = (d == 1), dk = (d == 2);
    const int pos = d == 0 ? i : (d == 1 ? j : k);
    const bool do_p = pos >= 0;
    const bool do_m = pos <= nd - 1;
    const int cun = FQ_U + d, cut = d == 0 ? FQ_V : (d == 1 ? FQ_W : FQ_U), cutt = d == 0 ? FQ_W : (d == 1 ? FQ_U : FQ_V);
    const idx_t c0 = cidx(I, i, j, k);
    const double cc = CA(x.Q, I, NFQ, FQ_C, c0);
    const double un = CA(x.Q, I, NFQ, cun, c0);
    const idx_t ec = eidx(I, i, j, k);
    const double flatn = EA(x.FL, I, 1, 0, ec);
    const double dtdx = x.dt_cur[0] / I.dx[d];
    idx_t cs[5];
#pragma unroll
    for (int s = -2; s <= 2; ++s) cs[s + 2] = cidx(I, i + s * di, j + s * dj, k + s * dk);
    const int vars[7] = {FQ_RHO, cun, FQ_P, FQ_RE, cut, cutt, FQ_G};
    const int qbv[7] = {QB_RHO, QB_U + d, QB_P, QB_RE, QB_U + (cut - FQ_U), QB_U + (cutt - FQ_U), QB_G};
    // Forward: the PPM integrals the projection reads.  Edge values are not
    // kept; the reverse sweep reads each stencil again (L2 hits) and rebuilds
    // them, which keeps the kernel within one register file per wave.
    const double spd[3] = {un - cc, un, un + cc};
    double Ip[3][4], Im[3][4];
    double gam_m, gam_p;
#pragma unroll
    for (int vv = 0; vv < 7; ++vv) {
        if (vv == 4 || vv == 5) continue;
        double s5[5], sm, sp;
#pragma unroll
        for (int q = 0; q < 5; ++q) s5[q] = CA(x.Q, I, NFQ, vars[vv], cs[q]);
        ppm_reconstruct(s5, flatn, sm, sp);
        const double s6 = ppm_s6(sm, sp, s5[2]);
        if (vv < 4) {
#pragma unroll
            for (int w = 0; w < 3; ++w) ppm_int_wave(sm, sp, s6, spd[w], dtdx, Ip[w][vv], Im[w][vv]);
        } else {
            double dummy;
            ppm_int_wave(sm, sp, s6, un - cc, dtdx, dummy, gam_m);
            ppm_int_wave(sm, sp, s6, un + cc, dtdx, gam_p, dummy);
        }
    }

    const idx_t ep = ec, em = eidx(I, i + di, j + dj, k + dk);
    double Ipb[3][4] = {{0}}, Imb[3][4] = {{0}};
    double gam_mb = 0.0, gam_pb = 0.0, Ip_utb = 0.0, Im_utb = 0.0, Ip_uttb = 0.0, Im_uttb = 0.0;
    if (do_p) {
        QInHB v;
        load_stateb(a.SPb[d], I, ep, v);
        ppm_project_b<true>(Im, gam_m, un, cc, v.rho, pick(d, v.u, v.v, v.w), v.rhoe, v.p, Imb, gam_mb);
        Im_utb = pick(d, v.v, v.w, v.u);
        Im_uttb = pick(d, v.w, v.u, v.v);
    }
    if (do_m) {
        QInHB v;
        load_stateb(a.SMb[d], I, em, v);
        ppm_project_b<false>(Ip, gam_p, un, cc, v.rho, pick(d, v.u, v.v, v.w), v.rhoe, v.p, Ipb, gam_pb);
        Ip_utb = pick(d, v.v, v.w, v.u);
        Ip_uttb = pick(d, v.w, v.u, v.v);
    }
    double unb = 0.0, flatb = 0.0;
    // c and Gamma_1: from the states' corrections and the faces' Riemann problems
    const dbl2 cgz = EF2(a.CG[d], I, 2, 0, ec);
    double ccb = cgz.x, gcb = cgz.y;
    if (do_p) {
        const dbl2 v = EF2(a.CGF[d], I, 4, 2, ep);
        ccb += v.x;
        gcb += v.y;
    }
    if (do_m) {
        const dbl2 v = EF2(a.CGF[d], I, 4, 0, em);
        ccb += v.x;
        gcb += v.y;
    }
    const bool inside = i >= 0 && i < I.n[0] && j >= 0 && j < I.n[1] && k >= 0 && k < I.n[2];
    // which zones of the stencil the brick has
    const bool b1 = l >= 1, b2 = l >= 2, a1 = l < top && pos < nd, a2 = l + 1 < top && pos + 1 < nd;
#pragma unroll
    for (int z = 0; z < 7; ++z) {
        constexpr int order[7] = {0, 2, 3, 4, 5, 6, 1};  // the normal velocity last: unb goes to it
        const int vv = order[z];
        double s5[5], SMv, SPv;
#pragma unroll
        for (int q = 0; q < 5; ++q) s5[q] = CA(x.Q, I, NFQ, vars[vv], cs[q]);
        ppm_reconstruct(s5, flatn, SMv, SPv);
        const double S6 = ppm_s6(SMv, SPv, s5[2]);
        double smb = 0.0, spb = 0.0, s6b = 0.0;
        if (vv < 4) {
#pragma unroll
            for (int w = 0; w < 3; ++w) {
                double spdb = 0.0;
                ppm_int_wave_b(SMv, SPv, S6, spd[w], dtdx, Ipb[w][vv], Imb[w][vv], smb, spb, s6b, spdb);
                unb += spdb;
                if (w == 0) ccb -= spdb;
                if (w == 2) ccb += spdb;
            }
        } else if (vv < 6) {
            double spdb = 0.0;
            ppm_int_wave_b(SMv, SPv, S6, un, dtdx, vv == 4 ? Ip_utb : Ip_uttb, vv == 4 ? Im_utb : Im_uttb,
                           smb, spb, s6b, spdb);
            unb += spdb;
        } else {
            double spdb = 0.0;
            ppm_int_wave_b(SMv, SPv, S6, un - cc, dtdx, 0.0, gam_mb, smb, spb, s6b, spdb);
            unb += spdb;
            ccb -= spdb;
            spdb = 0.0;
            ppm_int_wave_b(SMv, SPv, S6, un + cc, dtdx, gam_pb, 0.0, smb, spb, s6b, spdb);
            unb += spdb;
            ccb += spdb;
        }
        // s6 = 6 s0 - 3 (sm + sp)
        double s5b[5] = {0, 0, 0, 0, 0};
        s5b[2] += 6.0 * s6b;
        smb -= 3.0 * s6b;
        spb -= 3.0 * s6b;
        ppm_reconstruct_b(s5, flatn, smb, spb, s5b, flatb);
        if (vv == 1) s5b[2] += unb;
        if (vv == 6) s5b[2] += gcb;
        double(*S)[256] = ls[z & 1];
#pragma unroll
        for (int q = 0; q < 5; ++q) S[q][tid] = ok ? s5b[q] : 0.0;
        __syncthreads();
        if (ok) {
            double sum = s5b[2];
            if (b2) sum += S[4][tid - 2 * st];
            if (b1) sum += S[3][tid - st];
            if (a1) sum += S[1][tid + st];
            if (a2) sum += S[0][tid + 2 * st];
            if (inside) CA(a.QD[d], I, NQB, qbv[vv], c0) = sum;
            else aadd(CAp(a.Qb, I, NQB, qbv[vv], c0), sum);
            if (!b2) aadd(CAp(a.Qb, I, NQB, qbv[vv], cs[0]), s5b[0]);
            if (!b1) aadd(CAp(a.Qb, I, NQB, qbv[vv], cs[1]), s5b[1]);
            if (!a1) aadd(CAp(a.Qb, I, NQB, qbv[vv], cs[3]), s5b[3]);
            if (!a2) aadd(CAp(a.Qb, I, NQB, qbv[vv], cs[4]), s5b[4]);
        }
    }
    if (!ok) return;
    if (inside) CA(a.QD[d], I, NQB, QB_C, c0) = ccb;
    else aadd(CAp(a.Qb, I, NQB, QB_C, c0), ccb);
    EA(a.FLb[d], I, 1, 0, ec) = flatb;
}

// ------------------------------------------------------------------ A_flat
__global__ __launch_bounds__(256) void A_flat(Plan p, Ctx x, ACtx a)
{
    int m, i, j, k;
    if (!plan_cell(p, m, i, j, k)) return;
    const FInst &I = p.inst[m];
    const idx_t e = eidx(I, i, j, k);
    const double fb = EA(a.FLb[0], I, 1, 0, e) + EA(a.FLb[1], I, 1, 0, e) + EA(a.FLb[2], I, 1, 0, e);
    if (fb != 0.0) {
        double cur = 1.0;
        int arg = -1;
        for (int d = 0; d < 3; ++d) {
            const int ei = (d == 0), ej = (d == 1), ek = (d == 2);
            double p7[7], u7[7];
#pragma unroll
            for (int s = -3; s <= 3; ++s) {
                const idx_t c = cidx(I, i + s * ei, j + s * ej, k + s * ek);
                p7[s + 3] = CA(x.Q, I, NFQ, FQ_P, c);
                u7[s + 3] = CA(x.Q, I, NFQ, FQ_U + d, c);
            }
            const double f = flatten_dir(p7, u7);
            if (f < cur) {
                cur = f;
                arg = d;
            }
        }
        if (arg >= 0) {
            const int ei = (arg == 0), ej = (arg == 1), ek = (arg == 2);
            double p7[7], u7[7], p7b[7] = {0, 0, 0, 0, 0, 0, 0};
            idx_t cc[7];
#pragma unroll
            for (int s = -3; s <= 3; ++s) {
                cc[s + 3] = cidx(I, i + s * ei, j + s * ej, k + s * ek);
                p7[s + 3] = CA(x.Q, I, NFQ, FQ_P, cc[s + 3]);
                u7[s + 3] = CA_lane(x.Q, I, NFQ, FQ_U + arg, cc[s + 3]);  // arg differs per lane
            }
            flatten_dir_b(p7, u7, fb, p7b);
#pragma unroll
            for (int s = 0; s < 7; ++s) aadd(CAp(a.Qb, I, NQB, QB_P, cc[s]), p7b[s]);
        }
    }
    // div(u): the velocities of zone (i,j,k) from its eight nodes, 0..n
    double n8[2][2][2];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        const int ni = i + (q & 1), nj = j + ((q >> 1) & 1), nk = k + (q >> 2);
        n8[q >> 2][(q >> 1) & 1][q & 1] =
            ni <= I.n[0] && nj <= I.n[1] && nk <= I.n[2] ? EA(a.DVb, I, 1, 0, eidx(I, ni, nj, nk)) : 0.0;
    }
    const double du = FOURTH / I.dx[0] * ((n8[0][0][0] - n8[0][0][1]) + (n8[0][1][0] - n8[0][1][1]) +
                                          (n8[1][0][0] - n8[1][0][1]) + (n8[1][1][0] - n8[1][1][1]));
    const double dv = FOURTH / I.dx[1] * ((n8[0][0][0] - n8[0][1][0]) + (n8[0][0][1] - n8[0][1][1]) +
                                          (n8[1][0][0] - n8[1][1][0]) + (n8[1][0][1] - n8[1][1][1]));
    const double dw = FOURTH / I.dx[2] * ((n8[0][0][0] - n8[1][0][0]) + (n8[0][0][1] - n8[1][0][1]) +
                                          (n8[0][1][0] - n8[1][1][0]) + (n8[0][1][1] - n8[1][1][1]));
    const idx_t c0 = cidx(I, i, j, k);
    if (i >= 0 && i < I.n[0] && j >= 0 && j < I.n[1] && k >= 0 && k < I.n[2]) {
        CA(a.QD[0], I, NQB, QB_U, c0) += du;
        CA(a.QD[0], I, NQB, QB_V, c0) += dv;
        CA(a.QD[0], I, NQB, QB_W, c0) += dw;
    } else {
        aadd(CAp(a.Qb, I, NQB, QB_U, c0), du);
        aadd(CAp(a.Qb, I, NQB, QB_V, c0), dv);
        aadd(CAp(a.Qb, I, NQB, QB_W, c0), dw);
    }
}

// ------------------------------------------------------------------ A_prim
__global__ __launch_bounds__(256) void A_prim(Plan p, Ctx x, ACtx a)
{
    int m, i, j, k;
    if (!plan_cell(p, m, i, j, k)) return;
    const FInst &I = p.inst[m];
    idx_t c = cidx(I, i, j, k);
    double u1[NVAR], qb[NQB], ub[NHB];
#pragma unroll
    for (int n = 0; n < NU1; ++n) u1[n] = CA(x.U1, I, NU1, n, c);  // clean(clean(U)) of the forward
    const SpeciesPairs XU = cell_species(x.U1X, I);
#pragma unroll
    for (int pr = 0; pr < NSPEC_PAIRS; ++pr) {
        const dbl2 v = SP2(XU, pr, c);
        u1[UFS + 2 * pr] = v.x;
        if (2 * pr + 1 < NSPEC) u1[UFS + 2 * pr + 1] = v.y;
    }
#pragma unroll
    for (int q = 0; q < NQB; ++q)
        qb[q] = CA(a.Qb, I, NQB, q, c) + CA(a.QD[0], I, NQB, q, c) + CA(a.QD[1], I, NQB, q, c) +
                CA(a.QD[2], I, NQB, q, c);
#pragma unroll
    for (int h = 0; h < NHB; ++h) ub[h] = CA(a.U1b, I, NHB, h, c);
    ctoprim_b(u1, x.tab, qb, ub);
    // the old state is read behind these results (the compiler would start
    // everything at once and spill)
#pragma unroll
    for (int h = 0; h < NHB; ++h) asm volatile("" : "+v"(c), "+v"(ub[h]));
    double u0[NVAR], ua[NVAR];
#pragma unroll
    for (int n = 0; n < NVAR; ++n) ua[n] = u0[n] = a.Uold[(long)NVAR * I.offD + (long)n * I.nD + c];
    clean_hydro(ua, x.tab);
    clean_cell_b(ua, x.tab, ub);
    clean_cell_b(u0, x.tab, ub);
#pragma unroll
    for (int h = 0; h < NHB; ++h) CA(a.Ubo, I, NHB, h, c) += ub[h];
}

// seed: hydro components of a full NVAR adjoint (cell layout)
__global__ void A_seed(const double *src, double *Ub, long nD)
{
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nD) return;
#pragma unroll
    for (int h = 0; h < NHB; ++h) Ub[(long)h * nD + t] = src[(long)hb_comp(h) * nD + t];
}

__global__ void A_unseed(const double *Ub, double *dst, long nD)
{
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nD) return;
#pragma unroll
    for (int n = 0; n < NVAR; ++n) dst[(long)n * nD + t] = 0.0;
#pragma unroll
    for (int h = 0; h < NHB; ++h) dst[(long)hb_comp(h) * nD + t] = Ub[(long)h * nD + t];
}

} // namespace mc

using namespace mc;

struct mc_adjoint {
    FusedLevel *F = nullptr;
    int n[3];
    long nD = 0, nE = 0;
    int max_steps = 0;
    int nsteps = 0;
    double *ckpt = nullptr;       // max_steps x NVAR x nD
    std::vector<double> dts;
    double *abuf = nullptr;       // adjoint intermediates
    long abuf_n = 0;              // of them from the start, cleared every step
    Lines lines_final, lines_trans1, lines_trace;
    double *ub0 = nullptr, *ub1 = nullptr;  // NHB x nD each
    ACtx a;
    // Kept intermediates: step n of the forward pass writes its primitives,
    // traces and fluxes into sets[n], and the reverse pass reads them there
    // instead of recomputing the step.  Empty: recompute mode.
    std::vector<FusedArrays> sets;
    FusedArrays own;  // the engine's own set
};

static void adjoint_drop_sets(mc_adjoint *A)
{
    fused_set_intermediates(A->F, A->own);
    for (auto &S : A->sets) fused_free_intermediates(S);
    A->sets.clear();
    A->nsteps = 0;  // a kept forward pass is gone
}

// One set per step when max_steps sets fit in half of the free device memory.
static int adjoint_keep_sets(mc_adjoint *A, bool report)
{
    if (!A->sets.empty()) return 0;
    size_t free_b = 0, total_b = 0;
    if (check_hip(hipMemGetInfo(&free_b, &total_b), "hipMemGetInfo")) return -1;
    const size_t need = fused_intermediate_bytes(A->F) * (size_t)A->max_steps;
    if (need > free_b / 2) {
        if (report) set_error("mc_adjoint: the intermediates of max_steps steps do not fit in half the free device memory");
        return -1;
    }
    A->sets.resize(A->max_steps);
    for (auto &S : A->sets)
        if (fused_alloc_intermediates(A->F, S)) {
            adjoint_drop_sets(A);
            return -1;
        }
    A->nsteps = 0;
    return 0;
}

// Bricks of 256 threads along each direction: the length that wastes least
// (threads without a zone, zones that two bricks share; 64^3: 16 along, A_trans1
// 354 us against 414 with 8 and 381 with 32).
static Lines make_lines(const int *n, int ring, int ovl)
{
    Lines q;
    q.ring = ring;
    q.ovl = ovl;
    auto up = [](int a, int b) { return (a + b - 1) / b; };
    for (int d = 0; d < 3; ++d) {
        const int c0 = n[0] + 2 * ring, c1 = n[1] + 2 * ring, c2 = n[2] + 2 * ring;  // zones across
        long best = -1;
        for (int L = 64; L >= 8; L /= 2) {
            const int W = 256 / L, along = ovl ? up(n[d], L - ovl) : up(n[d] + 2, L);
            const int nb0 = d == 0 ? along : up(c0, W);
            const int nb1 = d == 1 ? along : (d == 0 ? up(c1, W) : c1);
            const long nb = (long)nb0 * nb1 * (d == 2 ? along : c2);
            if (best < 0 || nb < best) {
                best = nb;
                q.L[d] = L;
                q.W[d] = W;
                q.nb0[d] = nb0;
                q.nb1[d] = nb1;
                q.nb[d] = (int)nb;
            }
        }
    }
    return q;
}

static void launch_adj(mc_adjoint *A, int stage, hipStream_t s)
{
    FusedLevel *F = A->F;
    if (stage == FST_FINAL || stage == FST_TRANS1 || stage == FST_TRACE) {
        const Lines &q = stage == FST_FINAL ? A->lines_final : (stage == FST_TRANS1 ? A->lines_trans1 : A->lines_trace);
        const dim3 g(3 * std::max(q.nb[0], std::max(q.nb[1], q.nb[2]))), b(256);
        if (stage == FST_FINAL) hipLaunchKernelGGL(A_final, g, b, 0, s, q, F->inst, F->ctx, A->a);
        else if (stage == FST_TRANS1) hipLaunchKernelGGL(A_trans1, g, b, 0, s, q, F->inst, F->ctx, A->a);
        else hipLaunchKernelGGL(A_trace, g, b, 0, s, q, F->inst, F->ctx, A->a);
        return;
    }
    Plan p = get_plan(F, stage);
    const int nb = plan_blocks(F, p);
    const int nt = p.bx * p.by * p.bz;
    if (nb <= 0) return;
    // face stage: directions interleaved brick by brick, as forward
    const dim3 g(stage == FST_FLUX1 ? 3 * nb : nb), b(nt);
    F->ctx.tab = eos_table();
    switch (stage) {
    case FST_PRIM: hipLaunchKernelGGL(A_prim, g, b, 0, s, p, F->ctx, A->a); break;
    case FST_FLAT: hipLaunchKernelGGL(A_flat, g, b, 0, s, p, F->ctx, A->a); break;
    case FST_FLUX1: hipLaunchKernelGGL(A_flux1, g, b, 0, s, p, F->ctx, A->a); break;
    case FST_UPDATE: hipLaunchKernelGGL(A_update, g, b, 0, s, p, F->ctx, A->a); break;
    }
}

extern "C" {

void mc_adjoint_destroy(mc_adjoint_t *A);

mc_adjoint_t *mc_adjoint_create(const int *n_cell, const double *prob_lo, const double *prob_hi, int bc, int max_steps)
{
    if (!n_cell || !prob_lo || !prob_hi || max_steps < 1 || (bc != 0 && bc != 1)) {
        set_error("mc_adjoint_create: bad arguments");
        return nullptr;
    }
    for (int d = 0; d < 3; ++d)
        if (n_cell[d] < 4 || !(prob_hi[d] > prob_lo[d])) {
            set_error("mc_adjoint_create: bad domain");
            return nullptr;
        }
    mc_adjoint *A = new mc_adjoint();
    FusedInstanceSpec sp;
    for (int d = 0; d < 3; ++d) {
        sp.n[d] = n_cell[d];
        sp.dx[d] = (prob_hi[d] - prob_lo[d]) / n_cell[d];
        A->n[d] = n_cell[d];
    }
    sp.bc = bc;
    A->F = fused_create_set(std::vector<FusedInstanceSpec>{sp});
    if (!A->F) {
        delete A;
        return nullptr;
    }
    fused_set_keep_transverse(A->F, true);  // the reverse kernels read them
    A->nD = (long)n_cell[0] * n_cell[1] * n_cell[2];
    A->nE = fused_next(A->F, 0);  // the reverse kernels index with the engine's stride
    A->max_steps = max_steps;
    // intermediates: U1b, Qb (cells) and DVb, cleared every step; SMb, SPb,
    // CG, ZF, ZT.  Sb lies in ZT, which is written after A_final has read it;
    // CGF, FLb and QD in ZF, which A_trans1 is the last to read.
    const long nD = A->nD, nE = A->nE;
    A->abuf_n = (long)(NHB + NQB) * nD + nE;
    const long rest = (3 * (2 * NSB + 2) + 12 * NZB) * nE;
    bool ok = !check_hip(hipMalloc(&A->ckpt, sizeof(double) * NVAR * nD * (size_t)max_steps), "hipMalloc(ckpt)") &&
              !check_hip(hipMalloc(&A->abuf, sizeof(double) * (A->abuf_n + rest)), "hipMalloc(adjoint)") &&
              !check_hip(hipMalloc(&A->ub0, sizeof(double) * NHB * nD), "hipMalloc(adjoint)") &&
              !check_hip(hipMalloc(&A->ub1, sizeof(double) * NHB * nD), "hipMalloc(adjoint)");
    if (!ok) {
        mc_adjoint_destroy(A);
        return nullptr;
    }
    A->own = fused_get_intermediates(A->F);
    (void)adjoint_keep_sets(A, false);  // else recompute mode
    double *q = A->abuf;
    ACtx &a = A->a;
    a.U1b = q;
    q += NHB * nD;
    a.Qb = q;
    q += NQB * nD;
    a.DVb = q;
    q += nE;
    auto take = [&](double *&p, long n) {
        p = q;
        q += n;
    };
    for (int d = 0; d < 3; ++d) {
        take(a.SMb[d], NSB * nE);
        take(a.SPb[d], NSB * nE);
        take(a.CG[d], 2 * nE);
    }
    for (int c = 0; c < 6; ++c) take(a.ZF[c], NZB * nE);
    for (int c = 0; c < 6; ++c) take(a.ZT[c], NZB * nE);
    a.Sb = a.ZT[0];
    q = a.ZF[0];
    for (int d = 0; d < 3; ++d) {
        take(a.CGF[d], 4 * nE);
        take(a.FLb[d], nE);
        take(a.QD[d], NQB * nD);
    }
    A->lines_final = make_lines(A->n, 0, 2);
    A->lines_trans1 = make_lines(A->n, 1, 2);
    A->lines_trace = make_lines(A->n, 1, 0);
    return A;
}

void mc_adjoint_destroy(mc_adjoint_t *A)
{
    if (!A) return;
    if (A->F) {
        (void)hipDeviceSynchronize();
        adjoint_drop_sets(A);
        fused_destroy(A->F);
    }
    (void)hipFree(A->ckpt);
    (void)hipFree(A->abuf);
    (void)hipFree(A->ub0);
    (void)hipFree(A->ub1);
    delete A;
}

// Forward pass: U0 (device, NVAR x cells, Fortran order) advanced nsteps
// with checkpoints; the final state goes to U_out (device).  compute_dt != 0:
// dts[n] receive the CFL-limited sequence dt_0 = cfl * estdt(U0),
// dt_{n+1} = min(cfl * estdt(U_{n+1}), 1.1 dt_n); otherwise dts are used.
int mc_adjoint_forward(mc_adjoint_t *A, const double *U0, double *U_out, int nsteps, double *dts, int compute_dt)
{
    if (!A || !U0 || !U_out || !dts || nsteps < 1 || nsteps > A->max_steps) {
        set_error("mc_adjoint_forward: bad arguments");
        return -1;
    }
    if (!eos_ready()) {
        set_error("mc_adjoint_forward: EOS table not loaded");
        return -1;
    }
    hipStream_t s = cur_stream();
    FusedLevel *F = A->F;
    const size_t bytes = sizeof(double) * NVAR * A->nD;
    double *U = fused_state(F, 0);
    if (check_hip(hipMemcpyAsync(U, U0, bytes, hipMemcpyDeviceToDevice, s), "adjoint forward")) return -1;
    A->dts.assign(nsteps, 0.0);
    double est = 0.0;
    if (compute_dt) {
        if (fused_estimate(F, s) || fused_read_est(F, 0, &est, s)) return -1;
    }
    for (int n = 0; n < nsteps; ++n) {
        double dt;
        if (compute_dt) {
            dt = n == 0 ? cfl * est : fmin(cfl * est, 1.1 * A->dts[n - 1]);
            dts[n] = dt;
        } else dt = dts[n];
        A->dts[n] = dt;
        if (check_hip(hipMemcpyAsync(A->ckpt + (size_t)n * NVAR * A->nD, U, bytes, hipMemcpyDeviceToDevice, s),
                      "checkpoint"))
            return -1;
        if (!A->sets.empty()) fused_set_intermediates(F, A->sets[n]);
        if (fused_advance_dt(F, dt, s)) return -1;
        if (compute_dt && fused_read_est(F, 0, &est, s)) return -1;
    }
    if (!A->sets.empty()) fused_set_intermediates(F, A->own);
    A->nsteps = nsteps;
    if (check_hip(hipMemcpyAsync(U_out, U, bytes, hipMemcpyDeviceToDevice, s), "adjoint forward")) return -1;
    return check_hip(hipStreamSynchronize(s), "adjoint forward");
}

// Reverse pass of the last forward pass: Ub_final (device, NVAR x cells) is
// the adjoint of its final state; Ub0 (device, NVAR x cells) receives the
// adjoint of its initial state (hydro components; UTEMP and species zero).
int mc_adjoint_backward(mc_adjoint_t *A, const double *Ub_final, double *Ub0)
{
    if (!A || !Ub_final || !Ub0 || A->nsteps < 1) {
        set_error("mc_adjoint_backward: bad arguments or no forward pass");
        return -1;
    }
    if (!eos_ready()) {
        set_error("mc_adjoint_backward: EOS table not loaded");
        return -1;
    }
    hipStream_t s = cur_stream();
    FusedLevel *F = A->F;
    const long nD = A->nD;
    const size_t bytes = sizeof(double) * NVAR * nD;
    const unsigned gb = (unsigned)((nD + 255) / 256);
    hipLaunchKernelGGL(A_seed, dim3(gb), dim3(256), 0, s, Ub_final, A->ub0, nD);
    double *cur = A->ub0, *nxt = A->ub1;
    double *U = fused_state(F, 0);
    for (int n = A->nsteps - 1; n >= 0; --n) {
        const double *ck = A->ckpt + (size_t)n * NVAR * nD;
        if (!A->sets.empty()) {
            // the step's intermediates as the forward pass left them
            fused_set_intermediates(F, A->sets[n]);
            fill(F->ctx.dt_cur, 1, A->dts[n], s);
        } else {
            if (check_hip(hipMemcpyAsync(U, ck, bytes, hipMemcpyDeviceToDevice, s), "recompute")) return -1;
            if (fused_recompute_dt(F, A->dts[n], s)) return -1;  // recompute the step's intermediates
        }
        fill(A->abuf, A->abuf_n, 0.0, s);
        A->a.Uold = ck;
        A->a.Ub = cur;
        A->a.Ubo = nxt;
        launch_adj(A, FST_UPDATE, s);
        launch_adj(A, FST_FINAL, s);
        launch_adj(A, FST_TRANS1, s);
        launch_adj(A, FST_FLUX1, s);
        launch_adj(A, FST_TRACE, s);
        launch_adj(A, FST_FLAT, s);
        launch_adj(A, FST_PRIM, s);
        if (check_hip(hipGetLastError(), "adjoint step")) return -1;
        std::swap(cur, nxt);
    }
    if (!A->sets.empty()) fused_set_intermediates(F, A->own);
    hipLaunchKernelGGL(A_unseed, dim3(gb), dim3(256), 0, s, cur, Ub0, nD);
    return check_hip(hipStreamSynchronize(s), "adjoint backward");
}

// keep != 0: keep every step's intermediates (allocated now; fails if
// max_steps sets do not fit in half the free device memory); 0: recompute
// each step from its checkpoint.  Either change drops the last forward pass.
int mc_adjoint_keep_intermediates(mc_adjoint_t *A, int keep)
{
    if (!A) {
        set_error("mc_adjoint_keep_intermediates: null handle");
        return -1;
    }
    (void)hipDeviceSynchronize();
    if (!keep) {
        adjoint_drop_sets(A);
        return 0;
    }
    return adjoint_keep_sets(A, true);
}

int mc_adjoint_keeps_intermediates(const mc_adjoint_t *A) { return A && !A->sets.empty() ? 1 : 0; }

int mc_adjoint_steps(const mc_adjoint_t *A) { return A ? A->nsteps : -1; }

} // extern "C"
