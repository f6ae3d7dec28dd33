// The species stage of the fused step: the thirteen passive species through
// trace, first-stage flux, transverse corrections and final flux in one
// launch, nothing but their final fluxes leaving the chip.
//
// Species ride on a flow the hydro stages have already solved: of a face they
// need its mass flux and Riemann weight (FF_RHO / FF_W, FN_FR / FN_W), of a
// state its density (Ctx::RW).  Streaming their states and fluxes through
// memory stage by stage, in the hydro stages, moved two thirds of a step's
// bytes: at 256^3 the traces and first fluxes took 10.4 ms, the transverse
// stage 14.2, the final one 12.3.  Here a block owns a tile of columns and
// marches in z, so a species is read once (and its tile's halo) and three
// fluxes are written: 9.4 ms and 26 GB for all thirteen, the hydro stages alone
// 4.3, 5.0 and 4.6 ms.
//
// What bounds it: FP64 issue.  A wavefront issues about 1,200 vector
// instructions a plane for its 64 columns and two species, 60% of the rate
// its two wavefronts per SIMD could reach; the rest is waiting at the five
// barriers.  Before, in turn: the flow's data read from 16-byte strided
// arrays, every neighbour and both planes from memory (13.4 ms, the vector L1
// busy throughout); one species a block, three wavefronts per SIMD (18.7 ms,
// the same L1 limit); branches in the limiter (14.3 ms).
#pragma once

#include "mc_fused_impl.h"

namespace mc {

// Launch plan: per instance ntx * nty tiles of columns times chunks of lz
// planes, times the species groups (innermost, so that the groups of a tile
// run together on one XCD and share the flow's data in its L2).
struct SpecPlan {
    const FInst *inst;
    const int *blk0;  // first block of each instance, ninst + 1 entries
    int ninst, lz;
};

// G quotients by one divisor, exactly rounded.  r is 1/b after two
// Newton-Raphson steps and a quotient q = a r is corrected by its exact
// residual, q + (a - b q) r, which rounds to a/b (Markstein, IBM J. Res. Dev.
// 34, 1990) while nothing over- or underflows; operands outside a wide range
// are divided as such.  Three operations per quotient where a division takes
// about ten: the transverse corrections divide every species of a state by
// the same density.
template <int G>
__device__ __forceinline__ void sp_divide(double (&a)[G], double b)
{
    double r = __builtin_amdgcn_rcp(b), v[G];
    r = fma(r, fma(-b, r, 1.0), r);
    r = fma(r, fma(-b, r, 1.0), r);
    // smallest and largest magnitude by the high words
    unsigned lo = __double2hiint(b) & 0x7fffffff, hi = lo;
#pragma unroll
    for (int q = 0; q < G; ++q) {
        const unsigned h = __double2hiint(a[q]) & 0x7fffffff;
        lo = min(lo, h);
        hi = max(hi, h);
        const double t = a[q] * r;
        v[q] = fma(fma(-b, t, a[q]), r, t);
    }
    if (lo < 0x20000000u || hi > 0x5f000000u) {  // below 2^-511, above 2^497
#pragma unroll
        for (int q = 0; q < G; ++q) v[q] = a[q] / b;
    }
#pragma unroll
    for (int q = 0; q < G; ++q) a[q] = v[q];
}

// The PPM pieces of mc_hydro.h's ppm_reconstruct and ppm_int_wave, by
// themselves and without branches: the same expressions, so that neighbouring
// cells can share slopes and edge values.
// Twice the van Leer slope of the cell between the differences dl = s0 - s-1
// and dr = s1 - s0: multiplications by powers of two are exact, so the factor
// is taken off in sp_edge's constant.
__device__ __forceinline__ double sp_slope2(double dl, double dr, double dc)
{
    const double v = fsign1(dc) * fmin(fabs(dc), 4.0 * fmin(fabs(dl), fabs(dr)));
    return dl * dr > 0.0 ? v : 0.0;
}
// edge value between cells a (below) and b, with twice their slopes; the
// product 0.5 (b + a) is exact, so it fuses with the subtraction
__device__ __forceinline__ double sp_edge(double a, double b, double va, double vb)
{
    double e = fma(HALF, b + a, -((HALF * SIXTH) * (vb - va)));
    e = fmax(e, fmin(b, a));
    return fmin(e, fmax(b, a));
}
// what a direction's wave speed gives every species of a cell
struct SpWave {
    double hs, t;  // half the Courant number; 1 - 2/3 of it, negated for a positive speed
    bool neg;
    __device__ __forceinline__ SpWave(double u, double dtdx)
    {
        const double sigma = fabs(u) * dtdx;
        neg = u <= 0.0;
        hs = HALF * sigma;
        t = 1.0 - TWO3RD * sigma;
        t = neg ? t : -t;
    }
};
// limited, flattened parabola of cell value s0 with edges sm, sp, and its
// averages swept by the wave: the minus state of the high face (im), the plus
// state of the low face (ip)
__device__ __forceinline__ void sp_states(double s0, double sm, double sp, double fl, const SpWave &w, double &im,
                                          double &ip)
{
    const double f0 = (1.0 - fl) * s0;
    sm = fl * sm + f0;
    sp = fl * sp + f0;
    const double dp = sp - s0, dm = s0 - sm, ap = fabs(dp), am = fabs(dm);
    const bool flat = dp * dm <= 0.0, cp = ap >= 2.0 * am, cm = am >= 2.0 * ap;
    const double s3 = 3.0 * s0, np = fma(-2.0, sm, s3), nm = fma(-2.0, sp, s3);
    const double sp2 = flat ? s0 : (cp ? np : sp), sm2 = flat ? s0 : ((cm && !cp) ? nm : sm);
    const double s6 = 6.0 * s0 - 3.0 * (sm2 + sp2);
    const double h = w.hs * (sp2 - sm2 + w.t * s6);
    const double vp = sp2 - h, vm = sm2 + h;
    im = w.neg ? sp2 : vp;
    ip = w.neg ? vm : sm2;
}
// the same from the cell and two neighbours on either side
__device__ __forceinline__ void sp_trace(const double *s, double fl, const SpWave &w, double &im, double &ip)
{
    const double d0 = s[1] - s[0], d1 = s[2] - s[1], d2 = s[3] - s[2], d3 = s[4] - s[3];
    const double v1 = sp_slope2(d0, d1, s[2] - s[0]), v2 = sp_slope2(d1, d2, s[3] - s[1]),
                 v3 = sp_slope2(d2, d3, s[4] - s[2]);
    sp_states(s[2], sp_edge(s[1], s[2], v1, v2), sp_edge(s[2], s[3], v2, v3), fl, w, im, ip);
}

// a value that is the same in every lane, in scalar registers
__device__ __forceinline__ double uniform_d(double v)
{
    const long long b = __double_as_longlong(v);
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)b);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)((unsigned long long)b >> 32));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// the value of the lane below (DOWN) or above in the 16 lanes of a DPP row
template <bool DOWN>
__device__ __forceinline__ double lane_shift(double v)
{
    constexpr int ctrl = DOWN ? 0x111 : 0x101;  // row_shr:1, row_shl:1
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, ctrl, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), ctrl, 0xf, 0xf, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// Arrays whose base is held in scalar registers: a region of interleaved
// pairs (16 bytes an element) or of doubles.
struct PairBase {
    double *p;
    __device__ __forceinline__ gdbl2 &operator[](idx_t idx) const
    {
        typedef __attribute__((address_space(1))) char gchar;
        return *(gdbl2 *)((gchar *)p + idx * 16u);
    }
};
struct DblBase {
    double *p;
    __device__ __forceinline__ gdouble &operator[](idx_t idx) const
    {
        typedef __attribute__((address_space(1))) char gchar;
        return *(gdouble *)((gchar *)p + idx * 8u);
    }
};
__device__ __forceinline__ double *ring_base(double *a, const FInst &I, int C, int c)
{
    return uniform_ptr(a + ((long)C * I.offE + (long)c * I.nE));
}

// Riemann weight and mass flux of a face times the interface value
__device__ __forceinline__ double sp_flux(const dbl2 &rw, double xl, double xr)
{
    return rw.x * fma(rw.y, xl, (1.0 - rw.y) * xr);  // the weight is 0, 1/2 or 1: its product is exact
}

constexpr int SPEC_G = 2;                 // species of a block: one pair
constexpr int SPEC_TX = 16, SPEC_TY = 16; // columns of a tile, ring included

// One block: a tile of columns, one thread each (the interior, at most
// (TX - 2) x (TY - 2), and a ring of one), two species, a chunk of planes.  For
// every plane p of the ring-extended chunk: the species' x, y and z traces of
// plane p, the first-stage fluxes on its low faces, the transverse fluxes
// they allow (F^{x|y}, F^{y|x} on plane p, F^{z|x}, F^{z|y} on its low
// z-faces, F^{x|z}, F^{y|z} on plane p - 1) and the final fluxes of plane
// p - 1 in x and y and of the low z-faces of p.  An x-neighbour is a lane of
// the same 16-lane row, a y-neighbour's values go through LDS (five barriers a
// plane), what the next plane needs stays with the thread.
__global__ __launch_bounds__(SPEC_TX *SPEC_TY) __attribute__((amdgpu_waves_per_eu(2))) void K_species(SpecPlan sp,
                                                                                                     Ctx x)
{
    constexpr int G = SPEC_G, TX = SPEC_TX, TY = SPEC_TY, NT = TX * TY, LW = TX + 4, NF = 4 * (TX + TY);
    static_assert(TX == 16, "x-neighbours share a DPP row");
    static_assert(G == 2, "a block takes one pair");
    static_assert(NF <= NT, "one halo element per thread");
    __shared__ dbl2 LU[3][LW * (TY + 4)];  // U1's species of planes p - 1, p, p + 1, two cells beyond the ring
    __shared__ double LR[LW * (TY + 4)];   // 1/rho of plane p
    // exchanged with y-neighbours, with guard rows: minus states and fluxes, mass fluxes
    __shared__ dbl2 A[2][NT + 2 * TX], B[2][NT + 2 * TX];
    __shared__ double R[3][NT + 2 * TX];
    __shared__ dbl2 S[2][4][NT];           // the thread's x and y states of this plane and the one before
    const int lb = logical_block();
    int m;
    {
        int lo = 0, hi = sp.ninst - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (sp.blk0[mid] <= lb) lo = mid;
            else hi = mid - 1;
        }
        m = lo;
    }
    const FInst I = sp.inst[m];  // a copy: stores do not force its fields to be read again
    const int n0 = I.n[0], n1 = I.n[1], ex0 = I.ext[0];
    const int ntx = (n0 + TX - 3) / (TX - 2), nty = (n1 + TY - 3) / (TY - 2);
    int b = lb - sp.blk0[m];
    const int pr = b % NSPEC_PAIRS;
    b /= NSPEC_PAIRS;
    const int x0 = (b % ntx) * (TX - 2), y0 = ((b / ntx) % nty) * (TY - 2), zc0 = I.zlo + (b / (ntx * nty)) * sp.lz;
    const int w = min(TX - 2, n0 - x0), h = min(TY - 2, n1 - y0), ztop = I.zlo + I.zn;
    const int zc1 = min(zc0 + sp.lz, ztop);
    const int tid = threadIdx.x, tx = tid % TX, ty = tid / TX, at = tid + TX;
    // a wavefront (four rows) above the last tile's ring has nothing to do;
    // the barriers below wait for the wavefronts that are left.  The first
    // two, which load the halo, always stay.
    if (tid >= 128 && (tid & ~63) / TX > h + 1) return;
    const int iu = x0 - 1 + tx, ju = y0 - 1 + ty;  // the thread's column
    const int i = min(iu, n0), j = min(ju, n1);    // within the ring
    const idx_t cxy = (idx_t)bmap(iu, n0, I.periodic) + (idx_t)n0 * (idx_t)bmap(ju, n1, I.periodic);
    const idx_t cs = (idx_t)n0 * (idx_t)n1, es = (idx_t)ex0 * (idx_t)I.ext[1];  // plane strides
    auto zmap = [&](int k) -> idx_t { return cs * (idx_t)plane_w(I, k); };
    // bases of everything the block reads and writes, taken once
    const SpeciesPairs XU = cell_species(x.U1X, I);
    const PairBase PU{uniform_ptr(XU.base + pr * XU.stride)};
    const DblBase RI{uniform_ptr(x.Q + ((long)NFQ * I.offW + (long)FQ_RI * I.nW))};
    const DblBase QU{uniform_ptr(x.Q + ((long)NFQ * I.offW + (long)FQ_U * I.nW))};
    const DblBase FL{ring_base(x.FL, I, 1, 0)};
    const PairBase F0{ring_base(x.FD[0], I, NFF, FF_RHO)}, F1{ring_base(x.FD[1], I, NFF, FF_RHO)},
        F2{ring_base(x.FD[2], I, NFF, FF_RHO)};
    const PairBase R0{ring_base(x.RW, I, 6, 0)}, R1{ring_base(x.RW, I, 6, 2)}, R2{ring_base(x.RW, I, 6, 4)};
    const PairBase TYX{ring_base(x.FT[0], I, NFF, FF_RHO)}, TZX{ring_base(x.FT[1], I, NFF, FF_RHO)},
        TXY{ring_base(x.FT[2], I, NFF, FF_RHO)}, TZY{ring_base(x.FT[3], I, NFF, FF_RHO)},
        TXZ{ring_base(x.FT[4], I, NFF, FF_RHO)}, TYZ{ring_base(x.FT[5], I, NFF, FF_RHO)};
    const PairBase N0{ring_base(x.FN[0], I, NFN, FN_FR)}, N1{ring_base(x.FN[1], I, NFN, FN_FR)},
        N2{ring_base(x.FN[2], I, NFN, FN_FR)};
    const long odv = (long)(FN_DIV - FN_FR) * I.nE, osp = (long)(FN_X - FN_FR + 2 * pr) * I.nE;
    // the padding slot of the last pair stands in for a species that is not
    // there: its neighbour, so that it runs through the same arithmetic
    const bool pad = 2 * pr + 1 >= NSPEC;
    auto load_u = [&](idx_t c) -> dbl2 {
        dbl2 u = PU[c];
        if (pad) u.y = u.x;
        return u;
    };
    // the thread's halo element of LU and LR (threads below NF)
    int hx = 0, hy = 0;
    if (tid < 4 * TX) {
        const int r = tid / TX;
        hx = tid % TX;
        hy = r < 2 ? r - 2 : h + r;  // two rows below the ring, two above
    } else if (tid < NF) {
        const int t = tid - 4 * TX, r = t / TY;
        hy = t % TY;
        hx = r < 2 ? r - 2 : TX + r - 2;
    }
    const bool halo = tid < NF, ring = ty <= h + 1;
    const idx_t chxy = (idx_t)bmap(x0 - 1 + hx, n0, I.periodic) + (idx_t)n0 * (idx_t)bmap(y0 - 1 + hy, n1, I.periodic);
    const int lhalo = (hy + 2) * LW + hx + 2, lown = (ty + 2) * LW + tx + 2;
    const double dt = uniform_d(x.dt_cur[m]), dx0 = uniform_d(I.dx[0]), dx1 = uniform_d(I.dx[1]), dx2 = uniform_d(I.dx[2]);
    const double rx = uniform_d(dt / dx0), ry = uniform_d(dt / dx1), rz = uniform_d(dt / dx2);
    const double cx = uniform_d(rx / 3.0), cy = uniform_d(ry / 3.0), cz = uniform_d(rz / 3.0);
    const double hx2 = uniform_d(0.5 * dt / dx0), hy2 = uniform_d(0.5 * dt / dx1), hz2 = uniform_d(0.5 * dt / dx2);
    // which final fluxes the thread stores
    const bool col = tx >= 1 && tx <= w && ty >= 1 && ty <= h;
    const bool st_x = ty >= 1 && ty <= h && ((tx >= 1 && tx <= w) || (tx == w + 1 && iu == n0));
    const bool st_y = tx >= 1 && tx <= w && ((ty >= 1 && ty <= h) || (ty == h + 1 && ju == n1));

#define SP_EACH for (int q = 0; q < G; ++q)
    auto below = [&](const dbl2 &v) -> dbl2 { return dbl2{lane_shift<true>(v.x), lane_shift<true>(v.y)}; };
    auto above = [&](const dbl2 &v) -> dbl2 { return dbl2{lane_shift<false>(v.x), lane_shift<false>(v.y)}; };
    auto flux = [&](const dbl2 &rw, const dbl2 &l, const dbl2 &r) -> dbl2 {
        return dbl2{sp_flux(rw, l.x, r.x), sp_flux(rw, l.y, r.y)};
    };
    // a state corrected by one transverse flux difference (Source/trans.F90:151-158)
    auto corr1 = [&](const dbl2 &s, double rho, double cdt, double df, const dbl2 &dx_) -> dbl2 {
        double o[G] = {rho * s.x - cdt * dx_.x, rho * s.y - cdt * dx_.y};
        sp_divide<G>(o, rho - cdt * df);
        return dbl2{o[0], o[1]};
    };
    // and by two (Source/trans.F90:393-405)
    auto corr2 = [&](const dbl2 &s, double rho, double h2, double df2, const dbl2 &d2, double h3, double df3,
                     const dbl2 &d3) -> dbl2 {
        double o[G] = {rho * s.x - h2 * d2.x - h3 * d3.x, rho * s.y - h2 * d2.y - h3 * d3.y};
        sp_divide<G>(o, rho - h2 * df2 - h3 * df3);
        return dbl2{o[0], o[1]};
    };

    // carried from plane to plane
    dbl2 uc, uu, uuu;                  // U1's species of planes p, p + 1, p + 2
    double rc, ru, ruu;                // 1/rho of these planes
    dbl2 zs, ze;                       // z slope of plane p, edge value of z-face p
    const dbl2 zero = dbl2{0.0, 0.0};
    dbl2 zm = zero, zmx = zero, zmy = zero, zmz = zero;  // minus state of z-face p: traced, corrected by x, y, both
    dbl2 fzk = zero, fzxk = zero, fzyk = zero;           // F^z, F^{z|x}, F^{z|y} on z-face p - 1
    double rzk = 0.0, rzxk = 0.0, rzyk = 0.0;            // their mass fluxes
    dbl2 k0 = zero, k1 = zero;                           // x and y state densities of plane p - 1
    int p = zc0 - 1;
    {
        const idx_t cb = cxy + zmap(p - 2), ca = cxy + zmap(p - 1), c0 = cxy + zmap(p), c1 = cxy + zmap(p + 1),
                    c2 = cxy + zmap(p + 2);
        rc = RI[c0];
        ru = RI[c1];
        ruu = RI[c2];
        uc = load_u(c0);
        uu = load_u(c1);
        uuu = load_u(c2);
        const dbl2 xb = load_u(cb) * RI[cb], xa = load_u(ca) * RI[ca], xc = uc * rc, xu = uu * ru;
        SP_EACH
        {
            const double d0 = xa[q] - xb[q], d1 = xc[q] - xa[q], d2 = xu[q] - xc[q];
            zs[q] = sp_slope2(d1, d2, xu[q] - xa[q]);
            ze[q] = sp_edge(xa[q], xc[q], sp_slope2(d0, d1, xc[q] - xb[q]), zs[q]);
        }
    }
    idx_t e = (idx_t)(i + 1) + (idx_t)ex0 * ((idx_t)(j + 1) + (idx_t)I.ext[1] * (idx_t)(p - I.zlo + 1));
    dbl2 uh = zero;
    double rh = 0.0;
    if (halo) {
        const idx_t ch = chxy + zmap(p);
        uh = load_u(ch);
        rh = RI[ch];
    }
    int u0 = 1;  // LU's buffer of plane p
    if (ring) {
        LU[u0][lown] = uc;
        LR[lown] = rc;
    }
    if (halo) {
        LU[u0][lhalo] = uh;
        LR[lhalo] = rh;
    }
    double ux, uy, uz, fl;
    {
        const idx_t c = cxy + zmap(p);
        ux = QU[c];
        uy = DblBase{QU.p + I.nW}[c];
        uz = DblBase{QU.p + 2 * I.nW}[c];
        fl = FL[e];
    }
    __syncthreads();
    for (int par = 0; p <= zc1; ++p, e += es, par ^= 1) {
        const idx_t ek = p > I.zlo - 1 ? e - es : e;  // plane p - 1
        const dbl2 w0 = F0[e], w1 = F1[e], w2 = F2[e];
        // ---- traces of plane p (Source/ppm.F90:309-743, species): the minus
        // states of the cell's high faces, the plus states of its low faces
        dbl2 xm, xp, ym, yp, zmn, zp;
        {
            const SpWave wvx(ux, rx), wvy(uy, ry), wvz(uz, rz);
            const dbl2 xc = uc * rc, xu = uu * ru, xuu = uuu * ruu;
            const dbl2 *L = LU[u0];
            dbl2 s[5];
#pragma unroll
            for (int o = 0; o < 5; ++o) s[o] = o == 2 ? xc : L[lown + o - 2] * LR[lown + o - 2];
            SP_EACH
            {
                const double t[5] = {s[0][q], s[1][q], s[2][q], s[3][q], s[4][q]};
                double a, c;
                sp_trace(t, fl, wvx, a, c);
                xm[q] = a;
                xp[q] = c;
            }
#pragma unroll
            for (int o = 0; o < 5; ++o) s[o] = o == 2 ? xc : L[lown + (o - 2) * LW] * LR[lown + (o - 2) * LW];
            SP_EACH
            {
                const double t[5] = {s[0][q], s[1][q], s[2][q], s[3][q], s[4][q]};
                double a, c;
                sp_trace(t, fl, wvy, a, c);
                ym[q] = a;
                yp[q] = c;
            }
            // in z the slope and edge below come from the plane before
            SP_EACH
            {
                const double vu = sp_slope2(xu[q] - xc[q], xuu[q] - xu[q], xuu[q] - xc[q]);
                const double eu = sp_edge(xc[q], xu[q], zs[q], vu);
                double a, c;
                sp_states(xc[q], ze[q], eu, fl, wvz, a, c);
                zmn[q] = a;
                zp[q] = c;
                zs[q] = vu;
                ze[q] = eu;
            }
        }
        A[0][at] = ym;
        R[0][at] = w1.x;
        S[par][0][tid] = xm;
        S[par][1][tid] = xp;
        S[par][2][tid] = ym;
        S[par][3][tid] = yp;
        const dbl2 q0 = R0[e], q1 = R1[e], q2 = R2[e];
        __syncthreads();
        // ---- first-stage fluxes on the low faces of plane p
        const dbl2 fx = flux(w0, below(xm), xp), fy = flux(w1, A[0][at - TX], yp), fz = flux(w2, zm, zp);
        B[0][at] = fy;
        const dbl2 wxy = TXY[e], wyx = TYX[e], wzx = TZX[e], wzy = TZY[e], wxz = TXZ[ek], wyz = TYZ[ek];
        __syncthreads();
        // ---- one-direction corrections
        dbl2 zpx, zpy, zmxn, zmyn, xpy, xmy, ypx, xpz, xmz, ypz;
        {
            const dbl2 dX = above(fx) - fx, dY = B[0][at + TX] - fy, dZ = fz - fzk;
            const double dfx = lane_shift<false>(w0.x) - w0.x, dfy = R[0][at + TX] - w1.x, dfz = w2.x - rzk;
            xpy = corr1(xp, q0.x, cy, dfy, dY);
            xmy = corr1(xm, q0.y, cy, dfy, dY);
            ypx = corr1(yp, q1.x, cx, dfx, dX);
            A[0][at] = corr1(ym, q1.y, cx, dfx, dX);
            zpx = corr1(zp, q2.x, cx, dfx, dX);
            zpy = corr1(zp, q2.x, cy, dfy, dY);
            zmxn = corr1(zmn, q2.y, cx, dfx, dX);
            zmyn = corr1(zmn, q2.y, cy, dfy, dY);
            // zone p - 1
            xpz = corr1(S[par ^ 1][1][tid], k0.x, cz, dfz, dZ);
            xmz = corr1(S[par ^ 1][0][tid], k0.y, cz, dfz, dZ);
            ypz = corr1(S[par ^ 1][3][tid], k1.x, cz, dfz, dZ);
            A[1][at] = corr1(S[par ^ 1][2][tid], k1.y, cz, dfz, dZ);
        }
        R[1][at] = wyx.x;
        R[2][at] = wyz.x;
        __syncthreads();
        // ---- transverse fluxes
        const dbl2 fxy = flux(wxy, below(xmy), xpy), fyx = flux(wyx, A[0][at - TX], ypx),
                   fxz = flux(wxz, below(xmz), xpz), fyz = flux(wyz, A[1][at - TX], ypz), fzx = flux(wzx, zmx, zpx),
                   fzy = flux(wzy, zmy, zpy);
        B[0][at] = fyx;
        B[1][at] = fyz;
        // the next planes' cells
        dbl2 un;
        double rn;
        {
            const idx_t c = cxy + zmap(p + 3);
            un = load_u(c);
            rn = RI[c];
        }
        if (halo && p < zc1) {
            const idx_t c = chxy + zmap(p + 1);
            uh = load_u(c);
            rh = RI[c];
        }
        const dbl2 wf0 = N0[ek], wf1 = N1[ek], wf2 = N2[e];
        const double dv0 = DblBase{N0.p + odv}[ek], dv1 = DblBase{N1.p + odv}[ek], dv2 = DblBase{N2.p + odv}[e];
        __syncthreads();
        // ---- two-direction corrections
        dbl2 xpp, xmp, ypp, zpp, zmzn;
        {
            const dbl2 dXY = above(fxy) - fxy, dYX = B[0][at + TX] - fyx, dXZ = above(fxz) - fxz,
                       dYZ = B[1][at + TX] - fyz, dZX = fzx - fzxk, dZY = fzy - fzyk;
            const double rxy = lane_shift<false>(wxy.x) - wxy.x, ryx = R[1][at + TX] - wyx.x,
                         rxz = lane_shift<false>(wxz.x) - wxz.x, ryz = R[2][at + TX] - wyz.x, rzx = wzx.x - rzxk,
                         rzy = wzy.x - rzyk;
            xpp = corr2(S[par ^ 1][1][tid], k0.x, hy2, ryz, dYZ, hz2, rzy, dZY);
            xmp = corr2(S[par ^ 1][0][tid], k0.y, hy2, ryz, dYZ, hz2, rzy, dZY);
            ypp = corr2(S[par ^ 1][3][tid], k1.x, hx2, rxz, dXZ, hz2, rzx, dZX);
            A[1][at] = corr2(S[par ^ 1][2][tid], k1.y, hx2, rxz, dXZ, hz2, rzx, dZX);
            zpp = corr2(zp, q2.x, hx2, rxy, dXY, hy2, ryx, dYX);
            zmzn = corr2(zmn, q2.y, hx2, rxy, dXY, hy2, ryx, dYX);
        }
        const int un_ = u0 == 2 ? 0 : u0 + 1, uk_ = u0 == 0 ? 2 : u0 - 1;
        if (ring) {
            LU[un_][lown] = uu;
            LR[lown] = ru;
        }
        if (halo) {
            LU[un_][lhalo] = uh;
            LR[lhalo] = rh;
        }
        if (p < zc1) {  // the next plane's traces
            const idx_t c = cxy + zmap(p + 1);
            ux = QU[c];
            uy = DblBase{QU.p + I.nW}[c];
            uz = DblBase{QU.p + 2 * I.nW}[c];
            fl = FL[e + es];
        }
        __syncthreads();
        // ---- final fluxes with their artificial viscosity
        // (Source/Castro_hydro_nd.F90:174-245), before the normalisation
        auto store = [&](const PairBase &N, double dxd, idx_t ee, const dbl2 &wf, double dv, const dbl2 &l,
                         const dbl2 &r, const dbl2 &ur, const dbl2 &ul) {
            const dbl2 f = flux(wf, l, r);
            PairBase{N.p + osp}[ee] = dbl2{f.x + dxd * (dv * (ur.x - ul.x)), f.y + dxd * (dv * (ur.y - ul.y))};
        };
        const dbl2 xl = below(xmp);
        const dbl2 uk = LU[uk_][lown];
        if (p > zc0) {
            if (st_x) store(N0, dx0, ek, wf0, dv0, xl, xpp, uk, LU[uk_][lown - 1]);
            if (st_y) store(N1, dx1, ek, wf1, dv1, A[1][at - TX], ypp, uk, LU[uk_][lown - LW]);
        }
        if (col && p >= zc0 && (p < zc1 || zc1 == ztop)) store(N2, dx2, e, wf2, dv2, zmz, zpp, uc, uk);
        u0 = un_;
        uc = uu;
        uu = uuu;
        uuu = un;
        rc = ru;
        ru = ruu;
        ruu = rn;
        zm = zmn;
        zmx = zmxn;
        zmy = zmyn;
        zmz = zmzn;
        fzk = fz;
        fzxk = fzx;
        fzyk = fzy;
        rzk = w2.x;
        rzxk = wzx.x;
        rzyk = wzy.x;
        k0 = q0;
        k1 = q1;
    }
#undef SP_EACH
}

} // namespace mc
