// The transverse and final fluxes of the fused step, without the species, in
// one launch: a block owns a tile of columns and marches in z, so the six
// transverse fluxes of a cell never go through memory (the species stage
// gets their mass fluxes and Riemann weights).
#pragma once

#include "mc_species.h"

namespace mc {

// A transverse flux without species: URHO..UEDEN, Godunov p and u.
struct TFlux {
    double f[UEDEN + 1], gp, gu;
};
// Its difference across a zone, as the corrections use it (Source/trans.F90:
// 165-229): the conserved fluxes' differences and the pressure's.
struct TDiff {
    double f[UEDEN + 1], p;
};
__device__ __forceinline__ TDiff tdiff(const TFlux &r, const TFlux &l, double gamc)
{
    TDiff o;
#pragma unroll
    for (int n = 0; n <= UEDEN; ++n) o.f[n] = r.f[n] - l.f[n];
    const double dup = r.gp * r.gu - l.gp * l.gu;
    const double du = r.gu - l.gu;
    const double pav = HALF * (r.gp + l.gp);
    o.p = dup + pav * du * (gamc - 1.0);
    return o;
}

// trans1_hydro and trans2_hydro (mc_hydro.h) from the differences: the same
// expressions.  D: the face direction of the state.
template <int D>
__device__ __forceinline__ FaceH correct1(const QInH &q, const TDiff &t, double cdt)
{
    const double rr = q.rho;
    const double ru = rr * q.u, rv = rr * q.v, rw = rr * q.w;
    const double re = q.rhoe + HALF * rr * (q.u * q.u + q.v * q.v + q.w * q.w);
    double rn = rr - cdt * t.f[URHO];
    double un = ru - cdt * t.f[UMX], vn = rv - cdt * t.f[UMY], wn = rw - cdt * t.f[UMZ], en = re - cdt * t.f[UEDEN];
    const bool reset = rn < 0.0;
    if (reset) {
        rn = rr;
        un = ru;
        vn = rv;
        wn = rw;
        en = re;
    }
    const double ri = 1.0 / rn;
    const double ek = HALF * (un * un + vn * vn + wn * wn) * ri;
    const double p = reset ? q.p : fmax(q.p - cdt * t.p, small_pres);
    return face_of(D, rn, un * ri, vn * ri, wn * ri, p, en - ek);
}
template <int D>
__device__ __forceinline__ FaceH correct2(const QInH &q, const TDiff &a, double ha, const TDiff &b, double hb)
{
    const double rr = q.rho;
    const double ru = rr * q.u, rv = rr * q.v, rw = rr * q.w;
    const double re = q.rhoe + HALF * rr * (q.u * q.u + q.v * q.v + q.w * q.w);
    double rn = rr - ha * a.f[URHO] - hb * b.f[URHO];
    double un = ru - ha * a.f[UMX] - hb * b.f[UMX], vn = rv - ha * a.f[UMY] - hb * b.f[UMY],
           wn = rw - ha * a.f[UMZ] - hb * b.f[UMZ], en = re - ha * a.f[UEDEN] - hb * b.f[UEDEN];
    const bool reset = rn < 0.0;
    if (reset) {
        rn = rr;
        un = ru;
        vn = rv;
        wn = rw;
        en = re;
    }
    const double ek = HALF * (un * un + vn * vn + wn * wn) / rn;
    const double p = reset ? q.p : q.p - ha * a.p - hb * b.p;
    return face_of(D, rn, un / rn, vn / rn, wn / rn, fmax(p, small_pres), en - ek);
}

// Riemann problem on a D-face; its transverse flux in absolute order
template <int D>
__device__ __forceinline__ TFlux tflux(const FaceH &L, const FaceH &R, double cl, double cr, double gl, double gr,
                                       dbl2 &rw)
{
    RiemannH o;
    riemann_hydro(L, R, cl, cr, gl, gr, o);
    rw = dbl2{o.f_rho, o.fpl};
    TFlux f;
    f.f[URHO] = o.f_rho;
    f.f[UMX] = D == 0 ? o.f_mn : o.f_mt;
    f.f[UMY] = D == 0 ? o.f_mt : (D == 1 ? o.f_mn : o.f_mtt);
    f.f[UMZ] = D == 2 ? o.f_mn : o.f_mtt;
    f.f[UEDEN] = o.f_E;
    f.gp = o.g_p;
    f.gu = o.g_un;
    return f;
}

template <bool DOWN>
__device__ __forceinline__ FaceH lane_shift(const FaceH &f)
{
    return FaceH{lane_shift<DOWN>(f.rho), lane_shift<DOWN>(f.un), lane_shift<DOWN>(f.ut),
                 lane_shift<DOWN>(f.utt), lane_shift<DOWN>(f.p),  lane_shift<DOWN>(f.rhoe)};
}
__device__ __forceinline__ TFlux lane_above(const TFlux &t)
{
    TFlux o;
#pragma unroll
    for (int n = 0; n <= UEDEN; ++n) o.f[n] = lane_shift<false>(t.f[n]);
    o.gp = lane_shift<false>(t.gp);
    o.gu = lane_shift<false>(t.gu);
    return o;
}

// Order of evaluation: what follows is addressed through e, which waits for
// these values (left alone, the compiler loads and starts everything at once
// and spills a hundred registers).
__device__ __forceinline__ void finish(idx_t &e, double &v) { asm volatile("" : "+v"(e), "+v"(v)); }
__device__ __forceinline__ void finish(idx_t &e, FaceH &f)
{
    finish(e, f.rho);
    finish(e, f.un);
    finish(e, f.ut);
    finish(e, f.utt);
    finish(e, f.p);
    finish(e, f.rhoe);
}
__device__ __forceinline__ void finish(idx_t &e, TFlux &t)
{
#pragma unroll
    for (int n = 0; n <= UEDEN; ++n) finish(e, t.f[n]);
    finish(e, t.gp);
    finish(e, t.gu);
}
__device__ __forceinline__ void finish(idx_t &e, TDiff &t)
{
#pragma unroll
    for (int n = 0; n <= UEDEN; ++n) finish(e, t.f[n]);
    finish(e, t.p);
}

// Tiles, planes and threads as in K_species (trans1, Source/trans.F90:14-243;
// trans2, :250-505; Source/riemann.F90:10-331; apply_av,
// Source/Castro_hydro_nd.F90:174-245).  Three barriers a plane: the minus
// states and then the fluxes of the y-faces, and the twice-corrected minus
// states, go to the neighbouring row through LDS.
//
// K_trans1c and K_final write and read the six transverse fluxes, 8 doubles a
// face each, and read every state again; here 2 doubles a face are left of
// them.  256^3: 6.2 ms against 5.0 + 4.6.  A CU holds two blocks (registers)
// and its VALUs are 35% busy: what a plane waits for counts.  It moves 39 GB
// past the L2s where its arrays hold 15.5, as a plane of an XCD's 64 blocks
// does not fit its L2 between two uses of a state; but with the z- and
// x-states and the z-flux kept in LDS from use to use (46 pairs read a plane
// instead of 62, neighbouring rows by lane permutes to make room) it took 6.4.
// Reading a face's zones for the viscosity together instead of as they are
// used took it from 6.8 to 6.2, keeping a plane's states across two
// corrections from 7.6 to 7.0 and the next plane's first loads ahead of the
// last barrier to 6.8; keeping more spills (7.8).
__global__ __launch_bounds__(SPEC_TX *SPEC_TY) __attribute__((amdgpu_waves_per_eu(2))) void K_transfinal(SpecPlan sp,
                                                                                                        Ctx x)
{
    constexpr int TX = SPEC_TX, TY = SPEC_TY, NT = TX * TY, ND = NT + 2 * TX;
    __shared__ double A[3][6][ND], B[2][7][ND];
    int m, b;
    {
        const int lb = logical_block();
        int lo = 0, hi = sp.ninst - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (sp.blk0[mid] <= lb) lo = mid;
            else hi = mid - 1;
        }
        m = lo;
        b = lb - sp.blk0[m];
    }
    const FInst I = sp.inst[m];
    const int n0 = I.n[0], n1 = I.n[1], ex0 = I.ext[0];
    const int ntx = (n0 + TX - 3) / (TX - 2), nty = (n1 + TY - 3) / (TY - 2);
    const int x0 = (b % ntx) * (TX - 2), y0 = ((b / ntx) % nty) * (TY - 2), zc0 = I.zlo + (b / (ntx * nty)) * sp.lz;
    const int w = min(TX - 2, n0 - x0), h = min(TY - 2, n1 - y0), ztop = I.zlo + I.zn;
    const int zc1 = min(zc0 + sp.lz, ztop);
    const int tid = threadIdx.x, tx = tid % TX, ty = tid / TX, at = tid + TX;
    if ((tid & ~63) / TX > h + 1) return;  // a wavefront above the tile's ring (K_species)
    const int iu = x0 - 1 + tx, ju = y0 - 1 + ty;
    const int i = min(iu, n0), j = min(ju, n1);
    const idx_t cxy = (idx_t)bmap(i, n0, I.periodic) + (idx_t)n0 * (idx_t)bmap(j, n1, I.periodic);
    const idx_t cym = (idx_t)bmap(i, n0, I.periodic) + (idx_t)n0 * (idx_t)bmap(j - 1, n1, I.periodic);
    const idx_t cs = (idx_t)n0 * (idx_t)n1, es = (idx_t)ex0 * (idx_t)I.ext[1];
    const idx_t ox = i < n0 ? 1u : 0u, oy = j < n1 ? (idx_t)ex0 : 0u;
    const long np = 2 * I.nE;  // doubles from one pair region to the next
    const DblBase QC{uniform_ptr(x.Q + ((long)NFQ * I.offW + (long)FQ_C * I.nW))};
    const DblBase QG{uniform_ptr(x.Q + ((long)NFQ * I.offW + (long)FQ_G * I.nW))};
    const DblBase DV{ring_base(x.DV, I, 1, 0)}, U1{uniform_ptr(x.U1 + (long)NU1 * I.offW)};
    const PairBase F0{ring_base(x.FD[0], I, NFF, 0)}, F1{ring_base(x.FD[1], I, NFF, 0)}, F2{ring_base(x.FD[2], I, NFF, 0)};
    const PairBase P0{ring_base(x.SP[0], I, NFS, 0)}, P1{ring_base(x.SP[1], I, NFS, 0)}, P2{ring_base(x.SP[2], I, NFS, 0)};
    const PairBase M0{ring_base(x.SM[0], I, NFS, 0)}, M1{ring_base(x.SM[1], I, NFS, 0)}, M2{ring_base(x.SM[2], I, NFS, 0)};
    const PairBase TYX{ring_base(x.FT[0], I, NFF, 0)}, TZX{ring_base(x.FT[1], I, NFF, 0)},
        TXY{ring_base(x.FT[2], I, NFF, 0)}, TZY{ring_base(x.FT[3], I, NFF, 0)}, TXZ{ring_base(x.FT[4], I, NFF, 0)},
        TYZ{ring_base(x.FT[5], I, NFF, 0)};
    auto state = [&](const PairBase &S, idx_t q) -> QInH {
        const dbl2 a = S[q], c = PairBase{S.p + np}[q], d = PairBase{S.p + 2 * np}[q];
        return QInH{a.x, a.y, c.x, c.y, d.x, d.y, 0.0};
    };
    auto flux = [&](const PairBase &F, idx_t q) -> TFlux {
        const dbl2 a = PairBase{F.p + np}[q], c = PairBase{F.p + 2 * np}[q], d = PairBase{F.p + 3 * np}[q];
        TFlux o;
        o.f[URHO] = F[q].x;
        o.f[UMX] = a.x;
        o.f[UMY] = a.y;
        o.f[UMZ] = c.x;
        o.f[UEDEN] = c.y;
        o.gp = d.x;
        o.gu = d.y;
        return o;
    };
    auto zone = [&](idx_t c, double (&u)[UEINT + 1]) {
#pragma unroll
        for (int n = 0; n <= UEINT; ++n) u[n] = DblBase{U1.p + n * I.nW}[c];
    };
    // FaceAv of a face from its corner nodes, in face_av's order, and its zones
    auto av = [&](double d1, double d2, double d3, double d4, const double (&ur)[UEINT + 1],
                  const double (&ul)[UEINT + 1]) -> FaceAv {
        FaceAv v;
        v.div1 = 0.1 * fmin(0.0, FOURTH * (d1 + d2 + d3 + d4));
#pragma unroll
        for (int n = 0; n <= UEINT; ++n) v.d[n] = ur[n] - ul[n];
        return v;
    };
    auto put_face = [&](double (*S)[ND], const FaceH &f) {
        S[0][at] = f.rho;
        S[1][at] = f.un;
        S[2][at] = f.ut;
        S[3][at] = f.utt;
        S[4][at] = f.p;
        S[5][at] = f.rhoe;
    };
    auto get_face = [&](double (*S)[ND], int q) -> FaceH {
        return FaceH{S[0][q], S[1][q], S[2][q], S[3][q], S[4][q], S[5][q]};
    };
    auto put_flux = [&](double (*S)[ND], const TFlux &f) {
#pragma unroll
        for (int n = 0; n <= UEDEN; ++n) S[n][at] = f.f[n];
        S[5][at] = f.gp;
        S[6][at] = f.gu;
    };
    auto get_flux = [&](double (*S)[ND], int q) -> TFlux {
        TFlux o;
#pragma unroll
        for (int n = 0; n <= UEDEN; ++n) o.f[n] = S[n][q];
        o.gp = S[5][q];
        o.gu = S[6][q];
        return o;
    };
    const double dt = uniform_d(x.dt_cur[m]), dx0 = I.dx[0], dx1 = I.dx[1], dx2 = I.dx[2];
    const double rx = dt / dx0, ry = dt / dx1, rz = dt / dx2;
    const double cx = uniform_d(rx / 3.0), cy = uniform_d(ry / 3.0), cz = uniform_d(rz / 3.0);
    const double hx = uniform_d(0.5 * dt / dx0), hy = uniform_d(0.5 * dt / dx1), hz = uniform_d(0.5 * dt / dx2);
    // faces the thread stores: the tile's, and the ring's where the instance ends
    const bool inr = ((tx >= 1 && tx <= w) || iu == -1 || (iu == n0 && tx == w + 1)) &&
                     ((ty >= 1 && ty <= h) || ju == -1 || (ju == n1 && ty == h + 1));
    const bool col = tx >= 1 && tx <= w && ty >= 1 && ty <= h;
    const bool st_x = ty >= 1 && ty <= h && ((tx >= 1 && tx <= w) || (tx == w + 1 && iu == n0));
    const bool st_y = tx >= 1 && tx <= w && ((ty >= 1 && ty <= h) || (ty == h + 1 && ju == n1));

    // read ahead of the plane's other loads: the x-fluxes and y-states; carried
    // from plane to plane: the minus state of z-face p corrected by x,
    // by y and by both, F^{z|x} and F^{z|y} on z-face p - 1, c and Gamma_1 of the
    // cell and of its y-neighbour on plane p - 1
    FaceH zmx{}, zmy{}, zmz{};
    TFlux fzx{}, fzy{};
    double ck = 1.0, gk = 1.0, cky = 1.0, gky = 1.0;
    int p = zc0 - 1;
    idx_t e = (idx_t)(i + 1) + (idx_t)ex0 * ((idx_t)(j + 1) + (idx_t)I.ext[1] * (idx_t)(p - I.zlo + 1));
    TFlux nf = flux(F0, e);
    QInH nyl = state(M1, e + oy), nyr = state(P1, e);
    idx_t czk = cs * (idx_t)plane_w(I, p);
    for (; p <= zc1; ++p, e += es) {
        const bool top = p >= ztop, bot = p < I.zlo;
        auto ep = [&]() -> idx_t { return top ? e : e + es; };  // plane p + 1 (not read above the ring)
        auto ek = [&]() -> idx_t { return bot ? e : e - es; };  // plane p - 1
        const bool put = inr && ((p >= zc0 && p < zc1) || bot || top), putk = inr && p > zc0;
        const idx_t cz_ = cs * (idx_t)plane_w(I, p);
        const double cp = QC[cxy + cz_], gp = QG[cxy + cz_], cpy = QC[cym + cz_], gpy = QG[cym + cz_];
        dbl2 rw;
        FaceH yp1, yp2;
        TDiff dzx, dxz, dzy, dxy;
        QInH z_r, z_l;
        {  // corrections by the x-fluxes: y and z states of plane p
            z_r = state(P2, e);
            z_l = state(M2, ep());
            TDiff D = tdiff(lane_above(nf), nf, gp);
            finish(e, D);
            put_face(A[0], correct1<1>(nyl, D, cx));
            yp1 = correct1<1>(nyr, D, cx);
            finish(e, yp1);
            const FaceH r = correct1<2>(z_r, D, cx);
            TFlux t = tflux<2>(zmx, r, ck, cp, gk, gp, rw);
            if (put) TZX[e] = rw;
            dzx = tdiff(t, fzx, gk);
            fzx = t;
            finish(e, dzx);
            zmx = correct1<2>(z_l, D, cx);
            finish(e, zmx);
        }
        {  // by the y-fluxes: x and z states of plane p
            const TFlux f = flux(F1, e + oy), f0 = flux(F1, e);
            const QInH xl = state(M0, e + ox), xr = state(P0, e);
            TDiff D = tdiff(f, f0, gp);
            finish(e, D);
            const FaceH r = correct1<2>(z_r, D, cy);
            TFlux t = tflux<2>(zmy, r, ck, cp, gk, gp, rw);
            if (put) TZY[e] = rw;
            dzy = tdiff(t, fzy, gk);
            fzy = t;
            finish(e, dzy);
            zmy = correct1<2>(z_l, D, cy);
            finish(e, zmy);
            const FaceH l = lane_shift<true>(correct1<0>(xl, D, cy));
            const FaceH rr = correct1<0>(xr, D, cy);
            const TFlux u = tflux<0>(l, rr, lane_shift<true>(cp), cp, lane_shift<true>(gp), gp, rw);
            if (put) TXY[e] = rw;
            dxy = tdiff(lane_above(u), u, gp);
            finish(e, dxy);
        }
        const QInH kyl = state(M1, ek() + oy), kyr = state(P1, ek()), kxl = state(M0, ek() + ox), kxr = state(P0, ek());
        {  // by the z-fluxes: x and y states of plane p - 1
            TDiff D = tdiff(flux(F2, e), flux(F2, ek()), gk);
            finish(e, D);
            put_face(A[1], correct1<1>(kyl, D, cz));
            yp2 = correct1<1>(kyr, D, cz);
            finish(e, yp2);
            const FaceH l = lane_shift<true>(correct1<0>(kxl, D, cz));
            const FaceH r = correct1<0>(kxr, D, cz);
            const TFlux t = tflux<0>(l, r, lane_shift<true>(ck), ck, lane_shift<true>(gk), gk, rw);
            if (putk) TXZ[ek()] = rw;
            dxz = tdiff(lane_above(t), t, gk);
            finish(e, dxz);
        }
        __syncthreads();
        TFlux fyx = tflux<1>(get_face(A[0], at - TX), yp1, cpy, cp, gpy, gp, rw);
        if (put) TYX[e] = rw;
        put_flux(B[0], fyx);
        finish(e, fyx);
        TFlux fyz = tflux<1>(get_face(A[1], at - TX), yp2, cky, ck, gky, gk, rw);
        if (putk) TYZ[ek()] = rw;
        put_flux(B[1], fyz);
        finish(e, fyz);
        __syncthreads();
        // two-direction corrections and final fluxes: y states of plane p - 1
        double uk[UEINT + 1], up[UEINT + 1], un[UEINT + 1];
        const QInH kx2l = state(M0, ek() + ox), kx2r = state(P0, ek());
        put_face(A[2], correct2<1>(kyl, dxz, hx, dzx, hz));
        FaceH ypp = correct2<1>(kyr, dxz, hx, dzx, hz);
        finish(e, ypp);
        RiemannH o;
        const QInH zr2 = state(P2, e), zl2 = state(M2, ep());
        zone(cxy + czk, uk);
        double d00 = DV[ek()], d01 = DV[ek() + oy], d0p = DV[e];
        {  // x
            TDiff dyz = tdiff(get_flux(B[1], at + TX), fyz, gk);
            finish(e, dyz);
            const FaceH l = lane_shift<true>(correct2<0>(kx2l, dyz, hy, dzy, hz));
            const FaceH r = correct2<0>(kx2r, dyz, hy, dzy, hz);
            riemann_hydro(l, r, lane_shift<true>(ck), ck, lane_shift<true>(gk), gk, o);
#pragma unroll
            for (int n = 0; n <= UEINT; ++n) up[n] = lane_shift<true>(uk[n]);
            if (p > zc0 && st_x) final_hydro(x, I, 0, ek(), o, av(d00, d01, d0p, d01, uk, up));
        }
        zone(cxy + cz_, up);
        double d10 = DV[e + ox], d02 = DV[e + oy], d11 = DV[e + ox + oy];
        {  // z
            TDiff dyx = tdiff(get_flux(B[0], at + TX), fyx, gp);
            finish(e, dyx);
            const FaceH r = correct2<2>(zr2, dxy, hx, dyx, hy);
            riemann_hydro(zmz, r, ck, cp, gk, gp, o);
            if (col && p >= zc0 && (p < zc1 || zc1 == ztop))
                final_hydro(x, I, 2, e, o, av(d0p, d10, d02, d11, up, uk));
            zmz = correct2<2>(zl2, dxy, hx, dyx, hy);
            finish(e, zmz);
        }
        zone(cym + czk, un);
        d10 = DV[ek() + ox];
        nf = flux(F0, ep());
        nyl = state(M1, ep() + oy), nyr = state(P1, ep());
        __syncthreads();
        riemann_hydro(get_face(A[2], at - TX), ypp, cky, ck, gky, gk, o);
        if (p > zc0 && st_y) final_hydro(x, I, 1, ek(), o, av(d00, d10, d0p, d10, uk, un));
        czk = cz_;
        ck = cp;
        gk = gp;
        cky = cpy;
        gky = gpy;
    }
}

} // namespace mc
