// sph_learned.h -- the FP64 stages of the steps inside a learned run (coarse
// steps, judges, recorded targets), in an arithmetic of their own.
//
// A learned run rounds its state to FP32 records (mixed precision), its rates to
// FP32 features and the network's operands to BF16 in every advance.  A last-bit
// difference in an FP64 sum is a difference of FP32 size from the first of those
// roundings that it flips, and all later advances carry it on: with the pair
// terms of sph_fused.h in its place (equal to these to 1e-13 after 40 steps) a
// rollout of the 250k slope parted by 1.0e-8 in the velocities.  So the roundings
// here are part of what a learned run computes, and stay as they are:
//   - each term as written below, from the records' rho, m, vof and p (the packs
//     write these instead of V and vof / rho under KParams.learned);
//   - one lane per particle, partners in the order of its candidates;
//   - 1/d and 1/sqrt(d) from two Newton steps each;
//   - d^2 of a pair by dist2.
// Where the partners are read from (window, global memory, candidate rows) does
// not show in the results.  The windows are those of sph_fused.h; a listed
// candidate outside the support is skipped.
#pragma once
#include "sph_fused.h"

namespace learned {

__device__ __forceinline__ double rcp(double d)
{
    double x = __builtin_amdgcn_rcp(d);
    double e = fma(-d, x, 1.0);
    x = fma(x, e, x);
    e = fma(-d, x, 1.0);
    return fma(x, e, x);
}

__device__ __forceinline__ double rsq(double d)
{
    double y = __builtin_amdgcn_rsq(d);
    const double h = 0.5 * d;
    y = y * fma(-h, y * y, 1.5);
    y = y * fma(-h, y * y, 1.5);
    return y;
}

// The constants of a smoothing length.
struct KL {
    double inv_h, f, fh1, fh2;
};

__device__ __forceinline__ KL make_kl(int skf, double h)
{
    KL k;
    k.inv_h = 1.0 / h;
    double f;
    if (skf == 1) f = 15.0 / (7.0 * SPH_PI_F * h * h);
    else if (skf == 2) f = 1.0 / ((h * h) * SPH_PI_F);
    else if (skf == 3) f = 7.0 / (478.0 * SPH_PI_F * h * h);
    else f = 7.0 / (4.0 * SPH_PI_F * h * h);
    k.f = f;
    k.fh1 = f * k.inv_h;
    k.fh2 = f * k.inv_h * k.inv_h;
    return k;
}

// W and grad W of a pair (m_particles.f90:1469-1602); inv_r = 1/r.
template <int SKF, bool NEED_W>
__device__ __forceinline__ void kern(const KL& k, double r, double inv_r, double dx, double dy, double& w, double& gx,
                                     double& gy)
{
    const double q = r * k.inv_h;
    w = 0.0; gx = 0.0; gy = 0.0;
    if constexpr (SKF == 1) {
        const bool in1 = q <= 1.0, in2 = q <= 2.0;
        const double t = 2.0 - q;
        const double s1 = k.fh2 * (-2.0 + 1.5 * q);
        const double s2 = -(0.5 * k.fh1) * (t * t) * inv_r;
        const double s = in1 ? s1 : (in2 ? s2 : 0.0);
        if (NEED_W) {
            const double w1 = k.f * (SPH_C23_F - q * q + ((q * q) * q) * 0.5);
            const double w2 = k.f * (1.0 / 6.0) * ((t * t) * t);
            w = in1 ? w1 : (in2 ? w2 : 0.0);
        }
        gx = s * dx; gy = s * dy;
    } else if constexpr (SKF == 4) {
        const bool in2 = q <= 2.0;
        const double t = 1.0 - 0.5 * q;
        const double t2 = t * t;
        if (NEED_W) w = in2 ? k.f * ((t2 * t2) * (1.0 + 2.0 * q)) : 0.0;
        double s = k.fh2 * (-5.0 + 7.5 * q - 3.75 * (q * q) + 0.625 * ((q * q) * q));
        s = in2 ? s : 0.0;
        gx = s * dx; gy = s * dy;
    } else if constexpr (SKF == 2) {
        if (q <= 3.0) {
            const double e = k.f * exp(-q * q);
            if (NEED_W) w = e;
            const double s = -2.0 * e * (k.inv_h * k.inv_h);
            gx = s * dx; gy = s * dy;
        }
    } else {
        const double a = 3.0 - q, b = 2.0 - q, c = 1.0 - q;
        const double a2 = a * a, b2 = b * b, c2 = c * c;
        const double a4 = a2 * a2, b4 = b2 * b2, c4 = c2 * c2;
        if (q <= 1.0) {
            if (NEED_W) w = k.f * (a4 * a - 6.0 * (b4 * b) + 15.0 * (c4 * c));
            const double s = k.fh2 * (-120.0 + 120.0 * q - 50.0 * (q * q));
            gx = s * dx; gy = s * dy;
        } else if (q <= 2.0) {
            if (NEED_W) w = k.f * (a4 * a - 6.0 * (b4 * b));
            const double s = k.fh1 * (-(5.0 * a4) + 30.0 * b4) * inv_r;
            gx = s * dx; gy = s * dy;
        } else if (q <= 3.0) {
            if (NEED_W) w = k.f * (a4 * a);
            const double s = k.fh1 * (-(5.0 * a4)) * inv_r;
            gx = s * dx; gy = s * dy;
        }
    }
}

// Whether a listed candidate lies outside the support (U; the other paths have
// tested theirs): the exact predicate of a uniform smoothing length.
template <bool U>
__device__ __forceinline__ bool outside(double dx, double dy, double thr)
{
#pragma clang fp contract(off)
    return U && !(dx * dx + dy * dy < thr);
}

// d^2 of a pair's terms (written out: the contraction is the same in every
// kernel).  A crowded particle takes the predicate's, with both products rounded.
__device__ __forceinline__ double dist2(double dx, double dy, bool crowded)
{
#pragma clang fp contract(off)
    return crowded ? dx * dx + dy * dy : fma(dx, dx, dy * dy);
}

// More than 64 candidates in a row of cells or more than 128 in all.
__device__ __forceinline__ bool crowded(const Cand& C, int tt)
{
    int tot;
    const Ranges3 r = C.rows(tt, tot);
    return tot > 128 || r.s1 > 64 || r.s2 - r.s1 > 64 || tot - r.s2 > 64;
}

// repulsive_force's factor on a real particle from a virtual one (m_particles.f90:1605).
template <bool U>
__device__ __forceinline__ double rep_factor(const KParams& K, double dspp, double r, double idr)
{
    const double q = dspp / r;
    return (U ? ipow(q, K.ip1) - ipow(q, K.ip2) : pow(q, K.p1) - pow(q, K.p2)) * idr;
}

// The stages: the terms, inputs and outputs of the same stages of sph_fused.h.
template <int SKF, bool U>
__device__ __forceinline__ void water_x(unsigned char* lds, int blk, DPhase W, DPhase S, const double* recW,
                                        const double* recS, NList NL, Grid g, KParams K, FusedK F)
{
    const RecV RW = recv(recW, W.n), RS = recv(recS, S.n);
    const SubCtx wc = sub_ctx(W.n, blk, 0, lanes_of_one(NL.ix));
    const double2 xy = RW(wc.tt, 0), va = RW(wc.tt, 1), rm = RW(wc.tt, 2);
    const double xa = xy.x, ya = xy.y, vxa = va.x, vya = va.y, rhoa = rm.x, vofa = RW(wc.tt, 3).x;
    const double ha = U ? K.h1_water : RW(wc.tt, 6).x;
    const double irhoa = 1.0 / rhoa;
    const int a = W.order[wc.tt];
    const bool ux = U || F.uni_x;
    const Window win = open_window<U, 4>(lds, NL.ix, blk, wc, 0, W.n, RS);
    const Cand C{g, S.cell_start, NL.cell, xa, ya};
    const bool many = crowded(C, wc.tt);
    const Pred PX{xa, ya, ha, F.thr_x, ux ? 1 : 0, 0};
    const double cfa = vofa * rhoa * (-K.numeric_gravity) / K.s_perm;
    const KL kx = make_kl(SKF, sph_mhsml(ha, ux ? RS(0, 6).x : ha));
    double dg_x = 0.0, dg_y = 0.0, dvof_x = 0.0, vof2 = 0.0;
    int cntx = 0;
    visit<U, 4>(
        lds, win, C, NL.ix, W.n, wc, 0, -1, RS, NL.cross, [&](int k, double2 b) { return PX(b, ux ? ha : RS(k, 6).x, g, K); },
        [&](const auto& v, const auto& R, int k) {
            const double dx = xa - v[0].x, dy = ya - v[0].y;
            if (outside<U>(dx, dy, F.thr_x)) return;
            const double dr = dist2(dx, dy, many);
            const double ir = (dr > 0.0) ? rsq(dr) : 0.0;
            const double r = dr * ir;
            double ww, gx, gy;
            if (ux) kern<SKF, true>(kx, r, ir, dx, dy, ww, gx, gy);
            else kern<SKF, true>(make_kl(SKF, sph_mhsml(ha, R(k, 6).x)), r, ir, dx, dy, ww, gx, gy);
            ++cntx;
            const double mb = fabs(v[2].y), irb = rcp(v[2].x);
            const double dvx = vxa - v[1].x, dvy = vya - v[1].y;
            const double sc = mb * (cfa * v[3].x) * (ww * irhoa * irb);
            dg_x += sc * dvx;
            dg_y += sc * dvy;
            dvof_x += mb * (dvx * gx + dvy * gy);
            vof2 += mb * ww;
        });
    if (!wc.valid) return;
    W.drgx[a] = dg_x;
    W.drgy[a] = dg_y;
    W.dvof_x[a] = dvof_x * (1.0 / K.s_rho0);
    W.vof2[a] = 1.0 - vof2 / K.s_rho0;
    W.countiac[a] = cntx;
}

template <int SKF, bool U>
__device__ __forceinline__ void soil_x(unsigned char* lds, int blk, DPhase S, DPhase W, const double* recS,
                                       const double* recW, NList NL, Grid g, KParams K, FusedK F)
{
    const RecV RS = recv(recS, S.n), RW = recv(recW, W.n);
    const SubCtx wc = sub_ctx(S.n, blk, 0, lanes_of_one(NL.ix));
    const double2 xy = RS(wc.tt, 0), va = RS(wc.tt, 1), rm = RS(wc.tt, 2);
    const double xa = xy.x, ya = xy.y, vxa = va.x, vya = va.y, rhoa = rm.x, vofa = RS(wc.tt, 3).x;
    const double ha = U ? K.h1_soil : RS(wc.tt, 6).x;
    const double irhoa = 1.0 / rhoa;
    const int a = S.order[wc.tt];
    const bool ux = U || F.uni_x;
    const Window win = open_window<U, 4>(lds, NL.ix, blk, wc, 0, S.n, RW);
    const Cand C{g, W.cell_start, NL.cell, xa, ya};
    const Pred PX{xa, ya, ha, F.thr_x, ux ? 1 : 0, 0};
    const double cfs = vofa * (-K.numeric_gravity) / K.s_perm;
    const KL kx = make_kl(SKF, sph_mhsml(ux ? RW(0, 6).x : ha, ha));
    double dg_x = 0.0, dg_y = 0.0, po_x = 0.0, po_y = 0.0;
    int cntx = 0;
    visit<U, 4>(
        lds, win, C, NL.ix, S.n, wc, 0, -1, RW, NL.cross, [&](int k, double2 b) { return PX(b, ux ? ha : RW(k, 6).x, g, K); },
        [&](const auto& v, const auto& R, int k) {
            const double dx = v[0].x - xa, dy = v[0].y - ya;   // water - soil
            if (outside<U>(dx, dy, F.thr_x)) return;
            const double dr = dist2(dx, dy, false);
            const double ir = (dr > 0.0) ? rsq(dr) : 0.0;
            const double r = dr * ir;
            double ww, gx, gy;
            if (ux) kern<SKF, true>(kx, r, ir, dx, dy, ww, gx, gy);
            else kern<SKF, true>(make_kl(SKF, sph_mhsml(R(k, 6).x, ha)), r, ir, dx, dy, ww, gx, gy);
            ++cntx;
            const double mw = fabs(v[2].y), rhow = v[2].x, irb = rcp(v[2].x);
            const double sc = mw * (v[3].x * rhow * cfs) * (ww * irb * irhoa);
            dg_x += sc * (v[1].x - vxa);
            dg_y += sc * (v[1].y - vya);
            const double mprr = mw * v[3].y * (irb * irhoa);
            po_x += mprr * gx;
            po_y += mprr * gy;
        });
    if (!wc.valid) return;
    S.drgx[a] = dg_x;
    S.drgy[a] = dg_y;
    S.porx[a] = vofa * po_x;
    S.pory[a] = vofa * po_y;
    S.countiac[a] = cntx;
}

template <int SKF, bool U>
__device__ __forceinline__ void water_a(unsigned char* lds, int blk, DPhase W, const double* recW, double* recWw,
                                        NList NL, Grid g, KParams K, FusedK F)
{
    const RecV RW = recv(recW, W.n);
    const SubCtx wc = sub_ctx(W.n, blk, 0, lanes_of_one(NL.is));
    const int t = wc.t;
    auto RA = [&](int c) { return RW(wc.tt, c); };
    const double2 xy = RA(0), va = RA(1), rm = RA(2), hi = RA(6);
    const bool link = K.nnps == 2;
    const double xa = xy.x, ya = xy.y, vxa = va.x, vya = va.y, rhoa = rm.x, vofa = RA(3).x;
    const double ha = U ? K.h1_water : hi.x;
    const int ita = (int)hi.y;
    const int a = W.order[wc.tt];
    const double ca = W.c[a];
    const bool uni = U || link || F.uni_w;
    const KL kc = make_kl(SKF, link ? K.h1_water : ha);
    const Window win = open_window<U, 3>(lds, NL.is, blk, wc, 0, W.n, RW);
    const Cand C{g, W.cell_start, NL.cell, xa, ya};
    const bool many = crowded(C, wc.tt);
    const Pred P{xa, ya, ha, F.thr_w, uni ? 1 : 0, link ? 1 : 0};
    double con = 0.0, drd = 0.0, txx = 0.0, txy = 0.0, tyy = 0.0, avx = 0.0, avy = 0.0, repx = 0.0, repy = 0.0;
    int cnt = 0;
    visit<U, 3>(
        lds, win, C, NL.is, W.n, wc, 0, t, RW, NL.same, [&](int k, double2 b) { return P(b, uni ? ha : RW(k, 6).x, g, K); },
        [&](const auto& v, const auto& R, int k) {
            const double dx = xa - v[0].x, dy = ya - v[0].y;
            if (outside<U>(dx, dy, F.thr_w)) return;
            const double dr = dist2(dx, dy, many);
            const double ir = rsq(dr), r = dr * ir, idr = ir * ir;
            double ww, gx, gy;
            if (uni) kern<SKF, true>(kc, r, ir, dx, dy, ww, gx, gy);
            else kern<SKF, true>(make_kl(SKF, sph_mhsml(ha, R(k, 6).x)), r, ir, dx, dy, ww, gx, gy);
            ++cnt;
            const double mb = fabs(v[2].y), irb = rcp(v[2].x), Vb = mb * irb;
            const double dvx = vxa - v[1].x, dvy = vya - v[1].y;
            con += mb * (dvx * gx + dvy * gy);
            drd += mb * (2.0 * (rhoa - v[2].x) * idr * (dx * gx + dy * gy)) * irb;
            txx += Vb * (-2.0 * dvx * gx + dvy * gy);
            txy += Vb * (-(dvx * gy) - dvy * gx);
            tyy += Vb * (-2.0 * dvy * gy + dvx * gx);
            const double f = mb * ww * (2.0 * rcp(rhoa + v[2].x));
            avx -= dvx * f;
            avy -= dvy * f;
            if (ita > 0 && !(r > W.dspp) && (uni ? v[2].y : R(k, 6).y) < 0.0) {
                const double fr = rep_factor<U>(K, W.dspp, r, idr);
                repx += K.dd * dx * fr;
                repy += K.dd * dy * fr;
            }
        });
    if (!wc.valid) return;
    const double mu = K.w_mu;
    txx *= SPH_C23_F;
    tyy *= SPH_C23_F;
    W.drho[a] = K.artificial_density ? con + (K.delta * ha * ca) * drd : con;
    W.txx[a] = txx; W.txy[a] = txy; W.tyy[a] = tyy;
    if (ita > 0) { avx *= K.epsilon; avy *= K.epsilon; }
    if (K.average_velocity) { W.avx[a] = avx; W.avy[a] = avy; }
    W.repx[a] = repx; W.repy[a] = repy;
    W.nsame[a] = cnt;
    double2* WP = reinterpret_cast<double2*>(recWw) + t;
    const size_t nw = (size_t)W.n;
    reinterpret_cast<double*>(WP + 4 * nw)[0] = vofa * (mu * tyy);
    WP[5 * nw] = make_double2(vofa * (mu * txx), vofa * (mu * txy));
}

template <int SKF, bool U>
__device__ __forceinline__ void water_b(unsigned char* lds, int blk, DPhase W, const double* recW, NList NL, Grid g,
                                        KParams K, FusedK F, int mask)
{
    const RecV RW = recv(recW, W.n);
    const SubCtx wc = sub_ctx(W.n, blk, 0, lanes_of_one(NL.is));
    const int t = wc.t;
    auto RA = [&](int c) { return RW(wc.tt, c); };
    const double2 axy = RA(0), av = RA(1), arm = RA(2), a3 = RA(3), apc = RA(4), a12 = RA(5);
    const double xa = axy.x, ya = axy.y, vxa = av.x, vya = av.y, rhoa = arm.x, vofa = a3.x;
    const double ha = U ? K.h1_water : RA(6).x;
    const double pa = a3.y, ca = apc.y, fxx_a = a12.x, fxy_a = a12.y, fyy_a = apc.x;
    const double irhoa = 1.0 / rhoa;
    const int a = W.order[wc.tt];
    const bool link = K.nnps == 2;
    const bool uni = U || link || F.uni_w;
    const KL kc = make_kl(SKF, link ? K.h1_water : ha);
    const Window win = open_window<U, 6>(lds, NL.is, blk, wc, 0, W.n, RW);
    const Cand C{g, W.cell_start, NL.cell, xa, ya};
    const bool many = crowded(C, wc.tt);
    const Pred P{xa, ya, ha, F.thr_w, uni ? 1 : 0, link ? 1 : 0};
    const double et2 = K.etq * K.etq;
    double Px = 0.0, Py = 0.0, Sxx = 0.0, Sxyy = 0.0, Sxyx = 0.0, Syy = 0.0;
    double artx = 0.0, arty = 0.0, dvd = 0.0;
    visit<U, 6>(
        lds, win, C, NL.is, W.n, wc, 0, t, RW, NL.same, [&](int k, double2 b) { return P(b, uni ? ha : RW(k, 6).x, g, K); },
        [&](const auto& v, const auto& R, int k) {
            const double dx = xa - v[0].x, dy = ya - v[0].y;
            if (outside<U>(dx, dy, F.thr_w)) return;
            const double dr = dist2(dx, dy, many);
            const double ir = rsq(dr), r = dr * ir, idr = ir * ir;
            double ww, gx, gy;
            const double amh = uni ? ha : sph_mhsml(ha, R(k, 6).x);
            if (uni) kern<SKF, false>(kc, r, ir, dx, dy, ww, gx, gy);
            else kern<SKF, false>(make_kl(SKF, amh), r, ir, dx, dy, ww, gx, gy);
            const double mb = fabs(v[2].y), irb = rcp(v[2].x), Vb = mb * irb;
            const double ps = pa + v[3].y;
            Px += Vb * (ps * gx);
            Py += Vb * (ps * gy);
            const double sxy = fxy_a + v[5].y;
            Sxx += Vb * ((fxx_a + v[5].x) * gx);
            Sxyy += Vb * (sxy * gy);
            Sxyx += Vb * (sxy * gx);
            Syy += Vb * ((fyy_a + v[4].x) * gy);
            const double vr = (vxa - v[1].x) * dx + (vya - v[1].y) * dy;
            {   // art_visc: approaching pairs only (vr < 0)
                const double muv = amh * vr * rcp(dr + amh * amh * et2);
                const double mc = 0.5 * (ca + v[4].y);
                double piv = (K.beta * muv - K.alpha * mc) * muv * (2.0 * rcp(rhoa + v[2].x));
                piv = vr < 0.0 ? piv : 0.0;
                artx -= mb * piv * gx;
                arty -= mb * piv * gy;
            }
            dvd += mb * (2.0 * (vofa - v[3].x) * idr * (dx * gx + dy * gy)) * irb;
        });
    if (!wc.valid) return;
    double ax = -(vofa * Px) + Sxx + Sxyy;
    double ay = -(vofa * Py) + Sxyx + Syy;
    if (rhoa > 0.0) {
        ax = ax * irhoa;
        ay = ay * irhoa;
    }
    if (mask & M_ART) { ax = ax + artx; ay = ay + arty; }
    ax = ax + W.repx[a];
    ay = ay + W.repy[a];
    ay = ay + K.gravity;
    double dvof = (mask & M_DELTA_FIELD) ? (K.delta * ha * ca) * dvd : 0.0;
    if (mask & M_CROSS) {
        ax = ax - W.drgx[a];
        ay = ay - W.drgy[a];
        dvof = dvof - W.dvof_x[a];
    }
    W.ax[a] = ax;
    W.ay[a] = ay;
    W.dvof[a] = dvof;
}

template <int SKF, bool U>
__device__ __forceinline__ void soil_ab(unsigned char* lds, int blk, DPhase S, const double* recS, NList NL, Grid g,
                                        KParams K, FusedK F, int mask)
{
    const RecV RS = recv(recS, S.n);
    const SubCtx wc = sub_ctx(S.n, blk, 0, lanes_of_one(NL.is));
    const int t = wc.t;
    auto RA = [&](int c) { return RS(wc.tt, c); };
    const double2 xy = RA(0), va = RA(1), rm = RA(2), a3 = RA(3), a4 = RA(4), a12 = RA(5), hi = RA(6);
    const double xa = xy.x, ya = xy.y, vxa = va.x, vya = va.y, rhoa = rm.x, vofa = a3.x;
    const double ha = U ? K.h1_soil : hi.x;
    const double pa = a3.y, sxxa = a12.x, sxya = a12.y, syya = a4.x;
    const double ca = a4.y;          // sound speed before this step (delta_sph of rho)
    const double cn = K.s_c;         // sound speed after it (stage B)
    const double irhoa = 1.0 / rhoa, ir2a = irhoa * irhoa;
    const bool mc = !U && K.yield_criterion == 1;
    const double rhoa_pre = mc ? RA(7).x : rhoa;
    const double fpa = vofa * pa * ir2a, fxxa = vofa * sxxa * ir2a, fxya = vofa * sxya * ir2a,
                 fyya = vofa * syya * ir2a;
    const int ita = (int)hi.y;
    const int a = S.order[wc.tt];
    const bool link = K.nnps == 2;
    const bool uni = U || link || F.uni_s;
    const KL kc = make_kl(SKF, link ? K.h1_soil : ha);
    const Window win = open_window<U, 6>(lds, NL.is, blk, wc, 0, S.n, RS);
    const Cand C{g, S.cell_start, NL.cell, xa, ya};
    const bool many = crowded(C, wc.tt);
    const Pred P{xa, ya, ha, F.thr_s, uni ? 1 : 0, link ? 1 : 0};
    const double et2 = K.etq * K.etq;
    double con = 0.0, drd = 0.0, txx = 0.0, txy = 0.0, tyy = 0.0, vcc = 0.0, wxy = 0.0;
    double avx = 0.0, avy = 0.0, repx = 0.0, repy = 0.0;
    double Fx = 0.0, Fy = 0.0;
    double artx = 0.0, arty = 0.0, dP = 0.0, dXX = 0.0, dXY = 0.0, dYY = 0.0;
    int cnt = 0;
    visit<U, 6>(
        lds, win, C, NL.is, S.n, wc, 0, t, RS, NL.same, [&](int k, double2 b) { return P(b, uni ? ha : RS(k, 6).x, g, K); },
        [&](const auto& v, const auto& R, int k) {
            const double dx = xa - v[0].x, dy = ya - v[0].y;
            if (outside<U>(dx, dy, F.thr_s)) return;
            const double dr = dist2(dx, dy, many);
            const double ir = rsq(dr), r = dr * ir, idr = ir * ir;
            double ww, gx, gy;
            const double amh = uni ? ha : sph_mhsml(ha, R(k, 6).x);
            if (uni) kern<SKF, true>(kc, r, ir, dx, dy, ww, gx, gy);
            else kern<SKF, true>(make_kl(SKF, amh), r, ir, dx, dy, ww, gx, gy);
            ++cnt;
            const double mb = fabs(v[2].y), irb = rcp(v[2].x), Vb = mb * irb;
            // stage A
            const double dvx = vxa - v[1].x, dvy = vya - v[1].y;
            const double dvg = dvx * gx + dvy * gy;
            const double rb_pre = mc ? R(k, 7).x : v[2].x;
            const double irb_pre = mc ? rcp(rb_pre) : irb;
            const double Vb_pre = mc ? mb * irb_pre : Vb;
            con += mb * dvg;
            drd += mb * (2.0 * (rhoa_pre - rb_pre) * idr * (dx * gx + dy * gy)) * irb_pre;
            txx += Vb_pre * (-2.0 * dvx * gx + dvy * gy);
            txy += Vb_pre * (-(dvx * gy) - dvy * gx);
            tyy += Vb_pre * (-2.0 * dvy * gy + dvx * gx);
            vcc -= Vb_pre * dvg;
            wxy += Vb * (-(dvx * gy) + dvy * gx);
            const double f = mb * ww * (2.0 * rcp(rhoa + v[2].x));
            avx -= dvx * f;
            avy -= dvy * f;
            if (ita > 0 && !(r > S.dspp) && (uni ? v[2].y : R(k, 6).y) < 0.0) {
                const double fr = rep_factor<U>(K, S.dspp, r, idr);
                repx += K.dd * dx * fr;
                repy += K.dd * dy * fr;
            }
            // stage B
            const double vofb = v[3].x, ir2b = irb * irb;
            const double fp = fpa + vofb * v[3].y * ir2b;
            const double fxx = fxxa + vofb * v[5].x * ir2b;
            const double fxy = fxya + vofb * v[5].y * ir2b;
            const double fyy = fyya + vofb * v[4].x * ir2b;
            Fx += mb * ((fxx - fp) * gx + fxy * gy);
            Fy += mb * ((fyy - fp) * gy + fxy * gx);
            const double vr = dvx * dx + dvy * dy;
            {   // art_visc: approaching pairs only (vr < 0)
                const double muv = amh * vr * rcp(dr + amh * amh * et2);
                double piv = (K.beta * muv - K.alpha * cn) * muv * (2.0 * rcp(rhoa + v[2].x));
                piv = vr < 0.0 ? piv : 0.0;
                artx -= mb * piv * gx;
                arty -= mb * piv * gy;
            }
            const double hh = 2.0 * idr * (dx * gx + dy * gy) * mb * irb;
            dP += hh * (pa - v[3].y);
            dXX += hh * (sxxa - v[5].x);
            dXY += hh * (sxya - v[5].y);
            dYY += hh * (syya - v[4].x);
        });
    if (!wc.valid) return;
    txx *= SPH_C23_F;
    tyy *= SPH_C23_F;
    wxy *= 0.5;
    S.drho[a] = K.artificial_density ? con + (K.delta * ha * ca) * drd : con;
    S.txx[a] = txx; S.txy[a] = txy; S.tyy[a] = tyy; S.vcc[a] = vcc; S.wxy[a] = wxy;
    if (ita > 0) { avx *= K.epsilon; avy *= K.epsilon; }
    if (K.average_velocity) { S.avx[a] = avx; S.avy[a] = avy; }
    S.nsame[a] = cnt;
    S.c_next[a] = cn;
    StressRates d = stress_rates(S, K, a, txx, txy, tyy, vcc, wxy, pa, sxxa, sxya, syya);
    double ax = Fx * rhoa;
    double ay = Fy * rhoa;
    if (rhoa > 0.0) { ax = ax * irhoa; ay = ay * irhoa; }
    if (mask & M_ART) { ax = ax + artx; ay = ay + arty; }
    ax = ax + repx;
    ay = ay + repy;
    ay = ay + K.gravity;
    if (mask & M_CROSS) {
        ax = ax + S.drgx[a]; ay = ay + S.drgy[a];
        ax = ax + S.porx[a]; ay = ay + S.pory[a];
    }
    if (mask & M_DELTA_FIELD) {
        const double cf = K.delta * ha * cn;
        d.p = d.p + cf * dP;
        d.xx = d.xx + cf * dXX;
        d.xy = d.xy + cf * dXY;
        d.yy = d.yy + cf * dYY;
    }
    S.dsxx[a] = d.xx; S.dsxy[a] = d.xy; S.dsyy[a] = d.yy; S.dp[a] = d.p;
    S.ax[a] = ax;
    S.ay[a] = ay;
}

// One part of a step (0 soil_x, 1 water_a, 2 water_x; 3 soil_ab, 4 water_b).  U as
// in sph_fused.h: the phase (of the cross pairs: both phases) uniform in h, and for
// the same-phase parts integer repulsion exponents and, for the soil,
// Drucker-Prager.
template <int SKF, int PART, bool U>
__device__ __forceinline__ void part(unsigned char* lds, int blk, const StageArgs& A)
{
    if constexpr (PART == 0) soil_x<SKF, U>(lds, blk, A.S, A.W, A.rS, A.rW, A.nS, A.gS, A.K, A.F);
    if constexpr (PART == 1) water_a<SKF, U>(lds, blk, A.W, A.rW, A.rW, A.nW, A.gW, A.K, A.F);
    if constexpr (PART == 2) water_x<SKF, U>(lds, blk, A.W, A.S, A.rW, A.rS, A.nW, A.gW, A.K, A.F);
    if constexpr (PART == 3) soil_ab<SKF, U>(lds, blk, A.S, A.rS, A.nS, A.gS, A.K, A.F, A.mask_s);
    if constexpr (PART == 4) water_b<SKF, U>(lds, blk, A.W, A.rW, A.nW, A.gW, A.K, A.F, A.mask_w);
}

template <int PART, bool U>
constexpr size_t PART_LDS = STAGE_LDS<U ? WINDOWS : GENERAL, PART >= 3 ? 6 : PART == 1 ? 3 : 4>;

template <int SKF, int PART, bool U>
__global__ STAGE_ATTR void k_part(StageArgs A)
{
    __shared__ __align__(16) unsigned char lds[PART_LDS<PART, U>];
    if (PART == 0) post_flag(A.post, blockIdx.x);
    part<SKF, PART, U>(lds, xcd_block(), A);
}

// Stage 1 and stage 2 of a step uniform throughout, as k_stage1 and k_stage2.
template <int SKF>
__global__ STAGE_ATTR void k_stage1(StageArgs A)
{
    __shared__ __align__(16) unsigned char lds[VIS_LDS<4>];
    post_flag(A.post, blockIdx.x);
    const PartIdx p = part_of<3>(blockIdx.x, {A.nbXS, A.nbW, A.nbXW}, true);
    if (p.blk < 0) return;
    if (p.part == 0) part<SKF, 0, true>(lds, p.blk, A);
    else if (p.part == 1) part<SKF, 1, true>(lds, p.blk, A);
    else part<SKF, 2, true>(lds, p.blk, A);
}

template <int SKF>
__global__ STAGE_ATTR_AB void k_stage2(StageArgs A)
{
    __shared__ __align__(16) unsigned char lds[VIS_LDS<6>];
    const PartIdx p = part_of<2>(blockIdx.x, {A.nbS, A.nbW}, true);
    if (p.blk < 0) return;
    if (p.part == 0) part<SKF, 3, true>(lds, p.blk, A);
    else part<SKF, 4, true>(lds, p.blk, A);
}

}  // namespace learned
