// sph_single.h -- single-phase water step (single_step_for_water,
// declarations_sph.f90:1439-1526) on cell-sorted records.
//
// Three passes over the partners, since each needs the one before at the
// partners: the Shepard density (sum_density), then the rates and strains that
// use it, then the force that uses the strains.  The first pass scans the
// candidate rows with the exact predicate and stores each particle's partner
// mask; the other two visit the mask.  Records are chunk planes as in the
// two-phase step (chunk c of record t is element t of plane c, 16 bytes):
//   0 x,y | 1 vx,vy | 2 rho before the summation, m (negative: virtual) |
//   3 rho after it, m | 4 sxx - p, sxy | 5 syy - p, c | 6 h, itype
// Particles move up to about 1% of their support radius per step here (a
// dam break at a tenth of the sound speed), so the cell list is built every
// step rather than kept with a skin; its first pass (keys and arrival ranks)
// rides in the tail of the force pass, and its last (the rank inside the
// cell) in the pack.
//
// Lanes per particle: a particle's candidates are dealt over 1 << lg
// neighbouring lanes (candidate c to lane c mod 2^lg) and the sums combined by
// shuffles.  One lane per particle keeps the chip busy only from about 10^5
// particles on; below that the serial partner loop sets the time.
//
// Bound: latency below about 40k particles (six launches of 4-8 us), the
// partner gathers above.  Against one thread per particle over the unsorted
// state with exact divisions and a candidate test in each pass, per step:
// dam break of 7.5k particles 228 -> 40 us (leapfrog), 168k 292 -> 99 us
// (Verlet).
#pragma once
#include "sph_fused.h"

// Scan of the candidate rows by the lanes of a particle: the concatenated
// mask of its own candidates (ovf: more than 128 in all).
template <class A>
__device__ __forceinline__ CatMask scan_sub(const LaneRows& L, int lg, int sub, int self, const RecV& rec, A&& acc)
{
    const int s1 = L.k1[0] - L.k0[0], s2 = s1 + L.k1[1] - L.k0[1], tot = s2 + L.k1[2] - L.k0[2];
    const int e0 = L.k0[0], e1 = L.k0[1] - s1, e2 = L.k0[2] - s2;
    CatMask m{0, 0, tot > 128 ? 7 : 0};
    if (m.ovf) return m;
#pragma unroll 1
    for (int c0 = sub; c0 < tot; c0 += 4 << lg) {
        int k[4];
        double2 p[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {   // (a candidate past the end repeats the first)
            const int c = c0 + (j << lg), cc = c < tot ? c : c0;
            k[j] = cc + pick(cc < s1, e0, pick(cc < s2, e1, e2));
            p[j] = rec(k[j], 0);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int c = c0 + (j << lg);
            const uint64_t bit = (uint64_t)(c < tot && k[j] != self && acc(k[j], p[j])) << (c & 63);
            m.lo |= pick(c < 64, bit, (uint64_t)0);
            m.hi |= pick(c < 64, (uint64_t)0, bit);
        }
    }
    return m;
}

// Direct walk of an overflowed particle's rows (more than 128 candidates):
// the candidates of this lane that pass the predicate.
template <class A, class B>
__device__ __forceinline__ void walk_sub(const LaneRows& L, int lg, int sub, int self, A&& accept, B&& body)
{
    const int s1 = L.k1[0] - L.k0[0], s2 = s1 + L.k1[1] - L.k0[1], tot = s2 + L.k1[2] - L.k0[2];
    const int e0 = L.k0[0], e1 = L.k0[1] - s1, e2 = L.k0[2] - s2;
#pragma unroll 1
    for (int c = sub; c < tot; c += 1 << lg) {
        const int k = c + pick(c < s1, e0, pick(c < s2, e1, e2));
        if (k == self || !accept(k)) continue;
        body(k);
    }
}

// Partners of a lane: the set bits of its mask, then the rows of an overflow.
template <class A, class B>
__device__ __forceinline__ void visit_sub(const CatMask& m, const LaneRows& L, int lg, int sub, int self, A&& accept,
                                          B&& body)
{
    CatIter it = cat_iter(m, L);
#pragma unroll 1
    for (int k = it.next(); k >= 0; k = it.next()) body(k);
    if (m.ovf) walk_sub(L, lg, sub, self, accept, body);
}

// ------------------------------------------------------------------------
// Pack: record t of the cell order from the state, after first_half
// (do_half, declarations_sph.f90:643-684) when the step before has not
// applied it.  arr: the cell list's arrival order (the rank inside the cell
// is taken here), null: P.order is final.
// ------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_w1_pack(DPhase P, KParams K, double* rec, const int* arr, int do_half)
{
#pragma clang fp contract(off)
    const int u = blockIdx.x * blockDim.x + threadIdx.x;
    if (u >= P.n) return;
    int t = u, i;
    if (arr) {
        t = cell_place(P, arr, u, i);
        P.order[t] = i;
    } else {
        i = P.order[t];
    }
    const int it = P.itype[i];
    double rho = P.rho[i], vx = P.vx[i], vy = P.vy[i];
    if (do_half) {
        const double h = K.dt / 2.0;
        if (!K.summation_density) {
            P.rho_min[i] = rho;
            rho = rho + h * P.drho[i];
            P.rho[i] = rho;
        }
        if (it >= 0) {
            P.vx_min[i] = vx;
            P.vy_min[i] = vy;
            vx = vx + h * P.ax[i];
            vy = vy + h * P.ay[i];
            P.vx[i] = vx;
            P.vy[i] = vy;
        }
    }
    const double m = P.mass[i];
    double2* R = reinterpret_cast<double2*>(rec) + t;
    const size_t pn = (size_t)P.n;
    R[0 * pn] = make_double2(P.x[i], P.y[i]);
    R[1 * pn] = make_double2(vx, vy);
    R[2 * pn] = make_double2(rho, it < 0 ? -m : m);
    R[6 * pn] = make_double2(P.hsml[i], (double)it);
}

// What the three passes share: the particle, its rows and its predicate.
struct W1Self {
    double xa, ya, ha;
    LaneRows L;
    Pred P;
    bool uni, one_h;   // one kernel length for all pairs; one smoothing length
};

template <bool U>
__device__ __forceinline__ W1Self w1_self(const DPhase& W, const RecV& R, int tt, const Grid& g, const KParams& K,
                                          const FusedK& F)
{
    W1Self s;
    const double2 xy = R(tt, 0);
    const bool link = K.nnps == 2;
    s.xa = xy.x;
    s.ya = xy.y;
    s.ha = U ? K.h1_water : R(tt, 6).x;
    s.one_h = U;
    s.uni = U || link;
    s.L = lane_rows(block_rows(g, W.cell_start, s.xa, s.ya));
    s.P = Pred{s.xa, s.ya, s.ha, F.thr_w, s.uni ? 1 : 0, link ? 1 : 0};
    return s;
}

// Pair geometry: d, d^2, W and s = (grad W) / d, and the pair's mean smoothing
// length (art_visc's; the kernel takes hsml(1) under link_list).
struct W1Pair {
    double dx, dy, dr, w, s, h;
};

template <int SKF, bool NEED_W>
__device__ __forceinline__ W1Pair w1_pair(const W1Self& a, const KC& kc, const RecV& R, int k, double2 b)
{
    W1Pair p;
    p.dx = a.xa - b.x;
    p.dy = a.ya - b.y;
    p.dr = p.dx * p.dx + p.dy * p.dy;
    const double ir = p.dr > 0.0 ? fast_rsq(p.dr) : 0.0, r = p.dr * ir;
    p.h = a.one_h ? a.ha : sph_mhsml(a.ha, R(k, 6).x);
    if (a.uni) kern_s<SKF, NEED_W>(kc, r, ir, p.w, p.s);
    else kern_s<SKF, NEED_W>(make_kc(SKF, p.h), r, ir, p.w, p.s);
    return p;
}

// ------------------------------------------------------------------------
// Shepard summation density (sum_density, m_particles.f90:2243-2298) from
// the density before it, and the partner masks of the step.
// ------------------------------------------------------------------------
template <int SKF, bool U>
__global__ __launch_bounds__(256) void k_w1_density(DPhase W, double* recw, Masks MW, Grid g, KParams K, FusedK F,
                                                    int lg)
{
    const RecV R = recv(recw, W.n);
    const SubCtx sc = sub_ctx(W.n, xcd_block(), lg, 256);
    const W1Self a = w1_self<U>(W, R, sc.tt, g, K, F);
    const double2 rm = R(sc.tt, 2);
    const double ma = fabs(rm.y);
    const KC kc = make_kc(SKF, K.nnps == 2 ? K.h1_water : a.ha);
    auto acc = [&](int k, double2 b) { return a.P(b, a.uni ? a.ha : R(k, 6).x, g, K); };
    auto acc_k = [&](int k) { return acc(k, R(k, 0)); };
    const CatMask cm = scan_sub(a.L, lg, sc.sub, sc.t, R, acc);
    double wi = 0.0, rs = 0.0, cnt = 0.0;
    visit_sub(cm, a.L, lg, sc.sub, sc.t, acc_k, [&](int k) {
        const double2 b = R(k, 0), q = R(k, 2);
        const W1Pair p = w1_pair<SKF, true>(a, kc, R, k, b);
        const double mw = fabs(q.y) * p.w;
        wi += mw * fast_rcp(q.x);
        rs += mw;
        cnt += 1.0;
    });
    sub_sum(lg, wi, rs, cnt);
    const uint64_t lo = sub_or(lg, cm.lo), hi = sub_or(lg, cm.hi);
    if (!sc.valid || sc.sub) return;
    double self, d0, d1;
    sph_kernel(SKF, 0.0, 0.0, 0.0, a.ha, self, d0, d1);
    const double rho = (self * ma + rs) / (self * ma / rm.x + wi);
    MW.m[sc.t] = lo;
    MW.m[W.n + sc.t] = hi;
    MW.ovf[sc.t] = cm.ovf;
    const int i = W.order[sc.t];
    W.rho[i] = rho;
    W.countiac[i] = (int)cnt;
    reinterpret_cast<double2*>(recw)[3 * (size_t)W.n + sc.t] = make_double2(rho, ma);
}

// ------------------------------------------------------------------------
// drho = -rho (df2(vx,'x') + df2(vy,'y')) + delta_sph(rho); strains via df
// (:1482-1484); p = b ((rho/rho0)**gamma - 1) (:1478); av_vel.
// ------------------------------------------------------------------------
template <int SKF, bool U>
__global__ __launch_bounds__(256) void k_w1_rates(DPhase W, double* recw, Masks MW, Grid g, KParams K, FusedK F,
                                                  int mask, int lg)
{
    const RecV R = recv(recw, W.n);
    const SubCtx sc = sub_ctx(W.n, xcd_block(), lg, 256);
    const W1Self a = w1_self<U>(W, R, sc.tt, g, K, F);
    const double2 va = R(sc.tt, 1);
    const double rhoa = R(sc.tt, 3).x;
    const KC kc = make_kc(SKF, K.nnps == 2 ? K.h1_water : a.ha);
    auto acc_k = [&](int k) { return a.P(R(k, 0), a.uni ? a.ha : R(k, 6).x, g, K); };
    CatMask cm = mask_of(MW, W.n, sc.tt);
    cm.lo &= sub_bits(lg, sc.sub);
    cm.hi &= sub_bits(lg, sc.sub);
    if (!sc.valid) cm = CatMask{0, 0, 0};
    double con = 0.0, drd = 0.0, xx = 0.0, xy = 0.0, yx = 0.0, yy = 0.0, avx = 0.0, avy = 0.0;
    visit_sub(cm, a.L, lg, sc.sub, sc.t, acc_k, [&](int k) {
        const double2 b = R(k, 0), v = R(k, 1), q = R(k, 3);
        const W1Pair p = w1_pair<SKF, true>(a, kc, R, k, b);
        const double ms = q.y * p.s, Vs = ms * fast_rcp(q.x), wx = Vs * p.dx, wy = Vs * p.dy;
        const double dvx = va.x - v.x, dvy = va.y - v.y, svx = va.x + v.x, svy = va.y + v.y;
        con += ms * (dvx * p.dx + dvy * p.dy);
        drd += Vs * (rhoa - q.x);
        xx += wx * svx;
        xy += wy * svx;
        yx += wx * svy;
        yy += wy * svy;
        const double f = q.y * p.w * fast_rcp(rhoa + q.x);
        avx -= f * dvx;
        avy -= f * dvy;
    });
    sub_sum(lg, con, drd, xx, xy, yx, yy, avx, avy);
    if (!sc.valid || sc.sub) return;
    const int i = W.order[sc.t];
    const double c = W.c[i];
    const double txx = SPH_C23_F * (2.0 * xx - yy), txy = xy + yx, tyy = SPH_C23_F * (2.0 * yy - xx);
    W.drho[i] = (mask & M_DRHO_DELTA) ? con + (K.delta * a.ha * c) * (2.0 * drd) : con;
    W.txx[i] = txx;
    W.txy[i] = txy;
    W.tyy[i] = tyy;
    double p;
    if (rhoa > 0.0) {
        p = K.w_b * (pow(rhoa / K.w_rho0, K.w_gamma) - 1.0);
        W.p[i] = p;
    } else {
        p = W.p[i];
    }
    if (mask & M_XSPH) {
        const double e = W.itype[i] > 0 ? K.epsilon : 1.0;
        W.avx[i] = e * (2.0 * avx);
        W.avy[i] = e * (2.0 * avy);
    }
    double2* Rw = reinterpret_cast<double2*>(recw) + sc.t;
    const size_t pn = (size_t)W.n;
    Rw[4 * pn] = make_double2(K.w_mu * txx - p, K.w_mu * txy);
    Rw[5 * pn] = make_double2(K.w_mu * tyy - p, c);
}

// What follows the force of a step: nothing (the right-hand side alone), the
// leapfrog's first_step / second_half or the Verlet update; ahead: another
// step follows at once, so its first_half and its cell keys and arrival
// ranks (cell_count starts at zero) are taken here too.
struct W1End {
    int scheme;      // 0 none, 1 leapfrog, 2 Verlet
    int step, ahead;
    double *lvx, *lvy, *lrho, h2;
    int* err;
};

// ------------------------------------------------------------------------
// dvx = -df(p,'x') + df(sxx,'x') + df(sxy,'y') (:1494-1498), /rho, art_visc,
// gravity; then the update of the particle (the partners are read from the
// records alone, so the state may move).
// ------------------------------------------------------------------------
template <int SKF, bool U>
__global__ __launch_bounds__(256) void k_w1_force(DPhase W, const double* rec, Masks MW, Grid g, KParams K, FusedK F,
                                                  int mask, int lg, W1End E)
{
    const RecV R = recv(rec, W.n);
    const SubCtx sc = sub_ctx(W.n, xcd_block(), lg, 256);
    const W1Self a = w1_self<U>(W, R, sc.tt, g, K, F);
    const double2 va = R(sc.tt, 1), s4 = R(sc.tt, 4), s5 = R(sc.tt, 5);
    const double rhoa = R(sc.tt, 3).x;
    const KC kc = make_kc(SKF, K.nnps == 2 ? K.h1_water : a.ha);
    auto acc_k = [&](int k) { return a.P(R(k, 0), a.uni ? a.ha : R(k, 6).x, g, K); };
    CatMask cm = mask_of(MW, W.n, sc.tt);
    cm.lo &= sub_bits(lg, sc.sub);
    cm.hi &= sub_bits(lg, sc.sub);
    if (!sc.valid) cm = CatMask{0, 0, 0};
    const double et2 = K.etq * K.etq;
    double Fx = 0.0, Fy = 0.0, artx = 0.0, arty = 0.0;
    visit_sub(cm, a.L, lg, sc.sub, sc.t, acc_k, [&](int k) {
        const double2 b = R(k, 0), v = R(k, 1), q = R(k, 3), b4 = R(k, 4), b5 = R(k, 5);
        const W1Pair p = w1_pair<SKF, false>(a, kc, R, k, b);
        const double ms = q.y * p.s, Vs = ms * fast_rcp(q.x), wx = Vs * p.dx, wy = Vs * p.dy;
        const double sxy = s4.y + b4.y;
        Fx += (s4.x + b4.x) * wx + sxy * wy;
        Fy += (s5.x + b5.x) * wy + sxy * wx;
        const double vr = (va.x - v.x) * p.dx + (va.y - v.y) * p.dy;
        // art_visc, branch-free: approaching pairs only (vr < 0)
        const double muv = p.h * vr * fast_rcp(p.dr + p.h * p.h * et2);
        double piv = (K.beta * muv - K.alpha * (0.5 * (s5.y + b5.y))) * muv * (2.0 * fast_rcp(rhoa + q.x));
        piv = vr < 0.0 ? ms * piv : 0.0;
        artx -= piv * p.dx;
        arty -= piv * p.dy;
    });
    sub_sum(lg, Fx, Fy, artx, arty);
    const bool own = sc.valid && !sc.sub;
    const int i = sc.valid ? W.order[sc.t] : 0;
    double nx = 0.0, ny = 0.0;
    if (own) {
#pragma clang fp contract(off)
        const double irho = rhoa > 0.0 ? 1.0 / rhoa : 1.0;
        double ax = Fx * irho, ay = Fy * irho;
        if (mask & M_ART) { ax = ax + artx; ay = ay + arty; }
        ay = ay + K.gravity;
        W.ax[i] = ax;
        W.ay[i] = ay;
        const double dt = K.dt, h = dt / 2.0, drho = W.drho[i];
        nx = W.x[i];
        ny = W.y[i];
        if (E.scheme == 1) {
            const bool first = E.step == 1;
            double rho = rhoa;
            if (!K.summation_density) rho = first ? rho + h * drho : W.rho_min[i] + dt * drho;
            if (W.itype[i] >= 0) {
                const double k = first ? h : dt;
                double vx = (first ? va.x : W.vx_min[i]) + k * ax + W.avx[i];
                double vy = (first ? va.y : W.vy_min[i]) + k * ay + W.avy[i];
                nx = nx + dt * vx;
                ny = ny + dt * vy;
                W.x[i] = nx;
                W.y[i] = ny;
                if (E.ahead) {
                    W.vx_min[i] = vx;
                    W.vy_min[i] = vy;
                    vx = vx + h * ax;
                    vy = vy + h * ay;
                }
                W.vx[i] = vx;
                W.vy[i] = vy;
            }
            if (!K.summation_density) {
                if (E.ahead) {
                    W.rho_min[i] = rho;
                    rho = rho + h * drho;
                }
                W.rho[i] = rho;
            }
        } else if (E.scheme == 2) {
            // time_integration_for_water_by_verlet (declarations_sph.f90:889-974):
            // real particles (the first ntotal of the reference numbering)
            // move by dt v + h2 a with h2 = dt**2./2. and advance their other
            // velocity level by 2 dt a (every 50th step: restart from v + dt a);
            // every particle's other density level advances by 2 dt drho (step
            // 1 and every 50th step: restart); then both levels swap, as the
            // reference's whole-array swaps do (the virtual particles'
            // velocity levels swap unchanged)
            double nvx = E.lvx[i], nvy = E.lvy[i];
            if (W.id[i] < W.ntotal) {
                nx = nx + dt * va.x + E.h2 * ax;
                ny = ny + dt * va.y + E.h2 * ay;
                W.x[i] = nx;
                W.y[i] = ny;
                if (E.step % 50 != 0) {
                    nvx = nvx + 2.0 * dt * ax;
                    nvy = nvy + 2.0 * dt * ay;
                } else {
                    nvx = va.x + dt * ax;
                    nvy = va.y + dt * ay;
                }
            }
            W.vx[i] = nvx;
            W.vy[i] = nvy;
            E.lvx[i] = va.x;
            E.lvy[i] = va.y;
            double nr;
            if (E.step == 1) nr = rhoa + dt * 2.0 * drho;
            else if (E.step % 50 != 0) nr = E.lrho[i] + dt * 2.0 * drho;
            else nr = rhoa + dt * drho;
            W.rho[i] = nr;
            E.lrho[i] = rhoa;
        }
    }
    if (E.ahead) {
        const int key = own ? cell_key_of(g, nx, ny, E.err) : -1;
        // (the lanes of a particle share its key)
        const int gk = lg ? __shfl(key, (int)(threadIdx.x & 63) & ~((1 << lg) - 1), 64) : key;
        const int slot = cell_slot_of(W.cell_count, gk, lg);
        if (own) {
            W.key[i] = key;
            W.slot[i] = slot;
        }
    }
}

// ------------------------------------------------------------------------
// Single-phase soil: the pack (with the rank inside the cells, as
// k_w1_pack), then one pass over the partners (soil_ab4) with the step's final
// update and the next step's cell keys in its tail (the partners are read from
// the records alone).  Four launches a step instead of seven, and lanes per
// particle by size (solo_lanes); bound: launch latency to about 40k particles,
// then the candidate test and the partner gathers.  Per step: 3k particles 55
// -> 31 us, 65k 63 -> 47, 128k 84 -> 60.
// ------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_solo_pack(DPhase P, KParams K, double* rec, const int* arr, int do_half,
                                                   int ndp)
{
    const int u = blockIdx.x * blockDim.x + threadIdx.x;
    if (u >= P.n) return;
    int t = u, i;
    if (arr) {
        t = cell_place(P, arr, u, i);
        P.order[t] = i;
    } else {
        i = P.order[t];
    }
    pack_soil_state(P, K, rec, t, i, do_half, ndp, nullptr, Grid{}, 0.0, NRef{});
}

// What follows the rates: nothing (the right-hand side alone), or the update
// of the step; ahead: and the cell keys and arrival ranks of the next one
// (cell_count starts at zero).
struct SoloEnd {
    int update, first, ahead;
    int* err;
};

template <int SKF, int FORM>
__global__ __launch_bounds__(256) void k_solo_step(DPhase S, const double* recS, Grid g, KParams K, FusedK F, int mask,
                                                   int lg, SoloEnd E)
{
    NList NL{};
    NL.lg = lg;
    soil_ab4<SKF, FORM, true>(nullptr, xcd_block(), S, recS, NL, g, K, F, 0, mask, E.ahead);
    if (!E.update) return;
    const SubCtx sc = sub_ctx(S.n, xcd_block(), lg, STAGE_BLOCK);
    const bool own = sc.valid && !sc.sub;
    const int i = S.order[sc.tt];
    int key = -1;
    if (own) {
        const SoilEnd e = final_soil_at(S, K, i, E.first);
        if (E.ahead) key = cell_key_of(g, e.x, e.y, E.err);
    }
    if (E.ahead) {
        // (the lanes of a particle share its key)
        const int gk = lg ? __shfl(key, (int)(threadIdx.x & 63) & ~((1 << lg) - 1), 64) : key;
        const int slot = cell_slot_of(S.cell_count, gk, lg);
        if (own) {
            S.key[i] = key;
            S.slot[i] = slot;
        }
    }
}
