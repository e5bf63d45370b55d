// sph_fused.h -- the fused two-phase step (FP64), tuned for CDNA4.
//
// Per phase and step:
//   pack      thread t of the cell order: half-step update of particle order[t]
//             and its neighbour record t, cell-sorted and stored as chunk
//             planes (chunk c of record t is element t of plane c).  Record
//             chunks (16 bytes): 0 x,y | 1 vx,vy | 2 rho,V | 3 vof,p (soil:
//             vof/rho,p) | 4 s3,c | 5 s1,s2 | 6 h,itype; V = m/rho carries the
//             sign of itype (negative for virtual particles), so the pair
//             terms need no reciprocal of the partner's density (a step of a
//             learned run has m and the soil's vof instead, sph_learned.h).
//             The loops load only the chunks they use;
//   stage A   the same-phase terms that need only the packed values;
//   stage B   (water) the terms that need the partners' strain rates.  Soil
//             stage B needs nothing from the stage A of other soil particles,
//             so soil runs both stages in one kernel over one partner loop.
// The cross terms have passes of their own.  Lanes of a wavefront hold
// consecutive cell-sorted particles.
#pragma once
#include "sph_kernels.h"

// doubles per record
constexpr int R_STRIDE = 16;

#ifndef SPHG_WPB
#define SPHG_WPB 4           // waves per workgroup of the stage kernels (consecutive particles share a CU)
#endif
constexpr int STAGE_BLOCK = 64 * SPHG_WPB;
#ifndef SPHG_STAGE_WAVES
#define SPHG_STAGE_WAVES 0   // 0: compiler's choice; n: ask for at least n waves per SIMD
#endif
#if SPHG_STAGE_WAVES > 0
#define STAGE_ATTR __launch_bounds__(STAGE_BLOCK) __attribute__((amdgpu_waves_per_eu(SPHG_STAGE_WAVES, 8)))
#else
#define STAGE_ATTR __launch_bounds__(STAGE_BLOCK)
#endif
#ifndef SPHG_AB_WAVES
#define SPHG_AB_WAVES 0      // the same for the one-pass soil kernel
#endif
#if SPHG_AB_WAVES > 0
#define STAGE_ATTR_AB __launch_bounds__(STAGE_BLOCK) __attribute__((amdgpu_waves_per_eu(SPHG_AB_WAVES, 8)))
#else
#define STAGE_ATTR_AB __launch_bounds__(STAGE_BLOCK)
#endif

struct FusedK {
    // dr thresholds and uniform-h flags for same-phase (water, soil) and cross pairs
    double thr_w, thr_s, thr_x;
    int uni_w, uni_s, uni_x;
};

// q^n for an integer 0 <= n <= 64 by binary powering (within a few ulp of pow).
__device__ __forceinline__ double ipow(double q, int n)
{
    double r = 1.0, b = q;
#pragma unroll 1
    for (; n > 0; n >>= 1) {
        if (n & 1) r *= b;
        b *= b;
    }
    return r;
}

// 1/d and 1/sqrt(d) from the hardware estimates (about 2^-23) plus one
// third-order step (error below 2^-60 before its rounding), i.e. to about one
// ulp; far shorter dependency chains than IEEE-exact FP64 division and square
// root.
__device__ __forceinline__ double fast_rcp(double d)
{
    const double x = __builtin_amdgcn_rcp(d);
    const double e = fma(-d, x, 1.0);
    return fma(x, fma(e, e, e), x);
}

__device__ __forceinline__ double fast_rsq(double d)
{
    const double y = __builtin_amdgcn_rsq(d);
    const double e = fma(-(d * y), y, 1.0);
    return fma(y * e, fma(0.375, e, 0.5), y);
}

// Kernel constants for one smoothing length: the normalisation factor f,
// and per kernel the coefficients of W and of s = |grad W| / r.
struct KC {
    double inv_h, f, c1, c2, c3;
};

__device__ __forceinline__ KC make_kc(int skf, double h)
{
    KC k;
    k.inv_h = 1.0 / h;
    const double ih2 = k.inv_h * k.inv_h;
    if (skf == 1) {
        k.f = 15.0 / (7.0 * SPH_PI_F * h * h);
        k.c1 = 2.0 * (k.f * ih2);            // s, q <= 1: c1 (0.75 q - 1)
        k.c2 = -0.5 * (k.f * k.inv_h);       // s, q > 1: c2 (2 - q)^2 / r
        k.c3 = k.f * (1.0 / 6.0);            // W, q > 1
    } else if (skf == 2) {
        k.f = 1.0 / ((h * h) * SPH_PI_F);
        k.c1 = -2.0 * ih2;
        k.c2 = k.c3 = 0.0;
    } else if (skf == 3) {
        k.f = 7.0 / (478.0 * SPH_PI_F * h * h);
        k.c1 = k.f * ih2;
        k.c2 = k.f * k.inv_h;
        k.c3 = 0.0;
    } else {
        k.f = 7.0 / (4.0 * SPH_PI_F * h * h);
        k.c1 = k.f * ih2;
        k.c2 = k.c3 = 0.0;
    }
    return k;
}

// The same for the mean smoothing length of one pair: one short reciprocal
// instead of two divisions (2% of a step where h varies).
template <int SKF>
__device__ __forceinline__ KC pair_kc(double h)
{
    constexpr double norm = SKF == 1 ? 15.0 / (7.0 * SPH_PI_F) : SKF == 2 ? 1.0 / SPH_PI_F
                          : SKF == 3 ? 7.0 / (478.0 * SPH_PI_F) : 7.0 / (4.0 * SPH_PI_F);
    KC k;
    k.inv_h = fast_rcp(h);
    const double ih2 = k.inv_h * k.inv_h;
    k.f = norm * ih2;
    k.c1 = SKF == 1 ? 2.0 * (k.f * ih2) : SKF == 2 ? -2.0 * ih2 : k.f * ih2;
    k.c2 = SKF == 1 ? -0.5 * (k.f * k.inv_h) : SKF == 3 ? k.f * k.inv_h : 0.0;
    k.c3 = SKF == 1 ? k.f * (1.0 / 6.0) : 0.0;
    return k;
}

// W and s (grad W = s (dx, dy); m_particles.f90:1469-1602) of a pair inside
// the support; inv_r = 1/r.
template <int SKF, bool NEED_W>
__device__ __forceinline__ void kern_s(const KC& k, double r, double inv_r, double& w, double& s)
{
    const double q = r * k.inv_h;
    w = 0.0;
    if constexpr (SKF == 1) {
        // both pieces, then a select: no divergent branch in the pair loop
        const bool in1 = q <= 1.0;
        const double t = 2.0 - q, t2 = t * t;
        const double s1 = k.c1 * fma(0.75, q, -1.0), s2 = t2 * (k.c2 * inv_r);
        s = in1 ? s1 : s2;
        if (NEED_W) {
            const double w1 = k.f * fma(q * q, fma(0.5, q, -1.0), SPH_C23_F), w2 = t2 * (k.c3 * t);
            w = in1 ? w1 : w2;
        }
    } else if constexpr (SKF == 4) {
        const double t = fma(-0.5, q, 1.0), t2 = t * t;
        if (NEED_W) w = k.f * ((t2 * t2) * fma(2.0, q, 1.0));
        // (the reference's order of the terms: they cancel towards q = 2)
        s = k.c1 * (-5.0 + 7.5 * q - 3.75 * (q * q) + 0.625 * ((q * q) * q));
    } else if constexpr (SKF == 2) {
        w = k.f * exp(-q * q);
        s = k.c1 * w;
    } else {
        const double a = 3.0 - q, b = 2.0 - q, c = 1.0 - q;
        const double a2 = a * a, b2 = b * b, c2 = c * c;
        const double a4 = a2 * a2, b4 = b2 * b2, c4 = c2 * c2;
        if (q <= 1.0) {
            if (NEED_W) w = k.f * (a4 * a - 6.0 * (b4 * b) + 15.0 * (c4 * c));
            s = k.c1 * (-120.0 + 120.0 * q - 50.0 * (q * q));  // reference polynomial
        } else if (q <= 2.0) {
            if (NEED_W) w = k.f * (a4 * a - 6.0 * (b4 * b));
            s = k.c2 * (-(5.0 * a4) + 30.0 * b4) * inv_r;
        } else {
            if (NEED_W) w = k.f * (a4 * a);
            s = k.c2 * (-(5.0 * a4)) * inv_r;
        }
    }
}

// The records are stored as chunk planes: chunk c of record k is element k
// of plane c (n 16-byte elements per plane).  The lanes of a wave read one
// chunk of nearby partners at a time, so a plane layout touches a few cache
// lines per load where a 128-byte-per-record layout touches one per lane.
struct RecV {
    typedef double2 V;
    const double2* p;
    int n;
    // a record past the end of a list: far away, finite everywhere
    __device__ __forceinline__ static double2 stand_in(int c)
    {
        const double f = c == 0 ? 1.0e18 : 1.0;
        return make_double2(f, f);
    }
    // (uniform plane address plus a 32-bit lane offset: no 64-bit lane arithmetic)
    __device__ __forceinline__ double2 operator()(int k, int c) const
    {
        return *reinterpret_cast<const double2*>(reinterpret_cast<const char*>(p + (size_t)c * n) + ((uint32_t)k << 4));
    }
};

__device__ __forceinline__ RecV recv(const double* rec, int n)
{
    return RecV{reinterpret_cast<const double2*>(rec), n};
}

// Exact pair predicate: sqrt(dx^2+dy^2) < scale_k * mh  (direct_find) or
// < scale_k * h(1) within the reference grid reach (link_list).
__device__ __forceinline__ bool pred(bool uni, double thr, double dr, double ha, double hb, const KParams& K)
{
    if (uni) return dr < thr;
    return __builtin_sqrt(dr) < K.scale_k * sph_mhsml(ha, hb);
}

// Cell-row ranges of the 3 x 3 block around (x, y) in the cell order.
struct Rows {
    int k0[3], k1[3];
};

// Row ranges of the 3 x 3 block around cell (cx, cy).
__device__ __forceinline__ Rows block_rows_at(const Grid& g, const int* cell_start, int cx, int cy)
{
    Rows R;
    const int c0 = max(cx - 1, 0), c1 = min(cx + 1, g.ncx - 1);
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        const int row = cy - 1 + r;
        if (row >= 0 && row < g.ncy) {
            R.k0[r] = cell_start[row * g.ncx + c0];
            R.k1[r] = cell_start[row * g.ncx + c1 + 1];
        } else {
            R.k0[r] = 0;
            R.k1[r] = 0;
        }
    }
    return R;
}

// Cell of a position, clamped into the grid (a particle outside it has
// raised the out-of-range flag at the cell-list build).
__device__ __forceinline__ void clamped_cell(const Grid& g, double x, double y, int& cx, int& cy)
{
    grid_cell(g, x, y, cx, cy);
    cx = min(max(cx, 0), g.ncx - 1);
    cy = min(max(cy, 0), g.ncy - 1);
}

__device__ __forceinline__ Rows block_rows(const Grid& g, const int* cell_start, double x, double y)
{
    int cx, cy;
    clamped_cell(g, x, y, cx, cy);
    return block_rows_at(g, cell_start, cx, cy);
}

constexpr int Q_STRIDE = 16;   // floats per record: four float4 chunk planes

// FP32 records of the mixed-precision form, as chunk planes like RecV.
struct RecQ {
    typedef float4 V;
    const float4* p;
    int n;
    __device__ __forceinline__ static float4 stand_in(int c)
    {
        return c == 0 ? make_float4(1.0e12f, 1.0e12f, 0.0f, 1.0f) : make_float4(1.0f, 1.0f, 1.0f, 1.0f);
    }
    __device__ __forceinline__ float4 operator()(int k, int c) const { return p[(size_t)c * n + k]; }
};

__device__ __forceinline__ RecQ recqv(const float* q, int n)
{
    return RecQ{reinterpret_cast<const float4*>(q), n};
}

__device__ __forceinline__ int cell_tag(int cx, int cy, bool is_virtual)
{
    return (is_virtual ? (int)0x80000000 : 0) | (cx << 15) | cy;
}
__device__ __forceinline__ int tag_cx(int tag) { return (tag >> 15) & 0x7fff; }
__device__ __forceinline__ int tag_cy(int tag) { return tag & 0x7fff; }

// FP32 neighbour record of the mixed-precision form (the layout is
// described in sph_mixed.h): chunks q0 and q1 of the record at R (plane 0),
// planes pn elements apart.
// key >= 0: the record's cell is the row-major cell `key` (the cell of the
// particle at the neighbour-list rebuild, which it may have left since);
// otherwise the cell of its position.
__device__ __forceinline__ void write_q01(float4* R, size_t pn, const Grid& g, double cs, double x, double y, double h,
                                          bool virt, double vx, double vy, double drho, double m, int key)
{
    int cx, cy;
    if (key >= 0) {
        cy = key / g.ncx;
        cx = key - cy * g.ncx;
    } else {
        grid_cell(g, x, y, cx, cy);
        cx = min(max(cx, 0), g.ncx - 1);
        cy = min(max(cy, 0), g.ncy - 1);
    }
    const double xc = g.x0 + ((double)cx + 0.5) * cs, yc = g.y0 + ((double)cy + 0.5) * cs;
    R[0] = make_float4((float)(x - xc), (float)(y - yc), __int_as_float(cell_tag(cx, cy, virt)), (float)h);
    R[pn] = make_float4((float)vx, (float)vy, (float)drho, (float)m);
}

// ------------------------------------------------------------------------
// pack: half-step update (first_half, declarations_sph.f90:643-684, and the
// soil Drucker-Prager projections) fused with writing the neighbour record.
// ------------------------------------------------------------------------
// Displacement since the neighbour-list rebuild, per record slot t (the
// record order is fixed between rebuilds).  A rebuild (rebuild = 1) records
// the position.  Later steps raise bit 0 of flag (rebuild) when the
// displacement d passes trig, or when d plus `look` times the speed (look =
// a few steps' dt) passes near, so that a rebuild that takes effect two
// steps after the flag is raised still comes before d reaches half the
// skin; and bit 1 when d is past half the skin (d^2 > hard2): the lists may
// then have missed a pair.  One atomic per wave.  x == nullptr: no lists.
struct NRef {
    double *x, *y;
    int* flag;
    double trig, near, hard2, look;
    int rebuild;
    const int* cell;   // cell key per record slot since the rebuild (FP32 records)
    int* bad;          // raised by a record with an infinity or a NaN
};

// Raises bad when one of the values is not finite.
template <class... T>
__device__ __forceinline__ void check_finite(int* bad, T... v)
{
    if (bad && !((... + ((T)0 * v)) == 0)) atomicOr(bad, 1);
}

__device__ __forceinline__ int record_cell(const NRef& R, int t) { return R.cell && !R.rebuild ? R.cell[t] : -1; }

__device__ __forceinline__ void track_displacement(const NRef& R, int t, double x, double y, double vx, double vy)
{
    if (!R.x) return;
    if (R.rebuild) {
        R.x[t] = x;
        R.y[t] = y;
        return;
    }
    const double dx = x - R.x[t], dy = y - R.y[t];
    const double d2 = dx * dx + dy * dy;
    const double d = sqrt(d2);
    const bool hard = !(d2 <= R.hard2);
    const bool due = hard || !(d <= R.trig) || !(d + R.look * sqrt(vx * vx + vy * vy) <= R.near);
    const uint64_t any_due = __ballot(due), any_hard = __ballot(hard);
    const uint64_t active = __ballot(1);
    if (any_due && (int)(threadIdx.x & 63) == __ffsll((unsigned long long)active) - 1)
        atomicOr(R.flag, any_hard ? 3 : 1);
}

// q != nullptr selects the FP32 record of the mixed-precision form.
// Pack of water particle i into record slot t from its current values x,
// v, rho, vof (the state's, or those the final update of the step before has
// just computed): first_half (do_half), the equation of state, the record.
// lean: the half-step levels that nothing reads before the next final update
// (which starts from the saved full-step levels) stay out of the state; only
// for a pack that the next step's stages read from FP64 records alone.
// lean_v: the same for the velocity alone (no stage reads the state's).
__device__ __forceinline__ void pack_water_at(const DPhase& P, const KParams& K, double* rec, int t, int i,
                                              int do_half, bool lean, bool lean_v, float* q, const Grid& g,
                                              double cs, const NRef& NR, double x, double y, double rho, double vof,
                                              double vx, double vy)
{
#pragma clang fp contract(off)
    track_displacement(NR, t, x, y, vx, vy);
    const int it = P.itype[i];
    if (do_half) {
        const double h = K.dt / 2.0;
        if (!K.summation_density) {   // first_half's rho update (declarations_sph.f90:647-650)
            P.rho_min[i] = rho;
            rho = rho + h * P.drho[i];
            if (!lean) P.rho[i] = rho;
        }
        if (K.volume_fraction && K.two_phase) {
            P.vof_min[i] = vof;
            vof = vof + h * P.dvof[i];
            if (!lean || K.summation_density) P.vof[i] = vof;   // the renormalisation reads it then
        }
        if (it > 0) {
            P.vx_min[i] = vx;
            P.vy_min[i] = vy;
            vx = vx + h * P.ax[i];
            vy = vy + h * P.ay[i];
            if (!lean_v) {
                P.vx[i] = vx;
                P.vy[i] = vy;
            }
        }
    }
    const double m = P.mass[i];
    const double irho = 1.0 / rho;
    // equation of state (pressure(), new sound speed) at the half-step
    // density: pointwise, so the soil stage can read the new water pressure
    // without waiting for the water stage
    const double rr = rho / (K.w_rho0 * vof);
    const double p = K.w_b * (pow(rr, K.w_gamma) - 1.0);
    const double cn = K.w_c * pow(rr, 3.0);
    P.p[i] = p;
    P.c_next[i] = cn;
    if (q) {
        float4* Q = reinterpret_cast<float4*>(q) + t;
        const size_t pn = (size_t)P.n;
        write_q01(Q, pn, g, cs, x, y, P.hsml[i], it < 0, vx, vy, rho - K.w_rho0, m, record_cell(NR, t));
        Q[2 * pn] = make_float4((float)vof, (float)irho, (float)(m * irho), (float)p);
        Q[3 * pn] = make_float4((float)cn, 0.0f, 0.0f, 0.0f);
        check_finite(NR.bad, (float)x, (float)y, (float)vx, (float)vy, (float)rho, (float)m, (float)vof, (float)irho, (float)(m * irho),
                     (float)p, (float)cn);
        return;
    }
    double2* R = reinterpret_cast<double2*>(rec) + t;
    const size_t pn = (size_t)P.n;
    R[0 * pn] = make_double2(x, y);
    R[1 * pn] = make_double2(vx, vy);
    const double V = m * irho;
    const double mv = K.learned ? m : V;
    check_finite(NR.bad, x, y, vx, vy, rho, V, vof, p, cn);
    R[2 * pn] = make_double2(rho, it < 0 ? -mv : mv);   // the sign marks a virtual particle
    R[3 * pn] = make_double2(vof, p);
    R[4 * pn] = make_double2(0.0, cn);
    // (h and itype stay between list rebuilds, in the same slot: a lean pack
    // finds chunk 6 as the call's first pack or the rebuild's wrote it)
    if (!lean) R[6 * pn] = make_double2(P.hsml[i], (double)it);
}

__device__ __forceinline__ void pack_water_body(int blk, DPhase P, KParams K, double* rec, int do_half, float* q,
                                                Grid g, double cs, NRef NR)
{
    const int t = blk * blockDim.x + threadIdx.x;
    if (t >= P.n) return;
    const int i = P.order[t];
    pack_water_at(P, K, rec, t, i, do_half, false, false, q, g, cs, NR, P.x[i], P.y[i], P.rho[i], P.vof[i], P.vx[i], P.vy[i]);
}

__global__ void k_pack_water(DPhase P, KParams K, double* rec, int do_half, float* q, Grid g, double cs, NRef NR)
{
    pack_water_body(blockIdx.x, P, K, rec, do_half, q, g, cs, NR);
}

// The final update of step s fused with the pack of step s + 1 (first_half,
// full step): one pass over the state instead of two, with the same values
// in memory afterwards as k_final_water followed by k_pack_water(do_half =
// 1), apart from stores the pack would overwrite and the half-step levels
// the pack leaves out (lean with FP64 records, lean_v always).  The record
// order of step s + 1 must be the current one (neighbour lists kept, no
// cell-list rebuild), and step s + 1 must follow at once: its final update
// is the next reader of the state.
__device__ __forceinline__ void step_water(int blk, DPhase P, KParams K, double* rec, int first, int with_vof,
                                           int renorm, float* q, Grid g, double cs, NRef NR)
{
    const int t = blk * blockDim.x + threadIdx.x;
    if (t >= P.n) return;
    const int i = t;   // (lists kept: the state is in record order)
    const WaterEnd e = water_end(P, K, i, first, with_vof, renorm);
    const int it = P.itype[i];
    // the final update's stores that the pack does not overwrite
    if (K.summation_density && renorm) P.rho[i] = e.rho;
    if (with_vof && !(K.volume_fraction && K.two_phase)) P.vof[i] = e.vof;
    if (it >= 0) {
        P.x[i] = e.x;
        P.y[i] = e.y;
        if (it == 0) {
            P.vx[i] = e.vx;
            P.vy[i] = e.vy;
        }
    }
    pack_water_at(P, K, rec, t, i, 1, q == nullptr, true, q, g, cs, NR, e.x, e.y, e.rho, e.vof, e.vx, e.vy);
}

__global__ void k_step_water(DPhase P, KParams K, double* rec, int first, int with_vof, int renorm, float* q, Grid g,
                             double cs, NRef NR)
{
    step_water(blockIdx.x, P, K, rec, first, with_vof, renorm, q, g, cs, NR);
}

// Pack of soil particle i (values as for water, plus stress and pressure):
// first_half (do_half), ndp Drucker-Prager projections (the last one
// single_step's failure criterion), the record.  lean as for water: the
// soil density stays (the final update's vof reads it), and the stress
// levels stay unless the final update starts from the saved ones
// (stress_integration = 2).
__device__ __forceinline__ void pack_soil_at(const DPhase& P, const KParams& K, double* rec, int t, int i,
                                             int do_half, bool lean, bool lean_v, int ndp, float* q, const Grid& g,
                                             double cs, const NRef& NR, double x, double y, double rho, double vx,
                                             double vy, double p, double sxx, double sxy, double syy)
{
#pragma clang fp contract(off)
    track_displacement(NR, t, x, y, vx, vy);
    const int it = P.itype[i];
    if (do_half) {
        const double h = K.dt / 2.0;
        if (!K.summation_density) {   // first_half's rho update (declarations_sph.f90:647-650)
            P.rho_min[i] = rho;
            rho = rho + h * P.drho[i];
            P.rho[i] = rho;
        }
        if (it > 0) {
            P.vx_min[i] = vx;
            P.vy_min[i] = vy;
            vx = vx + h * P.ax[i];
            vy = vy + h * P.ay[i];
            if (!lean_v) {
                P.vx[i] = vx;
                P.vy[i] = vy;
            }
        }
    }
    const bool keep_stress = !lean || K.stress_integration != 2;
    if (do_half && K.stress_integration == 2) {   // first_half, declarations_sph.f90:664-672
        const double h = K.dt / 2.0;
        P.sxx_min[i] = sxx; P.sxy_min[i] = sxy; P.syy_min[i] = syy; P.p_min[i] = p;
        sxx = sxx + h * P.dsxx[i];
        sxy = sxy + h * P.dsxy[i];
        syy = syy + h * P.dsyy[i];
        p = p + h * P.dp[i];
        if (keep_stress) {
            P.p[i] = p; P.sxx[i] = sxx; P.sxy[i] = sxy; P.syy[i] = syy;
        }
    }
    // the last projection is single_step's failure criterion: Mohr-Coulomb
    // when yield_criterion = 1, which may also reset rho (the record then
    // keeps the density before it in chunk 7 for the terms evaluated before
    // the criterion: con_density's delta_sph, strain rate, divergence)
    const double rho_pre = rho;
    if (ndp > 0) {
        int f = 0;
        for (int k = 0; k < ndp; ++k) {
            if (k == ndp - 1 && K.yield_criterion == 1) f = mc_project(K, p, sxx, sxy, syy, rho);
            else f = dp_project(K.s_alpha1, p, sxx, sxy, syy);
        }
        if (keep_stress) {
            P.p[i] = p; P.sxx[i] = sxx; P.sxy[i] = sxy; P.syy[i] = syy;
        }
        P.fail[i] = f;
        if (rho != rho_pre) P.rho[i] = rho;
    }
    const double m = P.mass[i];
    const double irho = 1.0 / rho;
    if (q) {
        float4* Q = reinterpret_cast<float4*>(q) + t;
        const size_t pn = (size_t)P.n;
        write_q01(Q, pn, g, cs, x, y, P.hsml[i], it < 0, vx, vy, rho - K.s_rho0, m, record_cell(NR, t));
        Q[2 * pn] = make_float4((float)P.vof[i], (float)irho, (float)(m * irho), (float)p);
        Q[3 * pn] = make_float4((float)P.c[i], (float)sxx, (float)sxy, (float)syy);
        check_finite(NR.bad, (float)x, (float)y, (float)vx, (float)vy, (float)rho, (float)m, (float)P.vof[i], (float)irho,
                     (float)(m * irho), (float)p, (float)P.c[i], (float)sxx, (float)sxy, (float)syy);
        return;
    }
    double2* R = reinterpret_cast<double2*>(rec) + t;
    const size_t pn = (size_t)P.n;
    R[0 * pn] = make_double2(x, y);
    R[1 * pn] = make_double2(vx, vy);
    const double V = m * irho;
    const double mv = K.learned ? m : V, vof = P.vof[i];
    check_finite(NR.bad, x, y, vx, vy, rho, V, vof * irho, p, P.c[i], sxx, sxy, syy);
    R[2 * pn] = make_double2(rho, it < 0 ? -mv : mv);   // the sign marks a virtual particle
    R[3 * pn] = make_double2(K.learned ? vof : vof * irho, p);
    R[4 * pn] = make_double2(syy, P.c[i]);
    R[5 * pn] = make_double2(sxx, sxy);
    if (!lean) R[6 * pn] = make_double2(P.hsml[i], (double)it);   // (as for water)
    if (K.yield_criterion == 1) R[7 * pn] = make_double2(rho_pre, 0.0);
}

__device__ __forceinline__ void pack_soil_state(const DPhase& P, const KParams& K, double* rec, int t, int i,
                                                int do_half, int ndp, float* q, const Grid& g, double cs,
                                                const NRef& NR)
{
    pack_soil_at(P, K, rec, t, i, do_half, false, false, ndp, q, g, cs, NR, P.x[i], P.y[i], P.rho[i], P.vx[i], P.vy[i], P.p[i],
                 P.sxx[i], P.sxy[i], P.syy[i]);
}

__device__ __forceinline__ void pack_soil_body(int blk, DPhase P, KParams K, double* rec, int do_half, int ndp,
                                               float* q, Grid g, double cs, NRef NR)
{
    const int t = blk * blockDim.x + threadIdx.x;
    if (t < P.n) pack_soil_state(P, K, rec, t, P.order[t], do_half, ndp, q, g, cs, NR);
}

__global__ void k_pack_soil(DPhase P, KParams K, double* rec, int do_half, int ndp, float* q, Grid g, double cs,
                            NRef NR)
{
    pack_soil_body(blockIdx.x, P, K, rec, do_half, ndp, q, g, cs, NR);
}

// The soil final update of step s fused with its pack for step s + 1
// (first_half, two projections), as for water.  The pack reads vof from
// the state: the final update's vof is stored first.
__device__ __forceinline__ void step_soil(int blk, DPhase P, KParams K, double* rec, int first, float* q, Grid g,
                                          double cs, NRef NR)
{
    const int t = blk * blockDim.x + threadIdx.x;
    if (t >= P.n) return;
    const int i = t;   // (lists kept: the state is in record order)
    const SoilEnd e = soil_end(P, K, i, first);
    if (K.volume_fraction && K.two_phase) P.vof[i] = e.vof;
    if (P.itype[i] > 0) {
        P.x[i] = e.x;
        P.y[i] = e.y;
    }
    pack_soil_at(P, K, rec, t, i, 1, q == nullptr, true, 2, q, g, cs, NR, e.x, e.y, e.rho, e.vx, e.vy, e.p, e.sxx, e.sxy, e.syy);
}

__global__ void k_step_soil(DPhase P, KParams K, double* rec, int first, float* q, Grid g, double cs, NRef NR)
{
    step_soil(blockIdx.x, P, K, rec, first, q, g, cs, NR);
}

// ------------------------------------------------------------------------
// Masks of candidates: per particle t a 128-bit mask over its candidate list
// (the three cell rows of its 3 x 3 block, in cell order, concatenated, or its
// index list): m[t] low and m[n + t] high word, and an overflow flag (more
// candidates, or a row of over 64).
// ------------------------------------------------------------------------
struct Masks {
    uint64_t* m;   // [3][n] (the first two words are used)
    int* ovf;      // [n]
};

// ------------------------------------------------------------------------
// Neighbour lists with a skin (fused step).  At a rebuild the cell
// list is built on a grid of cell size >= R + skin (R the largest support
// radius), the records are written in its order, and every particle keeps
// (a) the key of its cell, (b) the candidates within R + skin (same phase and
// cross), as a 128-bit mask over its candidate rows and as a list of indices,
// and (c) its position.  The record order and the cell list then stay fixed
// until the next rebuild.  While no particle has moved more than skin / 2 from
// its rebuild position, every pair within R is listed, so each step tests only
// these candidates with the exact predicate instead of scanning the rows.
// ------------------------------------------------------------------------
// The list: candidates as positions in the window of the workgroup's particles:
// candidate j of record t is the window's record li[j * n + t], cnt[t] of them
// (-1: more than cap, the rows are walked).  win: WIN_INTS per workgroup: the
// first records of the window's three record ranges, their positions in it and
// its length.
struct IdxList {
    unsigned short* li;
    int *cnt, *win;
    int cap, lds;   // lds 0: the windows stay in global memory (predicates that need more than a distance)
    int pb;         // particles of a workgroup of the kernels that read it
    int crowd;      // the list of a crowded particle (mask overflow) counts as overflowed
    int* bad;       // set: a record is not finite, the rows are walked (their terms follow a test)
};

constexpr int WIN_INTS = 8;
constexpr int WIN_CAP = 846;             // records of a window in LDS: two workgroups' six chunks fill a CU's
constexpr int WIN_STRIDE = WIN_CAP + 1;  // (and the stand-in record)
// Lanes of a workgroup that take particles where its window is to fit the LDS (all
// of them otherwise).  The window holds three rows' worth of them: 633 records on
// average (848 at most, and that workgroup reads by lane) for 192 particles of a
// lattice at h = 1.2 dx (whose cell rows hold two or three lattice rows); with 240
// particles one window in four does not fit, and its workgroup takes the slow path
// at the occupancy the LDS leaves (1M slope, soil_ab 117 us against 102, water_b 72
// against 55).
constexpr int WIN_LANES = 192;

struct NList {
    Masks same, cross;   // candidates within R + skin: same phase, other phase
    const int* cell;     // [n] key of the particle's cell at the rebuild (record order)
    IdxList is, ix;      // the candidates as indices: same phase, other phase
    int lg;
};

// ------------------------------------------------------------------------
// Partner iteration.  A particle's candidates are the three cell rows of
// its 3 x 3 block, each a contiguous range [k0, k1) of the cell-sorted
// records.  A scan tests every candidate with the exact predicate and keeps
// one 64-bit mask per row; the three masks are concatenated into one
// 128-bit mask over row0 ++ row1 ++ row2, and the dense loops visit its set
// bits.  A row over 64 candidates, or more than 128 in all, sets the
// overflow flag and that particle walks its rows directly.
// ------------------------------------------------------------------------
struct LaneRows {
    int k0[3], k1[3];
};

__device__ __forceinline__ LaneRows lane_rows(const Rows& R)
{
    LaneRows L;
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        L.k0[r] = R.k0[r];
        L.k1[r] = R.k1[r];
    }
    return L;
}

__device__ __forceinline__ int ovf_of(const LaneRows& L)
{
    int o = 0;
#pragma unroll
    for (int r = 0; r < 3; ++r)
        if (L.k1[r] - L.k0[r] > 64) o |= 1 << r;
    return o;
}

// The three row masks of a lane concatenated into one 128-bit mask over
// the candidate list row0 ++ row1 ++ row2 (at most 128 candidates); a lane
// with more, or with a row over 64, walks its rows directly (ovf = 7).
struct CatMask {
    uint64_t lo, hi;
    int ovf;
};

__device__ __forceinline__ CatMask cat_masks(const LaneRows& L, uint64_t m0, uint64_t m1, uint64_t m2)
{
    const int l0 = L.k1[0] - L.k0[0], l1 = L.k1[1] - L.k0[1], l2 = L.k1[2] - L.k0[2];
    CatMask c;
    c.ovf = (ovf_of(L) || l0 + l1 + l2 > 128) ? 7 : 0;
    if (c.ovf) {
        c.lo = c.hi = 0;
        return c;
    }
    unsigned __int128 v = (unsigned __int128)m2;
    v = (v << l1) | m1;
    v = (v << l0) | m0;
    c.lo = (uint64_t)v;
    c.hi = (uint64_t)(v >> 64);
    return c;
}

// Value select.  A conditional expression over two lvalues (struct fields)
// is itself an lvalue: clang then selects between their addresses and loads
// through the result, which keeps the struct on the stack and puts a
// scratch load on every partner iteration.  Arguments taken by value make
// it a register select.
template <class T>
__device__ __forceinline__ T pick(bool c, T x, T y) { return c ? x : y; }

// Iterator over the set bits of a CatMask; branch-free apart from the loop.
// next() returns the record index of the next partner (-1 at the end).
struct CatIter {
    uint64_t lo, hi;
    int s1, s2;        // start of row 1 and row 2 in the concatenated list
    int e0, e1, e2;    // record index - list index, per row
    __device__ __forceinline__ int next()
    {
        const bool in_lo = lo != 0;
        const uint64_t m = pick(in_lo, lo, hi);
        if (m == 0) return -1;
        const int c = __builtin_ctzll(m) + (in_lo ? 0 : 64);
        const uint64_t rest = m & (m - 1);
        lo = pick(in_lo, rest, lo);
        hi = pick(in_lo, hi, rest);
        const bool a = c < s1, b = c < s2;
        return c + pick(a, e0, pick(b, e1, e2));
    }
};

__device__ __forceinline__ CatIter cat_iter(const CatMask& c, const LaneRows& L)
{
    CatIter it;
    it.lo = c.lo;
    it.hi = c.hi;
    const int l0 = L.k1[0] - L.k0[0], l1 = L.k1[1] - L.k0[1];
    it.s1 = l0;
    it.s2 = l0 + l1;
    it.e0 = L.k0[0];
    it.e1 = L.k0[1] - l0;
    it.e2 = L.k0[2] - l0 - l1;
    return it;
}

// Exact pair predicate on a candidate.
struct Pred {
    double xa, ya, ha, thr;
    int uni, link;
    __device__ __forceinline__ bool operator()(double2 b, double hb, const Grid& g, const KParams& K) const
    {
        const double dx = xa - b.x, dy = ya - b.y;
        double dr;
        {
#pragma clang fp contract(off)
            dr = dx * dx + dy * dy;
        }
        if (!pred(uni != 0, thr, dr, ha, hb, K)) return false;
        return !link || ll_reach(g, xa, ya, b.x, b.y);
    }
};

// The particle and candidate subset of a lane.
struct SubCtx {
    int t, tt, sub;
    bool valid;
};

// Particles of a workgroup whose kernel gives each one lane: those of its window
// with index lists.
__host__ __device__ __forceinline__ int lanes_of_one(const IdxList& I) { return I.li ? I.pb : STAGE_BLOCK; }

// lanes: lanes of the workgroup that take particles (a multiple of 2^lg).
__device__ __forceinline__ SubCtx sub_ctx(int n, int blk, int lg, int lanes)
{
    SubCtx c;
    const int i = (int)threadIdx.x;
    c.t = blk * (lanes >> lg) + (i >> lg);
    c.sub = i & ((1 << lg) - 1);
    c.valid = i < lanes && c.t < n;
    c.tt = c.valid ? c.t : n - 1;
    return c;
}

// Candidate bits of lane sub: every 2^lg-th.
__device__ __forceinline__ uint64_t sub_bits(int lg, int sub)
{
    const uint64_t pat = lg == 0 ? ~0ull : lg == 1 ? 0x5555555555555555ull : lg == 2 ? 0x1111111111111111ull
                                                                                     : 0x0101010101010101ull;
    return pat << sub;
}

__device__ __forceinline__ uint64_t sub_or(int lg, uint64_t v)
{
    for (int o = 1; o < (1 << lg); o <<= 1)
        v |= (uint64_t)__shfl_xor((unsigned long long)v, o, 64);
    return v;
}

__device__ __forceinline__ CatMask mask_of(const Masks& M, int n, int t)
{
    CatMask c;
    c.lo = M.m[t];
    c.hi = M.m[n + t];
    c.ovf = M.ovf[t];
    return c;
}

// Neighbour lists of phase A against phase B (cell list startB on grid g,
// candidate k at state slot ordB[k], or k when ordB is null: the state in
// cell order, as a rebuild leaves it): candidates with dr < thr (thr =
// (R + skin)^2 of the pair type), the particle itself excluded when same.
// Also records each particle's cell key.  Positions come from the state, so
// the FP64 and the FP32 records share the lists.
// The window of a workgroup of the stage kernels (pb consecutive particles):
// their cells are a run of row-major keys [ka, kb], so all their candidates
// lie in the runs [ka - 1, kb + 1] of the row below, the same row and the row
// above -- three contiguous ranges of records, also where the run wraps from
// one grid row into the next.
__device__ __forceinline__ void nlist_body(int blk, const double* xA, const double* yA, const int* ordA, int nA,
                                           const double* xB, const double* yB, const int* ordB, const int* startB,
                                           Grid g, double thr, int same, Masks VM, int* cell, IdxList IL, int pb)
{
    const int t = blk * blockDim.x + threadIdx.x;
    if (t >= nA) return;
    const int ncell = g.ncx * g.ncy;
    auto key_of = [&](int u) {
        const int i = ordA ? ordA[u] : u;
        int cx, cy;
        clamped_cell(g, xA[i], yA[i], cx, cy);
        return cy * g.ncx + cx;
    };
    const int ia = ordA ? ordA[t] : t;
    const double px = xA[ia], py = yA[ia];
    const int key = key_of(t), cy = key / g.ncx, cx = key - cy * g.ncx;
    if (cell) cell[t] = key;
    const int wb = t / pb, ka = key_of(wb * pb), kb = key_of(min(nA, (wb + 1) * pb) - 1);
    int lo[3], off[3], tot = 0;
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        const int a = max(ka + (r - 1) * g.ncx - 1, 0), b = min(kb + (r - 1) * g.ncx + 1, ncell - 1);
        lo[r] = a <= b ? startB[a] : 0;
        off[r] = tot;
        tot += a <= b ? startB[b + 1] - lo[r] : 0;
    }
    if (t == wb * pb) {
        int* w = IL.win + (size_t)wb * WIN_INTS;
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            w[r] = lo[r];
            w[3 + r] = off[r];
        }
        w[6] = tot;
    }
    const LaneRows L = lane_rows(block_rows_at(g, startB, cx, cy));
    auto acc = [&](int k) {
        const int ib = ordB ? ordB[k] : k;
        const double dx = px - xB[ib], dy = py - yB[ib];
        return dx * dx + dy * dy < thr;
    };
    const int self = same ? t : -1;
    uint64_t m[3];
    int cnt = 0;
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        const int k0 = r == 0 ? L.k0[0] : (r == 1 ? L.k0[1] : L.k0[2]);
        const int k1 = r == 0 ? L.k1[0] : (r == 1 ? L.k1[1] : L.k1[2]);
        uint64_t mm = 0;
#pragma unroll 4
        for (int k = k0; k < k1; ++k) {
            const bool ok = k != self && acc(k);
            if (k - k0 < 64) mm |= (uint64_t)ok << (k - k0);
            if (ok) {
                if (cnt < IL.cap) IL.li[(size_t)cnt * nA + t] = (unsigned short)(off[r] + (k - lo[r]));
                ++cnt;
            }
        }
        m[r] = k1 - k0 <= 64 ? mm : 0;
    }
    const CatMask cm = cat_masks(L, m[0], m[1], m[2]);
    VM.m[t] = cm.lo;
    VM.m[nA + t] = cm.hi;
    VM.ovf[t] = cm.ovf;
    IL.cnt[t] = cnt <= IL.cap && tot < 65536 && !(IL.crowd && cm.ovf) ? cnt : -1;
}

__global__ __launch_bounds__(256) void k_nlist(const double* xA, const double* yA, const int* ordA, int nA,
                                               const double* xB, const double* yB, const int* ordB, const int* startB,
                                               Grid g, double thr, int same, Masks VM, int* cell, IdxList IL, int pb)
{
    nlist_body(xcd_block(), xA, yA, ordA, nA, xB, yB, ordB, startB, g, thr, same, VM, cell, IL, pb);
}

// ------------------------------------------------------------------------
// Partner visit of the FP64 stage kernels.
//
// In list mode with a uniform smoothing length a workgroup first copies its
// window's record chunks into LDS, then every lane goes through its list,
// reading the partners there (the next partner's chunks in flight beside the
// current one's terms); candidates outside the support (about one in six, in
// the skin) are evaluated with W = s = 0 (once a record holds an infinity or a
// NaN, which would count so, the rows are walked instead).  What bound the gathers from global
// memory was the L1's tag lookups: a 64-lane 16-byte gather of such partners
// takes 34 of them (one per cycle and CU; 16 for contiguous lanes), where the
// same LDS read takes about 8 cycles.  The copy itself is contiguous.  What
// bounds the kernels now is the latency of the copy and of the particles' own
// loads at two to four workgroups per CU (without the partner loop soil_ab still
// takes 55 us of 102).  1M slope, us per launch, gathers from global memory
// through 128-bit masks -> this: soil_ab 130 -> 102, soil_x 82 -> 77, water_a
// 69 -> 48, water_b 73 -> 55, water_x 64 -> 50.
//
// Otherwise (no lists, smoothing lengths that vary, link_list's reach, a
// window that does not fit): the candidates are the particle's list, or its
// three candidate rows.  Four at a time their positions are tested with the
// exact predicate, into a mask of 128 candidates in registers, and the dense loop
// goes through its bits (water stage B takes the mask of stage A: with a test of its
// own 72 us against 42 for 250k particles with varying h).  One lane per particle
// starts from the rebuild's mask of listed candidates, whose rows it can index
// without a load (900k particles with varying h: 476 us per step, through the index
// list 557).
// ------------------------------------------------------------------------
// The forms of a stage kernel: WINDOWS as described, UNIFORM one smoothing length
// for all pairs but no windows in LDS (no lists, or link_list's reach), VARYING
// smoothing lengths that vary, GENERAL other than integer repulsion exponents or
// Drucker-Prager (pow and the Mohr-Coulomb terms in the pair loop are 47 registers
// of soil_ab's 204).  All but WINDOWS keep all lanes of a workgroup and take no
// LDS.  250k slope, us per step, with the windows' LDS and lanes for all -> this:
// varying h 248 -> 157, link_list 153 -> 114, lists off 231 -> 172 (both 335 -> 237),
// Mohr-Coulomb 164 -> 138, real exponents 177 -> 141.
enum : int { GENERAL, VARYING, UNIFORM, WINDOWS };

// Record index of a position of three concatenated ranges: starts s1 and s2
// of the second and third, record index - position in each.
struct Ranges3 {
    int s1, s2, e0, e1, e2;
    __device__ __forceinline__ int operator()(int i) const { return i + pick(i < s1, e0, pick(i < s2, e1, e2)); }
};

// Where a particle's candidates come from: its list, or (none, or one that
// overflowed: walk) the candidate rows of its cell.
struct Cand {
    const Grid& g;
    const int *cell_start, *cell;   // cell: key at the rebuild (null: the current position's)
    double xa, ya;
    __device__ __forceinline__ Ranges3 rows(int tt, int& tot) const
    {
        int cx, cy;
        if (cell) {
            const int key = cell[tt];
            cy = key / g.ncx;
            cx = key - cy * g.ncx;
        } else {
            clamped_cell(g, xa, ya, cx, cy);
        }
        const Rows R = block_rows_at(g, cell_start, cx, cy);
        Ranges3 r;
        r.s1 = R.k1[0] - R.k0[0];
        r.s2 = r.s1 + R.k1[1] - R.k0[1];
        tot = r.s2 + R.k1[2] - R.k0[2];
        r.e0 = R.k0[0];
        r.e1 = R.k0[1] - r.s1;
        r.e2 = R.k0[2] - r.s2;
        return r;
    }
};

__device__ __forceinline__ Ranges3 window_ranges(const int* w)
{
    return Ranges3{w[4], w[5], w[0], w[1] - w[4], w[2] - w[5]};
}

// A workgroup's window while its kernel runs.
struct Window {
    Ranges3 r;
    bool listed, lds;   // a list exists; the window is in LDS (or on its way)
    int cnt, k[4];      // the lane's list length (-1: rows) and, lds, its first entries
};

// The candidates sub, sub + 2^lg, ... of a particle from global memory:
// body(v, rec, k) for each that passes accept(k, xy), in order; self: own
// record index in the candidates' phase (-1: none).  All lanes of the wave call.
// KEEP: stores the mask of a particle's partners in MW (ovf: more than 128
// candidates); GIVEN: takes it from there instead of testing again.
enum : int { TEST, KEEP, GIVEN };

template <int NCH, int MODE, class A, class B>
__device__ __forceinline__ void visit_global(const Cand& C, const IdxList& I, const Window& w, int n, const SubCtx& sc,
                                             int lg, int self, const RecV& rec, const Masks& LM, const Masks& MW,
                                             A&& accept, B&& body)
{
    CatMask kept{0, 0, 1}, listed{0, 0, 1};
    if (MODE == GIVEN) kept = mask_of(MW, n, sc.tt);
    if (LM.m && lg == 0) listed = mask_of(LM, n, sc.tt);   // (several lanes: the list deals evenly)
    int tot = -1;
    if (w.listed && listed.ovf) tot = I.cnt[sc.tt];
    const bool by_row = tot < 0;
    Ranges3 rows = w.r;
    if (by_row) rows = C.rows(sc.tt, tot);
    if (!sc.valid) tot = 0;
    auto at = [&](int i) { return rows(by_row ? i : (int)I.li[(size_t)i * n + sc.tt]); };
#pragma unroll 1
    for (int base = 0; base < tot; base += 128) {
        const int end = min(tot - base, 128);
        uint64_t lo = 0, hi = 0;
        auto test = [&](const int(&c)[4]) {
            int k[4];
            double2 p[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) k[q] = at(base + c[q]);
#pragma unroll
            for (int q = 0; q < 4; ++q) p[q] = rec(k[q], 0);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint64_t bit = (uint64_t)(k[q] != self && accept(k[q], p[q])) << (c[q] & 63);
                lo |= pick(c[q] < 64, bit, (uint64_t)0);
                hi |= pick(c[q] < 64, (uint64_t)0, bit);
            }
        };
        if (MODE == GIVEN && !kept.ovf) {
            lo = kept.lo & sub_bits(lg, sc.sub);
            hi = kept.hi & sub_bits(lg, sc.sub);
        } else if (!listed.ovf) {
            uint64_t clo = listed.lo & sub_bits(lg, sc.sub), chi = listed.hi & sub_bits(lg, sc.sub);
            while (clo | chi) {
                int c[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {   // (past the last one: it again)
                    const bool in_lo = clo != 0;
                    const uint64_t m = pick(in_lo, clo, chi);
                    c[q] = m ? __builtin_ctzll(m) + (in_lo ? 0 : 64) : q ? c[q - 1] : 0;
                    const uint64_t rest = m & (m - 1);
                    clo = pick(in_lo, rest, clo);
                    chi = pick(in_lo, chi, rest);
                }
                test(c);
            }
        } else {
#pragma unroll 1
            for (int j = sc.sub; j < end; j += 4 << lg) {
                int c[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) c[q] = j + (q << lg) < end ? j + (q << lg) : j;
                test(c);
            }
        }
        if (MODE == KEEP) {
            kept.lo = lo;
            kept.hi = hi;
        }
        auto next = [&]() -> int {
            const bool in_lo = lo != 0;
            const uint64_t m = pick(in_lo, lo, hi);
            if (m == 0) return -1;
            const int i = __builtin_ctzll(m) + (in_lo ? 0 : 64);
            const uint64_t rest = m & (m - 1);
            lo = pick(in_lo, rest, lo);
            hi = pick(in_lo, hi, rest);
            return at(base + i);
        };
        int ahead = next();
#pragma unroll 1
        while (ahead >= 0) {
            const int k = ahead;
            double2 v[NCH];
#pragma unroll
            for (int ch = 0; ch < NCH; ++ch) v[ch] = rec(k, ch);
            ahead = next();
            body(v, rec, k);
        }
    }
    if (MODE == KEEP) {
        kept.lo = sub_or(lg, kept.lo);
        kept.hi = sub_or(lg, kept.hi);
        if (sc.valid && !sc.sub) {
            MW.m[sc.t] = kept.lo;
            MW.m[n + sc.t] = kept.hi;
            MW.ovf[sc.t] = tot > 128 ? 1 : 0;
        }
    }
}

// LDS of a stage kernel that reads NCH chunks per partner.
template <int NCH>
constexpr size_t VIS_LDS = sizeof(double2) * NCH * WIN_STRIDE;
template <int FORM, int NCH>
constexpr size_t STAGE_LDS = FORM == WINDOWS ? VIS_LDS<NCH> : sizeof(double2);

// Sends chunks 0 .. NCH - 1 of the workgroup's window on their way into LDS
// (straight from global memory, no registers: all of it is in flight at once),
// and a stand-in record (far away, finite everywhere) at WIN_CAP.  Called after
// a kernel's own loads: loads return in order, so a use of one issued behind
// the window would wait for all of it.
template <bool WIN, int NCH, class R>
__device__ __forceinline__ Window open_window(unsigned char* lds, const IdxList& I, int blk, const SubCtx& sc, int lg,
                                              int n, const R& rec)
{
    typedef typename R::V V;
    Window w{{0, 0, 0, 0, 0}, I.li != nullptr, false, 0, {0, 0, 0, 0}};
    if (!I.li) return w;
    const int* p = I.win + (size_t)blk * WIN_INTS;
    w.r = window_ranges(p);
    if constexpr (WIN) {
        const int tot = p[6];
        w.lds = I.lds && tot <= WIN_CAP;
        // (kernels beside this one may raise bad: read once, by lane; w.lds, on which
        // a barrier depends, is the workgroup's)
        w.cnt = __hip_atomic_load(I.bad, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ? -1 : I.cnt[sc.tt];
        if (w.lds) {
            const uint32_t o = (uint32_t)sc.sub * n + sc.tt;
            const size_t row = (size_t)n << lg;
#pragma unroll
            for (int q = 0; q < 4; ++q) w.k[q] = I.li[q * row + o];
            V* wl = reinterpret_cast<V*>(lds);
            if (threadIdx.x < NCH) wl[threadIdx.x * WIN_STRIDE + WIN_CAP] = R::stand_in(threadIdx.x);
            const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x & ~63);
            for (int i0 = wave; i0 < tot; i0 += STAGE_BLOCK) {
                const int i = i0 + (int)(threadIdx.x & 63);
                if (i < tot) {
                    const uint32_t at = (uint32_t)w.r(i) << 4;
#pragma unroll
                    for (int c = 0; c < NCH; ++c)
                        __builtin_amdgcn_global_load_lds(
                            (const __attribute__((address_space(1))) void*)(reinterpret_cast<const char*>(
                                                                                rec.p + (size_t)c * rec.n) + at),
                            (__attribute__((address_space(3))) void*)(wl + c * WIN_STRIDE + i0), 16, 0, 0);
                }
            }
        }
    }
    return w;
}

// body(v) over the listed candidates of the lane's particle, v the record
// chunks 0 .. NCH - 1 from the window in LDS (all lanes of the workgroup call;
// none of a list that overflowed).
template <int NCH, class V, class B>
__device__ __forceinline__ void visit_window(unsigned char* lds, const Window& w, const IdxList& I, int n,
                                             const SubCtx& sc, int lg, B&& body)
{
    const V* wl = reinterpret_cast<const V*>(lds);
    auto read = [&](V(&v)[NCH], int k) {
#pragma unroll
        for (int c = 0; c < NCH; ++c) v[c] = wl[c * WIN_STRIDE + k];
    };
    // The lane's candidates i = 0, 1, ... are sub, sub + 2^lg, ... of
    // the list; past its end the stand-in.  Indices are loaded two
    // rounds ahead (the buffer is padded), chunks one.
    const unsigned short* l = I.li;
    const uint32_t o = (uint32_t)sc.sub * n + sc.tt;
    const size_t row = (size_t)n << lg;
    int k0 = w.k[0], k1 = w.k[1], n0 = w.k[2], n1 = w.k[3];
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    const int mine = sc.valid ? (max(w.cnt, 0) - sc.sub + (1 << lg) - 1) >> lg : 0;
    V a[NCH], b[NCH];
    read(a, pick(0 < mine, k0, WIN_CAP));
    k1 = pick(1 < mine, k1, WIN_CAP);
#pragma unroll 1
    for (int i = 0; __any(i < mine); i += 2) {
        l += 2 * row;
        k0 = pick(i + 2 < mine, n0, WIN_CAP);
        const int k2 = pick(i + 3 < mine, n1, WIN_CAP);
        n0 = l[2 * row + o];
        n1 = l[3 * row + o];
        read(b, k1);
        body(a);
        read(a, k0);
        k1 = k2;
        body(b);
    }
}

// body(v, R, k) over the partners of the lane's particle, v the record chunks
// 0 .. NCH - 1 and R(k, c) any other (all lanes of the workgroup call).
template <bool WIN, int NCH, int MODE = TEST, class A, class B>
__device__ __forceinline__ void visit(unsigned char* lds, const Window& w, const Cand& C, const IdxList& I, int n,
                                      const SubCtx& sc, int lg, int self, const RecV& rec, const Masks& LM,
                                      A&& accept, B&& body, const Masks& MW = Masks{})
{
    // (a window that does not fit: several lanes go through the list at once, as
    // through a window, one lane tests it first: savage column of 2k 3.24 ms for 100
    // steps against 3.39, 250k slope 11.4 against 11.8)
    if (WIN && (w.lds || lg > 0)) {
        if (w.lds) visit_window<NCH, double2>(lds, w, I, n, sc, lg, [&](const auto& v) { body(v, rec, 0); });
        // a particle whose list overflowed walks its rows
        int tot = w.lds ? min(w.cnt, 0) : w.cnt;
        const bool walk = tot < 0;
        Ranges3 rows = w.r;
        if (walk) rows = C.rows(sc.tt, tot);
        if (!sc.valid) tot = 0;
        auto at = [&](int i) { return rows(walk || i >= tot ? i : (int)I.li[(size_t)i * n + sc.tt]); };
        int next = at(sc.sub);
#pragma unroll 1
        for (int i = sc.sub; i < tot; i += 1 << lg) {
            const int k = next;
            next = at(i + (1 << lg));
            if (walk && (k == self || !accept(k, rec(k, 0)))) continue;
            double2 v[NCH];
#pragma unroll
            for (int c = 0; c < NCH; ++c) v[c] = rec(k, c);
            body(v, rec, k);
        }
        return;
    }
    visit_global<NCH, MODE>(C, I, w, n, sc, lg, self, rec, LM, MW, accept, body);
}

// ------------------------------------------------------------------------
// Pair terms.  With grad W = s d (d the separation) every product of a
// stage is a combination of s, d, the velocity difference u and vr = u.d:
// u.grad W = s vr, and delta_sph's 2 (d.grad W) / d^2 = 2 s.  Records hold the
// partner's volume V = m / rho, so V s d and m = V rho replace its
// reciprocals.
// ------------------------------------------------------------------------
struct Sep {
    double dx, dy, dr, ir, w, s;
    bool in;
};

// thr: W = s = 0 at and beyond dr = thr (the exact predicate of a uniform
// smoothing length; listed candidates may lie outside the support).
template <int SKF, bool NEED_W>
__device__ __forceinline__ Sep sep_of(const KC& kc, double dx, double dy, double thr, bool coincident)
{
    Sep p;
    p.dx = dx;
    p.dy = dy;
    {
#pragma clang fp contract(off)
        p.dr = dx * dx + dy * dy;
    }
    // (co-located particles of two phases: W(0), no gradient direction)
    p.ir = coincident && !(p.dr > 0.0) ? 0.0 : fast_rsq(p.dr);
    kern_s<SKF, NEED_W>(kc, p.dr * p.ir, p.ir, p.w, p.s);
    p.in = p.dr < thr;
    p.s = p.in ? p.s : 0.0;
    if (NEED_W) p.w = p.in ? p.w : 0.0;
    return p;
}

// ------------------------------------------------------------------------
// Cross terms, water side (stage A of single_step's interaction block,
// declarations_sph.f90:1380-1410): darcy_law's drag on the water,
// volume_fraction_water2's dvof and volume_fraction_water's vof2 from the
// soil partners (direct_find_2's pairs, virtual x virtual and r = 0
// included).  Its own kernel: the loop needs few registers, so it runs at
// twice the occupancy of the same-phase stage.
// lean (all stages): another step of the same call follows and this one does
// not renormalise (its final update reads vof2), so the values that only a
// download or the last step's diagnostics would read stay out.
// ------------------------------------------------------------------------
template <int SKF, int FORM>
__device__ __forceinline__ void water_x4(unsigned char* lds, int blk, DPhase W, DPhase S, const double* recW, const double* recS,
                                         NList NL, Grid g, KParams K, FusedK F, int lean)
{
    constexpr bool U = FORM >= UNIFORM, WIN = FORM == WINDOWS;
    const RecV RW = recv(recW, W.n), RS = recv(recS, S.n);
    const SubCtx wc = sub_ctx(W.n, blk, NL.lg, NL.ix.pb << NL.lg);
    const double2 xy = RW(wc.tt, 0), va = RW(wc.tt, 1);
    const double xa = xy.x, ya = xy.y, vxa = va.x, vya = va.y, vofa = RW(wc.tt, 3).x;
    const double ha = U ? K.h1_water : RW(wc.tt, 6).x;
    const int a = NL.cell ? wc.tt : W.order[wc.tt];
    const bool ux = U || F.uni_x;
    const Window win = open_window<WIN, 4>(lds, NL.ix, blk, wc, NL.lg, W.n, RS);
    const Cand C{g, S.cell_start, NL.cell, xa, ya};
    const Pred PX{xa, ya, ha, F.thr_x, ux ? 1 : 0, 0};
    const KC kx = make_kc(SKF, sph_mhsml(ha, ux ? RS(0, 6).x : ha));
    double dg_x = 0.0, dg_y = 0.0, dvof_x = 0.0, vof2 = 0.0;
    int cntx = 0;
    visit<WIN, 4>(
        lds, win, C, NL.ix, W.n, wc, NL.lg, -1, RS, NL.cross, [&](int k, double2 b) { return PX(b, ux ? ha : RS(k, 6).x, g, K); },
        [&](const auto& v, const auto& R, int k) {
            const double2 b = v[0], u = v[1], q = v[2];
            const double vr_b = v[3].x;   // vof / rho
            KC kc = kx;
            if (!ux) kc = pair_kc<SKF>(sph_mhsml(ha, R(k, 6).x));
            const Sep p = sep_of<SKF, true>(kc, xa - b.x, ya - b.y, U ? F.thr_x : INFINITY, true);
            cntx += p.in ? 1 : 0;
            const double m = fabs(q.y) * q.x, mw = m * p.w;
            const double dvx = vxa - u.x, dvy = vya - u.y;
            const double sc = mw * vr_b;
            dg_x += sc * dvx;
            dg_y += sc * dvy;
            dvof_x += (m * p.s) * (dvx * p.dx + dvy * p.dy);
            vof2 += mw;
        });
    sub_sum(NL.lg, dg_x, dg_y, dvof_x, vof2);
    cntx = sub_count(NL.lg, cntx);
    if (!wc.valid || wc.sub) return;
    // vof_a vof_b rho_a (-g) / perm * W / (rho_a rho_b): rho_a cancels
    const double cfa = vofa * (-K.numeric_gravity) / K.s_perm;
    W.drgx[a] = cfa * dg_x;
    W.drgy[a] = cfa * dg_y;
    W.dvof_x[a] = dvof_x * (1.0 / K.s_rho0);
    if (!lean) {
        W.vof2[a] = 1.0 - vof2 / K.s_rho0;
        W.countiac[a] = cntx;
    }
}

template <int SKF, int FORM>
__global__ STAGE_ATTR void k_water_x4(DPhase W, DPhase S, const double* recW, const double* recS, NList NL, Grid g,
                                      KParams K, FusedK F, int lean)
{
    __shared__ __align__(16) unsigned char lds[STAGE_LDS<FORM, 4>];
    water_x4<SKF, FORM>(lds, xcd_block(), W, S, recW, recS, NL, g, K, F, lean);
}

// ------------------------------------------------------------------------
// Cross terms, soil side: darcy_law's drag on the soil and
// pore_water_pressure (m_particles.f90:3832-3909) from the water partners
// (whose pressure is the new one the water pack evaluated).
// ------------------------------------------------------------------------
template <int SKF, int FORM>
__device__ __forceinline__ void soil_x4(unsigned char* lds, int blk, DPhase S, DPhase W, const double* recS, const double* recW, NList NL,
                                        Grid g, KParams K, FusedK F, int lean)
{
    constexpr bool U = FORM >= UNIFORM, WIN = FORM == WINDOWS;
    const RecV RS = recv(recS, S.n), RW = recv(recW, W.n);
    const SubCtx wc = sub_ctx(S.n, blk, NL.lg, NL.ix.pb << NL.lg);
    const double2 xy = RS(wc.tt, 0), va = RS(wc.tt, 1);
    const double xa = xy.x, ya = xy.y, vxa = va.x, vya = va.y;
    const double vra = RS(wc.tt, 3).x;   // vof / rho
    const double ha = U ? K.h1_soil : RS(wc.tt, 6).x;
    const int a = NL.cell ? wc.tt : S.order[wc.tt];
    const bool ux = U || F.uni_x;
    const Window win = open_window<WIN, 4>(lds, NL.ix, blk, wc, NL.lg, S.n, RW);
    const Cand C{g, W.cell_start, NL.cell, xa, ya};
    const Pred PX{xa, ya, ha, F.thr_x, ux ? 1 : 0, 0};
    const KC kx = make_kc(SKF, sph_mhsml(ux ? RW(0, 6).x : ha, ha));
    double dg_x = 0.0, dg_y = 0.0, po_x = 0.0, po_y = 0.0;
    int cntx = 0;
    visit<WIN, 4>(
        lds, win, C, NL.ix, S.n, wc, NL.lg, -1, RW, NL.cross, [&](int k, double2 b) { return PX(b, ux ? ha : RW(k, 6).x, g, K); },
        [&](const auto& v, const auto& R, int k) {
            const double2 b = v[0], u = v[1], q = v[2], f = v[3];   // f = (vof, p)
            KC kc = kx;
            if (!ux) kc = pair_kc<SKF>(sph_mhsml(R(k, 6).x, ha));
            // water - soil
            const Sep p = sep_of<SKF, true>(kc, b.x - xa, b.y - ya, U ? F.thr_x : INFINITY, true);
            cntx += p.in ? 1 : 0;
            const double V = fabs(q.y);
            // m_w vof_w rho_w W / (rho_w rho_s): the soil's factors outside
            const double sc = (V * q.x) * (f.x * p.w);
            dg_x += sc * (u.x - vxa);
            dg_y += sc * (u.y - vya);
            const double vp = (V * f.y) * p.s;
            po_x += vp * p.dx;
            po_y += vp * p.dy;
        });
    sub_sum(NL.lg, dg_x, dg_y, po_x, po_y);
    cntx = sub_count(NL.lg, cntx);
    if (!wc.valid || wc.sub) return;
    const double cfs = vra * (-K.numeric_gravity) / K.s_perm;
    S.drgx[a] = cfs * dg_x;
    S.drgy[a] = cfs * dg_y;
    S.porx[a] = vra * po_x;
    S.pory[a] = vra * po_y;
    if (!lean) S.countiac[a] = cntx;
}

template <int SKF, int FORM>
__global__ STAGE_ATTR void k_soil_x4(DPhase S, DPhase W, const double* recS, const double* recW, NList NL, Grid g,
                                     KParams K, FusedK F, int lean)
{
    __shared__ __align__(16) unsigned char lds[STAGE_LDS<FORM, 4>];
    soil_x4<SKF, FORM>(lds, xcd_block(), S, W, recS, recW, NL, g, K, F, lean);
}

// repulsive_force on a real particle from a virtual partner within r0
// (m_particles.f90:1605): D ((r0/r)^p1 - (r0/r)^p2) d / r^2; ir = 1/r.
template <bool INT>
__device__ __forceinline__ double rep_factor(const KParams& K, double r0, double ir)
{
    const double q = r0 * ir;
    return K.dd * (INT ? ipow(q, K.ip1) - ipow(q, K.ip2) : pow(q, K.p1) - pow(q, K.p2)) * (ir * ir);
}

// ------------------------------------------------------------------------
// Stage A, water: same-phase terms (con_density, delta_sph(rho),
// shear_strain_rate, av_vel, repulsive_force), then pressure() per particle.
// Writes a-space outputs and the record slots vof*sigma for stage B.  cross:
// two-phase run (countiac then counts the soil partners, which k_water_x4
// writes).
// ------------------------------------------------------------------------
template <int SKF, int FORM>
__device__ __forceinline__ void water_a4(unsigned char* lds, int blk, DPhase W, const double* recW, double* recWw, NList NL, Masks MW,
                                         Grid g, KParams K, FusedK F, int cross, int lean)
{
    constexpr bool U = FORM >= UNIFORM, WIN = FORM == WINDOWS;
    const RecV RW = recv(recW, W.n);
    const SubCtx wc = sub_ctx(W.n, blk, NL.lg, NL.is.pb << NL.lg);
    const int t = wc.t;
    auto RA = [&](int c) { return RW(wc.tt, c); };
    const double2 xy = RA(0), va = RA(1);
    const bool link = K.nnps == 2;
    // U (checked by the host): h uniform in the phase (hsml(1) everywhere, a
    // wave-uniform value), integer repulsion exponents
    const double xa = xy.x, ya = xy.y, vxa = va.x, vya = va.y, rhoa = RA(2).x, vofa = RA(3).x;
    const double ha = U ? K.h1_water : RA(6).x;
    const int a = NL.cell ? wc.tt : W.order[wc.tt];
    const double ca = W.c[a];
    const bool uni = U || link || F.uni_w;
    const KC kc0 = make_kc(SKF, link ? K.h1_water : ha);
    const int ita = W.itype[a];
    const Window win = open_window<WIN, 3>(lds, NL.is, blk, wc, NL.lg, W.n, RW);
    const Cand C{g, W.cell_start, NL.cell, xa, ya};
    const Pred P{xa, ya, ha, F.thr_w, uni ? 1 : 0, link ? 1 : 0};
    const double rep2 = ita > 0 ? W.dspp * W.dspp : -1.0;   // real particles feel the wall
    double con = 0.0, drd = 0.0, xx = 0.0, yy = 0.0, xy2 = 0.0, avx = 0.0, avy = 0.0, repx = 0.0, repy = 0.0;
    int cnt = 0;
    visit<WIN, 3, KEEP>(
        lds, win, C, NL.is, W.n, wc, NL.lg, t, RW, NL.same, [&](int k, double2 b) { return P(b, uni ? ha : RW(k, 6).x, g, K); },
        [&](const auto& v, const auto& R, int k) {
            const double2 b = v[0], u = v[1], q = v[2];
            KC kc = kc0;
            if (!uni) kc = pair_kc<SKF>(sph_mhsml(ha, R(k, 6).x));
            const Sep p = sep_of<SKF, true>(kc, xa - b.x, ya - b.y, U ? F.thr_w : INFINITY, false);
            cnt += p.in ? 1 : 0;
            const double V = fabs(q.y), dvx = vxa - u.x, dvy = vya - u.y, vr = dvx * p.dx + dvy * p.dy;
            const double Vs = V * p.s, wx = Vs * p.dx, wy = Vs * p.dy;
            con += (Vs * q.x) * vr;
            drd += Vs * (rhoa - q.x);
            xx += wx * dvx;
            yy += wy * dvy;
            xy2 += wy * dvx;
            xy2 += wx * dvy;
            const double f = (V * q.x) * (p.w * fast_rcp(rhoa + q.x));
            avx -= f * dvx;
            avy -= f * dvy;
            if (q.y < 0.0 && p.dr <= rep2 && p.in) {
                const double fr = rep_factor<FORM != GENERAL>(K, W.dspp, p.ir);
                repx += p.dx * fr;
                repy += p.dy * fr;
            }
        }, MW);
    sub_sum(NL.lg, con, drd, xx, yy, xy2, avx, avy, repx, repy);
    cnt = sub_count(NL.lg, cnt);
    if (!wc.valid || wc.sub) return;
    const double mu = K.w_mu;
    const double txx = SPH_C23_F * (yy - 2.0 * xx), tyy = SPH_C23_F * (xx - 2.0 * yy), txy = -xy2;
    // delta_sph(rho) and av_vel only under their switches (artificial_density,
    // average_velocity); without av_vel the reference leaves av as it was
    W.drho[a] = K.artificial_density ? con + (K.delta * ha * ca) * (2.0 * drd) : con;
    if (K.average_velocity) {
        const double e = ita > 0 ? 2.0 * K.epsilon : 2.0;
        W.avx[a] = e * avx;
        W.avy[a] = e * avy;
    }
    W.repx[a] = repx;
    W.repy[a] = repy;
    if (!lean) {
        W.txx[a] = txx;
        W.txy[a] = txy;
        W.tyy[a] = tyy;
        if (!cross) W.countiac[a] = cnt;
        W.nsame[a] = cnt;
    }
    // p and the new c (chunks 3 and 4) come from the pack
    double2* WP = reinterpret_cast<double2*>(recWw) + t;
    const size_t nw = (size_t)W.n;
    reinterpret_cast<double*>(WP + 4 * nw)[0] = vofa * (mu * tyy);
    WP[5 * nw] = make_double2(vofa * (mu * txx), vofa * (mu * txy));
    if (WIN) check_finite(NL.is.bad, txx, txy, tyy);   // (stage B reads them)
}

template <int SKF, int FORM>
__global__ STAGE_ATTR void k_water_a4(DPhase W, const double* recW, double* recWw, NList NL, Masks MW, Grid g,
                                      KParams K, FusedK F, int cross, int lean)
{
    __shared__ __align__(16) unsigned char lds[STAGE_LDS<FORM, 3>];
    water_a4<SKF, FORM>(lds, xcd_block(), W, recW, recWw, NL, MW, g, K, F, cross, lean);
}

// ------------------------------------------------------------------------
// Stage B, water: -vof*df(p) + df(vof*sigma) (declarations_sph.f90:1257-1265),
// art_visc, delta_sph(vof, dvof); /rho, + repulsion, + gravity, - Darcy drag.
// ------------------------------------------------------------------------
template <int SKF, int FORM>
__device__ __forceinline__ void water_b4(unsigned char* lds, int blk, DPhase W, const double* recW, NList NL, Masks MW, Grid g,
                                         KParams K, FusedK F, int mask)
{
    constexpr bool U = FORM >= UNIFORM, WIN = FORM == WINDOWS;
    const RecV RW = recv(recW, W.n);
    const SubCtx wc = sub_ctx(W.n, blk, NL.lg, NL.is.pb << NL.lg);
    const int t = wc.t;
    auto RA = [&](int c) { return RW(wc.tt, c); };
    const double2 axy = RA(0), av = RA(1), arv = RA(2), a3 = RA(3), a4 = RA(4), a12 = RA(5);
    // U: h uniform in the phase (checked by the host)
    const double xa = axy.x, ya = axy.y, vxa = av.x, vya = av.y, rhoa = arv.x, vofa = a3.x;
    const double ha = U ? K.h1_water : RA(6).x;
    const double pa = a3.y, ca = a4.y;
    const int a = NL.cell ? wc.tt : W.order[wc.tt];
    const bool link = K.nnps == 2;
    const bool uni = U || link || F.uni_w;
    const KC kc0 = make_kc(SKF, link ? K.h1_water : ha);
    // (the tail's inputs, loaded before the loop)
    const double repx = W.repx[a], repy = W.repy[a];
    double drgx = 0.0, drgy = 0.0, dvx = 0.0;
    if (mask & M_CROSS) {
        drgx = W.drgx[a];
        drgy = W.drgy[a];
        dvx = W.dvof_x[a];
    }
    const Window win = open_window<WIN, 6>(lds, NL.is, blk, wc, NL.lg, W.n, RW);
    const Cand C{g, W.cell_start, NL.cell, xa, ya};
    const Pred P{xa, ya, ha, F.thr_w, uni ? 1 : 0, link ? 1 : 0};
    const double et2 = K.etq * K.etq;
    double Wx = 0.0, Wy = 0.0, Fx = 0.0, Fy = 0.0, artx = 0.0, arty = 0.0, dvd = 0.0;
    visit<WIN, 6, GIVEN>(
        lds, win, C, NL.is, W.n, wc, NL.lg, t, RW, NL.same, [&](int k, double2 b) { return P(b, uni ? ha : RW(k, 6).x, g, K); },
        [&](const auto& v, const auto& R, int k) {
            const double2 b = v[0], u = v[1], q = v[2], f = v[3], s3 = v[4], s12 = v[5];
            KC kc = kc0;
            double amh = ha;
            if (!uni) {
                amh = sph_mhsml(ha, R(k, 6).x);
                kc = pair_kc<SKF>(amh);
            }
            const Sep p = sep_of<SKF, false>(kc, xa - b.x, ya - b.y, U ? F.thr_w : INFINITY, false);
            const double Vs = fabs(q.y) * p.s, wx = Vs * p.dx, wy = Vs * p.dy;
            const double vr = (vxa - u.x) * p.dx + (vya - u.y) * p.dy;
            // -vof_a (p_a + p_b) + (f_a + f_b) as twice the own value (outside,
            // times the sum of V grad W) plus the difference, which is small
            // where the sum is not: fewer digits cancel in the total
            const double dp = f.y - pa, fxy = a12.y + s12.y;
            Wx = fma(Vs, p.dx, Wx);
            Wy = fma(Vs, p.dy, Wy);
            Fx += ((s12.x - a12.x) - vofa * dp) * wx;
            Fx += fxy * wy;
            Fy += ((s3.x - a4.x) - vofa * dp) * wy;
            Fy += fxy * wx;
            {   // art_visc, branch-free: approaching pairs only (vr < 0)
                const double rs = rhoa + q.x, d2 = p.dr + amh * amh * et2;
                const double it = fast_rcp(rs * d2), hv = amh * vr, muv = hv * (it * rs);
                const double piv = (K.beta * muv - 0.5 * K.alpha * (ca + s3.y)) * (hv * it);
                const double mp = vr < 0.0 ? (Vs * q.x) * piv : 0.0;
                artx -= mp * p.dx;
                arty -= mp * p.dy;
            }
            dvd += Vs * (vofa - f.x);
        }, MW);
    sub_sum(NL.lg, Wx, Wy, Fx, Fy, artx, arty, dvd);
    if (!wc.valid || wc.sub) return;
    double ax = Fx + 2.0 * (a12.x - vofa * pa) * Wx;
    double ay = Fy + 2.0 * (a4.x - vofa * pa) * Wy;
    if (rhoa > 0.0) {
        const double irhoa = 1.0 / rhoa;
        ax = ax * irhoa;
        ay = ay * irhoa;
    }
    if (mask & M_ART) { ax = ax + 2.0 * artx; ay = ay + 2.0 * arty; }
    ax = ax + repx;
    ay = ay + repy;
    ay = ay + K.gravity;
    double dvof = (mask & M_DELTA_FIELD) ? (K.delta * ha * ca) * (2.0 * dvd) : 0.0;
    if (mask & M_CROSS) {
        ax = ax - drgx;
        ay = ay - drgy;
        dvof = dvof - dvx;
    }
    W.ax[a] = ax;
    W.ay[a] = ay;
    W.dvof[a] = dvof;
}

template <int SKF, int FORM>
__global__ STAGE_ATTR void k_water_b4(DPhase W, const double* recW, NList NL, Masks MW, Grid g, KParams K,
                                      FusedK F, int mask)
{
    __shared__ __align__(16) unsigned char lds[STAGE_LDS<FORM, 6>];
    water_b4<SKF, FORM>(lds, xcd_block(), W, recW, NL, MW, g, K, F, mask);
}

// Stress and pressure rates of soil particle a from its strain rate t, divergence
// and spin: plastic_or_not + plastic_flow_rule3 + Jaumann_rate (and the
// accumulated plastic strain).
struct StressRates {
    double xx, xy, yy, p;
};

__device__ __forceinline__ StressRates stress_rates(const DPhase& S, const KParams& K, int a, double txx, double txy,
                                                    double tyy, double vcc, double wxy, double pa, double sxxa,
                                                    double sxya, double syya)
{
    const double alpha = K.s_alpha1, G = K.s_G, Kb = K.s_k;
    double dsxx = 0.0, dsxy = 0.0, dsyy = 0.0, dpv = 0.0;
    // plasticity 3: plastic_or_not + plastic_flow_rule3 (failed points);
    // plasticity 1: plastic_flow_rule (m_particles.f90:3571-3633), the same
    // correction at every point, with the criterion's fail flags left as they are
    if (K.plasticity == 3 || K.plasticity == 1) {
        const double I1 = 3.0 * pa;
        const double j2r = sxxa * sxxa + 2.0 * (sxya * sxya) + syya * syya + (sxxa + syya) * (sxxa + syya);
        const double J2 = __builtin_sqrt(j2r / 2.0) + 1.0e-6;
        const int fail = fabs(J2 - alpha * I1) < SPH_YIELD_TOL_F ? 1 : 0;
        if (fail || K.plasticity == 1) {
            const double exx = txx * 0.5 + vcc * (1.0 / 3.0);
            const double exy = txy * 0.5;
            const double eyy = tyy * 0.5 + vcc * (1.0 / 3.0);
            const double sde = sxxa * exx + 2.0 * sxya * exy + syya * eyy;
            const double sj = __builtin_sqrt(j2r / 2.0 + 1.0e-10);
            const double gs = G / sj;
            const double dl = (3.0 * alpha * Kb * vcc + gs * sde) / (9.0 * (alpha * alpha) * Kb + G);
            if (!(dl < 0.0)) {
                dsxx = -dl * (gs * sxxa);
                dsxy = -dl * (gs * sxya);
                dsyy = -dl * (gs * syya);
                dpv = 3.0 * Kb * alpha * dl;
                S.eps_p[a] = S.eps_p[a] + dl * sxya / (2.0 * sj) * SPH_EPSP_F;
            }
        }
        if (K.plasticity == 3) S.fail[a] = fail;
    }
    if (K.plasticity == 2) {
        // plastic_flow_rule2 (m_particles.f90:3636-3697): at every point and
        // without the sign test; its rates act in the return mapping
        const double j2r = sxxa * sxxa + 2.0 * (sxya * sxya) + syya * syya + (sxxa + syya) * (sxxa + syya);
        const double exx = txx * 0.5 + vcc * (1.0 / 3.0);
        const double exy = txy * 0.5;
        const double eyy = tyy * 0.5 + vcc * (1.0 / 3.0);
        const double sde = sxxa * exx + 2.0 * sxya * exy + syya * eyy;
        const double sj = __builtin_sqrt(j2r / 2.0 + 1.0e-10);
        const double gs = G / sj;
        const double dl = (3.0 * alpha * Kb * vcc + gs * sde) / (9.0 * (alpha * alpha) * Kb + G);
        S.dsxx2[a] = -dl * (gs * sxxa);
        S.dsxy2[a] = -dl * (gs * sxya);
        S.dsyy2[a] = -dl * (gs * syya);
        S.dp2[a] = 3.0 * Kb * alpha * dl;
    }
    dsxx = dsxx + G * txx + 2.0 * sxya * wxy;
    dsxy = dsxy + G * txy - (sxxa - syya) * wxy;
    dsyy = dsyy + G * tyy - 2.0 * sxya * wxy;
    dpv = dpv - Kb * vcc;
    return StressRates{dsxx, dsxy, dsyy, dpv};
}

// ------------------------------------------------------------------------
// Soil, stages A and B in one kernel (SOLO: single-phase soil,
// single_step_for_soil, declarations_sph.f90:1530-1655: the df form of the
// momentum without vof factors, no repulsion, no water partners).  Soil stage B reads only what the pack
// wrote (p, sigma, vof of the partners) and the new sound speed, which is the
// constant s_c for every soil particle, so both stages share one scan and one
// dense loop over the same partner set (no stored masks, one partner load):
//   same phase  con_density, delta_sph(rho), shear_strain_rate,
//               velocity_divergence, Jaumann spin, av_vel, repulsive_force
//               (stage A); -df3(vof*p) + df3(vof*sigma) (:1270-1277),
//               art_visc, delta_sph on p, sxx, sxy, syy (stage B);
//   tail        plastic_or_not + plastic_flow_rule3 + Jaumann_rate, then
//               /rho, + repulsion, + gravity, + Darcy drag, + pore pressure
//               (the cross terms k_soil_x4 wrote; cross: two-phase run).
// ------------------------------------------------------------------------
template <int SKF, int FORM, bool SOLO>
__device__ __forceinline__ void soil_ab4(unsigned char* lds, int blk, DPhase S, const double* recS, NList NL, Grid g, KParams K, FusedK F,
                                         int cross, int mask, int lean)
{
    constexpr bool U = FORM >= UNIFORM, WIN = FORM == WINDOWS;
    const RecV RS = recv(recS, S.n);
    const SubCtx wc = sub_ctx(S.n, blk, NL.lg, SOLO ? STAGE_BLOCK : NL.is.pb << NL.lg);
    const int t = wc.t;
    auto RA = [&](int c) { return RS(wc.tt, c); };
    const double2 xy = RA(0), va = RA(1), a3 = RA(3), a4 = RA(4), a12 = RA(5);
    // U (checked by the host): h uniform in the phase (hsml(1) everywhere, a
    // wave-uniform value), integer repulsion exponents, Drucker-Prager
    const double xa = xy.x, ya = xy.y, vxa = va.x, vya = va.y, rhoa = RA(2).x;
    const double ha = U ? K.h1_soil : RA(6).x;
    const double pa = a3.y, sxxa = a12.x, sxya = a12.y, syya = a4.x;
    const double cn = K.s_c;         // sound speed after this step (stage B)
    // Mohr-Coulomb (general instantiation only): the criterion may have reset
    // rho; con_density's delta_sph, the strain rate and the divergence come
    // before it in single_step and use the density before it (chunk 7)
    const bool mc = FORM == GENERAL && K.yield_criterion == 1;
    const double rhoa_pre = mc ? RA(7).x : rhoa;
    const int a = NL.cell ? wc.tt : S.order[wc.tt];
    const int ita = S.itype[a];
    const bool link = K.nnps == 2;
    const bool uni = U || link || F.uni_s;
    const KC kc0 = make_kc(SKF, link ? K.h1_soil : ha);
    // (the tail's inputs, loaded before the loop)
    double drgx = 0.0, drgy = 0.0, porx = 0.0, pory = 0.0;
    if (mask & M_CROSS) {
        drgx = S.drgx[a];
        drgy = S.drgy[a];
        porx = S.porx[a];
        pory = S.pory[a];
    }
    const Window win = open_window<WIN, 6>(lds, NL.is, blk, wc, NL.lg, S.n, RS);
    const Cand C{g, S.cell_start, NL.cell, xa, ya};
    const Pred P{xa, ya, ha, F.thr_s, uni ? 1 : 0, link ? 1 : 0};
    const double rep2 = !SOLO && ita > 0 ? S.dspp * S.dspp : -1.0;   // real particles feel the wall
    const double et2 = K.etq * K.etq;
    const bool art = (mask & M_ART) != 0;
    double con = 0.0, drd = 0.0, sxx = 0.0, syy = 0.0, sxy = 0.0, syx = 0.0, spin = 0.0;
    double avx = 0.0, avy = 0.0;
    const double own = SOLO ? 1.0 : a3.x / rhoa;   // vof / rho^2
    const double oxx = own * (sxxa - pa), oyy = own * (syya - pa), oxy = own * sxya;
    double Fx = 0.0, Fy = 0.0;
    double artx = 0.0, arty = 0.0, dP = 0.0, dXX = 0.0, dXY = 0.0, dYY = 0.0;
    int cnt = 0;
    visit<WIN, 6>(
        lds, win, C, NL.is, S.n, wc, NL.lg, t, RS, NL.same, [&](int k, double2 b) { return P(b, uni ? ha : RS(k, 6).x, g, K); },
        [&](const auto& v, const auto& R, int k) {
            const double2 b = v[0], u = v[1], q = v[2], f = v[3], s3 = v[4], s12 = v[5];
            KC kc = kc0;
            double amh = ha;
            if (!uni) {
                amh = sph_mhsml(ha, R(k, 6).x);
                kc = pair_kc<SKF>(amh);
            }
            const Sep p = sep_of<SKF, true>(kc, xa - b.x, ya - b.y, U ? F.thr_s : INFINITY, false);
            cnt += p.in ? 1 : 0;
            const double V = fabs(q.y), m = V * q.x;
            const double dvx = vxa - u.x, dvy = vya - u.y, vr = dvx * p.dx + dvy * p.dy;
            const double Vs = V * p.s, wx = Vs * p.dx, wy = Vs * p.dy;
            // stage A
            con += (m * p.s) * vr;
            if constexpr (FORM == GENERAL) {   // (a branch for each criterion: 14 more registers and spills)
                const double rp = mc ? R(k, 7).x : q.x, t = mc ? q.x * fast_rcp(rp) : 1.0, tx = t * wx, ty = t * wy;
                drd += t * Vs * (rhoa_pre - rp);
                sxx += tx * dvx;
                syy += ty * dvy;
                sxy += ty * dvx;
                syx += tx * dvy;
                spin += wx * dvy - wy * dvx;
            } else {
                drd += Vs * (rhoa - q.x);
                sxx += wx * dvx;
                syy += wy * dvy;
                sxy += wy * dvx;
                syx += wx * dvy;
            }
            // one reciprocal for art_visc's denominator and the mean density
            const double rs = rhoa + q.x, d2 = p.dr + amh * amh * et2;
            const double it = fast_rcp(rs * d2);
            const double fv = (m * p.w) * (it * d2);
            avx -= fv * dvx;
            avy -= fv * dvy;
            if (!SOLO && q.y < 0.0 && p.dr <= rep2 && p.in) {
                const double fr = rep_factor<FORM != GENERAL>(K, S.dspp, p.ir);
                artx += p.dx * (0.5 * fr);
                arty += p.dy * (0.5 * fr);
            }
            // stage B
            if constexpr (SOLO) {
                // -df(p) + df(sigma) (single_step_for_soil :1596-1597):
                // m_b/rho_b (f_a + f_b) grad W, no vof factors
                const double fxy = oxy + s12.y;
                Fx += (oxx + (s12.x - f.y)) * wx;
                Fx += fxy * wy;
                Fy += (oyy + (s3.x - f.y)) * wy;
                Fy += fxy * wx;
            } else {
                // m (f_a / rho_a^2 + f_b / rho_b^2) grad W with m = V rho_b
                const double fxy = fma(q.x, oxy, f.x * s12.y);
                Fx += fma(q.x, oxx, f.x * (s12.x - f.y)) * wx;
                Fx += fxy * wy;
                Fy += fma(q.x, oyy, f.x * (s3.x - f.y)) * wy;
                Fy += fxy * wx;
            }
            {   // art_visc, branch-free: approaching pairs only (vr < 0)
                const double hv = amh * vr, muv = hv * (it * rs);
                const double piv = (K.beta * muv - K.alpha * cn) * (hv * it);
                const double mp = art && vr < 0.0 ? (m * p.s) * piv : 0.0;
                artx -= mp * p.dx;
                arty -= mp * p.dy;
            }
            dP += Vs * (pa - f.y);
            dXX += Vs * (sxxa - s12.x);
            dXY += Vs * (sxya - s12.y);
            dYY += Vs * (syya - s3.x);
        });

    sub_sum(NL.lg, con, drd, sxx, syy, sxy, syx, avx, avy, Fx, Fy, artx, arty, dP, dXX, dXY, dYY);
    if (mc) sub_sum(NL.lg, spin);
    cnt = sub_count(NL.lg, cnt);
    if (!wc.valid || wc.sub) return;
    const double irhoa = 1.0 / rhoa;
    const double ca = a4.y;          // sound speed before this step (delta_sph of rho)
    const double txx = SPH_C23_F * (syy - 2.0 * sxx), tyy = SPH_C23_F * (sxx - 2.0 * syy);
    const double txy = -(sxy + syx), vcc = -(sxx + syy), wxy = 0.5 * (mc ? spin : syx - sxy);
    // delta_sph(rho) and av_vel only under their switches (artificial_density,
    // average_velocity); without av_vel the reference leaves av as it was
    // single-phase soil under summation_density: sum_density replaced rho and
    // drho keeps only the delta-SPH term (declarations_sph.f90:1558-1570)
    if (SOLO && K.summation_density) con = 0.0;
    S.drho[a] = K.artificial_density ? con + (K.delta * ha * ca) * (2.0 * drd) : con;
    if (K.average_velocity) {
        const double e = ita > 0 ? 2.0 * K.epsilon : 2.0;
        S.avx[a] = e * avx;
        S.avy[a] = e * avy;
    }
    if (!lean) {
        S.txx[a] = txx; S.txy[a] = txy; S.tyy[a] = tyy; S.vcc[a] = vcc; S.wxy[a] = wxy;
        if (!cross) S.countiac[a] = cnt;
        S.nsame[a] = cnt;
    }
    S.c_next[a] = cn;

    StressRates d = stress_rates(S, K, a, txx, txy, tyy, vcc, wxy, pa, sxxa, sxya, syya);

    double ax = Fx, ay = Fy;
    if (!SOLO) { ax = ax * rhoa; ay = ay * rhoa; }
    if (rhoa > 0.0) { ax = ax * irhoa; ay = ay * irhoa; }
    ax = ax + 2.0 * artx;   // art_visc and repulsion
    ay = ay + 2.0 * arty;
    ay = ay + K.gravity;
    if (mask & M_CROSS) {
        ax = ax + drgx;
        ay = ay + drgy;
        ax = ax + porx;
        ay = ay + pory;
    }
    if (mask & M_DELTA_FIELD) {
        const double cf = K.delta * ha * cn * 2.0;
        d.p = d.p + cf * dP;
        d.xx = d.xx + cf * dXX;
        d.xy = d.xy + cf * dXY;
        d.yy = d.yy + cf * dYY;
    }
    S.dsxx[a] = d.xx; S.dsxy[a] = d.xy; S.dsyy[a] = d.yy; S.dp[a] = d.p;
    S.ax[a] = ax;
    S.ay[a] = ay;
}

template <int SKF, int FORM>
__global__ STAGE_ATTR_AB void k_soil_ab4(DPhase S, const double* recS, NList NL, Grid g, KParams K, FusedK F,
                                         int cross, int mask, int lean)
{
    __shared__ __align__(16) unsigned char lds[STAGE_LDS<FORM, 6>];
    soil_ab4<SKF, FORM, false>(lds, xcd_block(), S, recS, NL, g, K, F, cross, mask, lean);
}

// ------------------------------------------------------------------------
// A whole step in three launches on one stream (the phases uniform in h):
// stage 1 (water stage A and both cross passes: they read packed records
// alone), stage 2 (water stage B and the soil pass, which add the cross terms)
// and the final updates.  The parts of a launch are ranges of its workgroups;
// each keeps the registers and the LDS of the dearest part, and still the
// merged step is the faster at every size: the eight launches on two streams
// with an event at each dependence cost 40 us of a step (us per step, apart
// and merged: 1.5k particles 83 / 40, 33k 82 / 45, 125k 100 / 77, 258k 127 /
// 108, 1M 369 / 364).
// ------------------------------------------------------------------------
// A device flag word (two bits) that a kernel posts to the host: the word and
// the number of its step, in pinned memory that the host watches.  A copy
// engine's copy with an event behind it kept the queue for 10 us of every step
// (4 us, and 5.5 until the next kernel started).
struct FlagPost {
    const int* flag;
    int* slot;   // null: nothing to post
    int seq;
};

// By the first workgroup of a launch; the flag is of kernels before it.
__device__ __forceinline__ void post_flag(const FlagPost& p, int blk)
{
    if (!p.slot || blk != 0 || threadIdx.x != 0) return;
    const unsigned v = ((unsigned)p.seq << 2) | ((unsigned)*p.flag & 3u);
    __hip_atomic_store(p.slot, (int)v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);   // (the word alone)
}

__global__ void k_post_flag(FlagPost p) { post_flag(p, blockIdx.x); }

struct StageArgs {
    DPhase W, S;
    double *rW, *rS;
    NList nW, nS;
    Masks MW;
    Grid gW, gS;
    KParams K;
    FusedK F;
    int mask_w, mask_s, lean;
    int nbW, nbS, nbXW, nbXS;   // workgroups of the same-phase and the cross passes
    FlagPost post;              // (stage 1)
};

// The part of a launch that workgroup l belongs to, in the order of the counts
// nb (each padded to a multiple of 8, so that a part's workgroups keep the
// XCDs of their launch index), and its index there (-1: padding).  spread:
// consecutive workgroups of a part go to the same XCD (a batch gives each XCD
// a run of its cases instead).
struct PartIdx {
    int part, blk;
};

template <int N>
__device__ __forceinline__ PartIdx part_of(int l, const int (&nb)[N], bool spread)
{
    PartIdx p{0, l};
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int pad = (nb[i] + 7) & ~7;
        if (p.part == i && i + 1 < N && p.blk >= pad) {
            p.blk -= pad;
            p.part = i + 1;
        }
    }
    int n = nb[0];
#pragma unroll
    for (int i = 1; i < N; ++i)
        if (p.part == i) n = nb[i];
    if (spread) p.blk = (p.blk & 7) * ((n + 7) >> 3) + (p.blk >> 3);
    if (p.blk >= n) p.blk = -1;
    return p;
}

// FS, FX: the form of the same-phase and of the cross passes.
template <int SKF, int FS, int FX>
__device__ __forceinline__ void stage1(int l, const StageArgs& A, bool spread)
{
    __shared__ __align__(16) unsigned char lds[STAGE_LDS<FX, 4>];
    static_assert(STAGE_LDS<FX, 4> >= STAGE_LDS<FS, 3>, "both passes");
    post_flag(A.post, l);
    const PartIdx p = part_of<3>(l, {A.nbXS, A.nbW, A.nbXW}, spread);
    if (p.blk < 0) return;
    if (p.part == 0) soil_x4<SKF, FX>(lds, p.blk, A.S, A.W, A.rS, A.rW, A.nS, A.gS, A.K, A.F, A.lean);
    else if (p.part == 1) water_a4<SKF, FS>(lds, p.blk, A.W, A.rW, A.rW, A.nW, A.MW, A.gW, A.K, A.F, 1, A.lean);
    else water_x4<SKF, FX>(lds, p.blk, A.W, A.S, A.rW, A.rS, A.nW, A.gW, A.K, A.F, A.lean);
}

template <int SKF, int FS>
__device__ __forceinline__ void stage2(int l, const StageArgs& A, bool spread)
{
    __shared__ __align__(16) unsigned char lds[STAGE_LDS<FS, 6>];
    const PartIdx p = part_of<2>(l, {A.nbS, A.nbW}, spread);
    if (p.blk < 0) return;
    if (p.part == 0) soil_ab4<SKF, FS, false>(lds, p.blk, A.S, A.rS, A.nS, A.gS, A.K, A.F, 1, A.mask_s, A.lean);
    else water_b4<SKF, FS>(lds, p.blk, A.W, A.rW, A.nW, A.MW, A.gW, A.K, A.F, A.mask_w);
}

template <int SKF, int FS, int FX>
__global__ STAGE_ATTR void k_stage1(StageArgs A)
{
    stage1<SKF, FS, FX>(blockIdx.x, A, true);
}

template <int SKF, int FS>
__global__ STAGE_ATTR_AB void k_stage2(StageArgs A)
{
    stage2<SKF, FS>(blockIdx.x, A, true);
}

// The final updates of both phases, with the next step's packs when ahead.
struct FinalsArgs {
    DPhase W, S;
    KParams K;
    double *rW, *rS;
    int first, vf, renorm, ahead;
    float *qW, *qS;   // the FP32 records (mixed precision)
    Grid gW, gS;
    double cs;
    NRef nW, nS;
    int nbW, nbS;
};

__device__ __forceinline__ void finals(int l, const FinalsArgs& A, bool spread)
{
    const PartIdx p = part_of<2>(l, {A.nbS, A.nbW}, spread);
    if (p.blk < 0) return;
    if (p.part == 0) {
        if (A.ahead) step_soil(p.blk, A.S, A.K, A.rS, A.first, A.qS, A.gS, A.cs, A.nS);
        else final_soil(p.blk, A.S, A.K, A.first);
    } else {
        if (A.ahead) step_water(p.blk, A.W, A.K, A.rW, A.first, A.vf, A.renorm, A.qW, A.gW, A.cs, A.nW);
        else final_water(p.blk, A.W, A.K, A.first, A.vf, A.renorm);
    }
}

__global__ __launch_bounds__(256) void k_finals(FinalsArgs A)
{
    finals(blockIdx.x, A, true);
}
