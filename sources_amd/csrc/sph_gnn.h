// sph_gnn.h -- learned multi-step surrogate on the cell-list graph.
//
// A message-passing network advances the particles K leapfrog steps at once:
// one leapfrog step of size K dt (the coarse step, one right-hand side), plus
// the network's correction of velocity and density towards K steps of size
// dt:  v += c_v,  rho += c_rho,  x += K dt c_v / 2.
// Its graph is the same-phase neighbour graph of the SPH step (pairs with
// r < 2h, at most DEG per node); it sees node features (rates, velocity,
// density, stress) and edge features (relative position / h, velocity,
// density and rate differences) of the state the advance starts from.
//
// Network (weights FP32 master copy, BF16 operands, FP32 accumulation):
//   edge layer  z_ij = e_ij W1            (e_ij: FE features, e_ij[0] = 1 = bias)
//   message     m_i  = (sum_j relu(z_ij) / 16) W2
//   node MLP    y_i  = W5 relu(W4 relu(W3 [n_i, m_i] + b3) + b4) + b5
// Since W2 is linear, the sum over edges is taken before it: the per-edge
// work is one 32 x 32 x 16 MFMA per neighbour slot for 32 particles.
//
// One wavefront handles 32 particles; every matrix product is a
// v_mfma_f32_32x32x16_bf16.  Operand layout (gfx950, wave64): lane l holds row
// l % 32 of A and column l % 32 of B, k = (l / 32) * 8 + [0, 8); the 16 results
// of lane l are C[(v / 4) * 8 + (l / 32) * 4 + v % 4][l % 32], v = 0..15.
#pragma once
#include "sph_fused.h"

namespace gnn {

constexpr int FE = 16;    // edge input features
constexpr int HE = 32;    // edge hidden width = message width
constexpr int FN = 32;    // node input features
constexpr int FR = 16;    // features FR..FR+2: rate-change estimates of the correction (vx, vy, rho)
constexpr int FI = FN + HE;  // node MLP input width
constexpr int D = 64;     // node hidden width
constexpr int NO = 4;     // outputs used: c_vx, c_vy, c_rho, (spare)
constexpr int NOP = 32;   // output tile width
constexpr int DEG = 48;   // neighbour slots per node
constexpr int RAW = 12;   // per-node floats feeding the edge features
constexpr float EDGE_NORM = 1.0f / 16.0f;

// parameter offsets (floats), row-major [in][out]
constexpr int O_W1 = 0;
constexpr int O_W2 = O_W1 + FE * HE;
constexpr int O_W3 = O_W2 + HE * HE;
constexpr int O_B3 = O_W3 + FI * D;
constexpr int O_W4 = O_B3 + D;
constexpr int O_B4 = O_W4 + D * D;
constexpr int O_W5 = O_B4 + D;
constexpr int O_B5 = O_W5 + D * NOP;
constexpr int NPARAM = O_B5 + NOP;

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ int lane_id() { return threadIdx.x & 63; }

__device__ __forceinline__ f32x16 zero16()
{
    f32x16 z;
#pragma unroll
    for (int v = 0; v < 16; ++v) z[v] = 0.0f;
    return z;
}

// The 16 results of a lane are rows perm(h, v) = (v >> 2) * 8 + h * 4 + (v & 3)
// of its column, so a 32-node x 32-feature block comes out of a product in one
// of two forms, and both are operands of the next product, in registers:
//   node form     mfma(W, X): lane (r, h) holds node r.  Rounded to BF16, two
//                 v_permlane32_swap per 16 features exchange features 4-7 of
//                 the lower half-wave with 8-11 of the upper: k = h * 8 + [0, 8),
//                 the next layer's operand.
//   feature form  mfma(X, W): lane (c, h) holds feature c, nodes perm(h, v).
//                 Operand of a sum over nodes (gradients) as it stands: the
//                 order of k is free as long as both operands share it.
// So a chain of layers needs neither LDS nor barriers.
struct Op2 {
    bf16x8 k[2];   // the two k-steps of a block, rounded to BF16
};

__device__ __forceinline__ f32x16 mfma(const bf16x8& a, const bf16x8& b, const f32x16& c)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// Operand in feature form.
__device__ __forceinline__ Op2 round_feat(const f32x16& c)
{
    Op2 o;
#pragma unroll
    for (int v = 0; v < 16; ++v) o.k[v >> 3][v & 7] = (__bf16)c[v];
    return o;
}

// Result order <-> operand order of a block in node form (its own inverse).
__device__ __forceinline__ Op2 swap_order(const Op2& x)
{
    Op2 o;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
        u32x4 d = __builtin_bit_cast(u32x4, x.k[ks]);
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            // upper lanes of the first <-> lower lanes of the second
            const auto sw = __builtin_amdgcn_permlane32_swap(d[q], d[q + 2], false, false);
            d[q] = sw[0];
            d[q + 2] = sw[1];
        }
        o.k[ks] = __builtin_bit_cast(bf16x8, d);
    }
    return o;
}

// Operand in node form.
__device__ __forceinline__ Op2 round_node(const f32x16& c) { return swap_order(round_feat(c)); }

// Packed weights, in entries of one k-step of one 32-wide tile (64 lanes x 8
// values): each matrix by output tile (forward) and by input tile (backward;
// only what the gradients use: the message rows of W3, 16 of W5's columns).
constexpr int P_W1 = 0;
constexpr int P_W2 = P_W1 + 64;        // HE x HE
constexpr int P_W3 = P_W2 + 2 * 64;    // FI x D: 2 tiles x 4 k-steps
constexpr int P_W4 = P_W3 + 8 * 64;    // D x D: 2 x 4
constexpr int P_W5 = P_W4 + 8 * 64;    // D x NOP: 1 x 4
constexpr int P_B2 = P_W5 + 4 * 64;    // W2^T: 1 x 2
constexpr int P_B3 = P_B2 + 2 * 64;    // W3^T, rows FN..FI-1: 1 x 4
constexpr int P_B4 = P_B3 + 4 * 64;    // W4^T: 2 x 4
constexpr int P_B5 = P_B4 + 8 * 64;    // W5^T: 2 x 1
constexpr int NPACK = P_B5 + 2 * 64;

// Element (in BF16 values) of row r of a tile at k, the matrix having nks k-steps.
__host__ __device__ __forceinline__ int pack_at(int entry, int r, int nks, int k)
{
    return (entry + ((r >> 5) * nks + (k >> 4)) * 64 + (r & 31) + 32 * ((k >> 3) & 1)) * 8 + (k & 7);
}

// Where parameter e goes in the packed weights: f(element) up to two times.
template <class F>
__host__ __device__ __forceinline__ void pack_places(int e, F&& f)
{
    if (e < O_W2) {
        const int i = e / HE, o = e % HE;
        f(pack_at(P_W1, o, 1, i));
    } else if (e < O_W3) {
        const int i = (e - O_W2) / HE, o = (e - O_W2) % HE;
        f(pack_at(P_W2, o, 2, i));
        f(pack_at(P_B2, i, 2, o));
    } else if (e < O_B3) {
        const int i = (e - O_W3) / D, o = (e - O_W3) % D;
        f(pack_at(P_W3, o, 4, i));
        if (i >= FN) f(pack_at(P_B3, i - FN, 4, o));
    } else if (e >= O_W4 && e < O_B4) {
        const int i = (e - O_W4) / D, o = (e - O_W4) % D;
        f(pack_at(P_W4, o, 4, i));
        f(pack_at(P_B4, i, 4, o));
    } else if (e >= O_W5 && e < O_B5) {
        const int i = (e - O_W5) / NOP, o = (e - O_W5) % NOP;
        f(pack_at(P_W5, o, 4, i));
        if (o < 16) f(pack_at(P_B5, i, 1, o));
    }
}

__device__ __forceinline__ int wave_max(int v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o));
    return v;
}

// Scales of the features and outputs (set from the first recorded sample).
struct Scales {
    float inv_v;     // 1 / velocity scale
    float inv_a;     // K dt / velocity scale (acceleration -> velocity change)
    float inv_r;     // 1 / density-deviation scale (relative)
    float inv_s;     // 1 / stress scale
    float kdt;       // K dt
    float out[NO];   // output scales of the training targets (target = y * out)
    float gain[NO];  // calibrated shrinkage of the applied correction: c = y * out * gain
};

// One graph: nodes [0, n) = water (cell order) then soil.
struct Graph {
    int n;
    const float* nf;   // [n][FN]
    const float* raw;  // [n][RAW]
    const int* nb;     // [DEG][n]: slot-major, so a wave's 32 nodes read one slot contiguously
    const int* nd;     // [n]
};

// Edge features of node i (raw ri) and neighbour j (raw rj); zero when j < 0.
__device__ __forceinline__ void edge_features(const float* ri, const float* rj, bool has, float* e)
{
#pragma unroll
    for (int f = 0; f < FE; ++f) e[f] = 0.0f;
    if (!has) return;
    const float ih = 1.0f / ri[7];
    const float dx = ri[0] - rj[0], dy = ri[1] - rj[1];
    const float r = sqrtf(__builtin_fmaf(dx, dx, dy * dy));   // (written out: the same value in every kernel)
    const float q = fminf(r * ih * 0.5f, 1.0f);
    e[0] = 1.0f;
    e[1] = dx * ih;
    e[2] = dy * ih;
    e[3] = r * ih;
    e[4] = (1.0f - q) * (1.0f - q);
    e[5] = ri[2] - rj[2];
    e[6] = ri[3] - rj[3];
    e[7] = ri[4] - rj[4];
    e[8] = ri[5] - rj[5];
    e[9] = ri[6] - rj[6];
    e[10] = rj[8];
}

struct GnnArgs {
    Graph G;
    const float* W;      // [NPARAM]
    const bf16x8* Wp;    // [NPACK] packed weights
    float* out;          // [n][NO] (forward)
    // training
    const float* tgt;    // [n][NO] targets (normalised)
    const float* tw;     // [n] loss weight (1 real, 0 virtual)
    float4* part;        // [workgroups][NPART / 4] gradient sums of the workgroups
    float inv_count;     // gradient scale: 1 / (number of weighted terms)
    float inv_out[NO];   // targets are physical corrections; y predicts target * inv_out
    float cw[NO];        // loss weight of each output
};

// The edges of node i (one per lane r of both halves), two slots at a time:
// f(o1, o2) gets the BF16 features of slots s and s + 1 as operands (zero past
// the node's degree).  Half-wave h builds the 16
// features of slot s + h of its node, then lanes r and r + 32 exchange the
// feature half the other slot's operand needs (v_permlane32_swap), so each
// edge's features are computed once.  The neighbour's row of the next pair and
// the index of the one after it are in flight meanwhile.
// s0: the first slot (even); f also gets s.  Returns the largest degree.
template <class F>
__device__ __forceinline__ int for_edge_pairs(const Graph& G, int i, int s0, F&& f)
{
    const int h = lane_id() >> 5;
    const bool valid = i < G.n;
    const int deg = valid ? G.nd[i] : 0;
    const int maxdeg = __builtin_amdgcn_readfirstlane(wave_max(deg));
    float ri[RAW];
#pragma unroll
    for (int q = 0; q < RAW; ++q) ri[q] = valid ? G.raw[(size_t)i * RAW + q] : 1.0f;
    auto nbr = [&](int s) { return (s < deg) ? G.nb[(size_t)s * G.n + i] : -1; };
    struct Row {
        float4 a, b;
        float c;
    };
    auto row_of = [&](int j) {
        Row r{};
        if (j >= 0) {
            const float* p = G.raw + (size_t)j * RAW;
            r.a = reinterpret_cast<const float4*>(p)[0];
            r.b = reinterpret_cast<const float4*>(p)[1];
            r.c = p[8];
        }
        return r;
    };
    int j = nbr(s0 + h), jn = nbr(s0 + 2 + h);
    Row rn = row_of(j);
#pragma unroll 1
    for (int s = s0; s < maxdeg; s += 2) {
        const Row r = rn;
        const bool has = j >= 0;
        j = jn;
        rn = row_of(j);
        jn = nbr(s + 4 + h);
        const float rj[RAW] = {r.a.x, r.a.y, r.a.z, r.a.w, r.b.x, r.b.y, r.b.z, r.b.w, r.c, 0.0f, 0.0f, 0.0f};
        float e[FE];
        edge_features(ri, rj, has, e);
        bf16x8 flo, fhi;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            flo[q] = (__bf16)e[q];
            fhi[q] = (__bf16)e[8 + q];
        }
        const u32x4 lo = __builtin_bit_cast(u32x4, flo), hi = __builtin_bit_cast(u32x4, fhi);
        u32x4 o1, o2;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            // lane r offers features 8-15 of slot s, lane r + 32 features 0-7
            // of slot s + 1; each takes the other's (first result: the lower
            // lanes' values in both halves, second: the upper lanes')
            const unsigned x = h ? lo[q] : hi[q];
            const auto sw = __builtin_amdgcn_permlane32_swap(x, x, false, false);
            const unsigned y = h ? sw[0] : sw[1];
            o1[q] = h ? y : lo[q];   // slot s: features 0-7 | 8-15
            o2[q] = h ? hi[q] : y;   // slot s + 1
        }
        f(__builtin_bit_cast(bf16x8, o1), __builtin_bit_cast(bf16x8, o2), s);
    }
    return maxdeg;
}

// Forward pass of node i in node form, weights through w(entry) and biases
// through b(index): leaves the operands the backward pass needs.
struct Layers {
    Op2 x0[2];   // node features | message
    Op2 hs;      // summed edge layer / 16
    Op2 h3[2], h4[2];
    f32x16 y;    // outputs 0-3 in elements 0-3 of the lower half-wave, no bias
    int maxdeg;  // largest degree of the tile
};

// relu(z + bias) in node form; bias: the tile's 32 values
__device__ __forceinline__ Op2 relu_bias(f32x16 z, const float* bias)
{
    const int h = lane_id() >> 5;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const float4 b = *reinterpret_cast<const float4*>(bias + q * 8 + h * 4);
        z[4 * q] = fmaxf(z[4 * q] + b.x, 0.0f);
        z[4 * q + 1] = fmaxf(z[4 * q + 1] + b.y, 0.0f);
        z[4 * q + 2] = fmaxf(z[4 * q + 2] + b.z, 0.0f);
        z[4 * q + 3] = fmaxf(z[4 * q + 3] + b.w, 0.0f);
    }
    return round_node(z);
}

// keep(o, s): sees the edge operand of each slot.
template <class K>
__device__ __forceinline__ Layers forward_tile(const Graph& G, const float* inv_out, const bf16x8* Wp, const float* b3,
                                               const float* b4, int i, K&& keep)
{
    const int l = lane_id(), h = l >> 5;
    Layers L;
    const bf16x8 w1 = Wp[P_W1 + l];
    f32x16 t = zero16();
    L.maxdeg = for_edge_pairs(G, i, 0, [&](const bf16x8& o1, const bf16x8& o2, int s) {
        keep(o1, s);
        keep(o2, s + 1);
        const f32x16 za = mfma(w1, o1, zero16()), zb = mfma(w1, o2, zero16());
#pragma unroll
        for (int v = 0; v < 16; ++v) t[v] += fmaxf(za[v], 0.0f);
#pragma unroll
        for (int v = 0; v < 16; ++v) t[v] += fmaxf(zb[v], 0.0f);
    });
#pragma unroll
    for (int v = 0; v < 16; ++v) t[v] *= EDGE_NORM;
    L.hs = round_node(t);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
        float f[8] = {};
        if (i < G.n) {
            const float4* p = reinterpret_cast<const float4*>(G.nf + (size_t)i * FN + ks * 16 + h * 8);
            const float4 u = p[0], v = p[1];
            f[0] = u.x; f[1] = u.y; f[2] = u.z; f[3] = u.w;
            f[4] = v.x; f[5] = v.y; f[6] = v.z; f[7] = v.w;
        }
        if (ks * 16 == FR && h == 0) {   // physical units -> target units
#pragma unroll
            for (int q = 0; q < 3; ++q) f[q] *= inv_out[q];
        }
#pragma unroll
        for (int q = 0; q < 8; ++q) L.x0[0].k[ks][q] = (__bf16)f[q];
    }
    t = mfma(Wp[P_W2 + l], L.hs.k[0], zero16());
    L.x0[1] = round_node(mfma(Wp[P_W2 + 64 + l], L.hs.k[1], t));
    auto dense = [&](int entry, const Op2* x) {
        f32x16 z = zero16();
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) z = mfma(Wp[entry + ks * 64 + l], x[ks >> 1].k[ks & 1], z);
        return z;
    };
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) L.h3[nt] = relu_bias(dense(P_W3 + nt * 4 * 64, L.x0), b3 + nt * 32);
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) L.h4[nt] = relu_bias(dense(P_W4 + nt * 4 * 64, L.h3), b4 + nt * 32);
    L.y = dense(P_W5, L.h4);
    return L;
}

// Inference: one wavefront per 32 nodes, four to a workgroup.  Bound by the
// vector instructions of the edge features and by the gathers of the
// neighbours' rows: without the LDS tiles that layers exchanged before (two
// wavefronts per SIMD; now five) a rollout of 20 advances of 250k particles
// takes 9.1 ms against 9.9, with the same bits.
__global__ __launch_bounds__(256, 4) void k_gnn(GnnArgs A)
{
    const int tile = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (tile * 32 >= A.G.n) return;
    const int i = tile * 32 + (lane_id() & 31);
    const Layers L = forward_tile(A.G, A.inv_out, A.Wp, A.W + O_B3, A.W + O_B4, i, [](const bf16x8&, int) {});
    if (lane_id() < 32 && i < A.G.n) {
        const float* b5 = A.W + O_B5;
        reinterpret_cast<float4*>(A.out)[i] =
            make_float4(L.y[0] + b5[0], L.y[1] + b5[1], L.y[2] + b5[2], L.y[3] + b5[3]);
    }
}

// Training: forward and backward with the gradients of all matrices held in
// the accumulators of each wavefront over all its nodes (176 registers, so one
// wavefront per SIMD).  A workgroup sums its wavefronts' gradients through LDS
// and stores them once; k_gnn_update sums the workgroups'.  What bound the
// earlier form was one atomic per parameter and 32 nodes (23 million of them on
// 12 thousand addresses at 63k nodes), operands gathered from FP32 weights and
// a barrier per neighbour slot: 12 iterations on 63k nodes with the fit of the
// gains 2.64 ms, now 0.87 (52 us per launch of this kernel; 58 when the backward
// pass gathered its edges again).  The sums have a fixed order: the same call
// gives the same weights.
constexpr int TRAIN_WAVES = 4;      // wavefronts per workgroup
constexpr int TRAIN_GROUPS = 256;   // most workgroups: one per CU
// Neighbour slots whose edge operands a wavefront keeps in LDS for its backward
// pass (a lattice at h = 1.2 dx has 20 neighbours; slots past these are built
// again): with the weights 152 KB of the CU's 160.
constexpr int EDGE_SLOTS = 28;
static_assert(EDGE_SLOTS % 2 == 0 && EDGE_SLOTS * 64 >= 512, "pairs of slots; room for the sums");
// gradient tiles of a workgroup, in accumulator layout (element
// (v >> 2) * 256 + lane * 4 + (v & 3)): W1, W2, W3 (2 x 2), W4 (2 x 2), W5
// transposed (rows 0-3: outputs x features 0-31, rows 8-11: x features 32-63),
// and one of single values: v = 0, 1: b3, 2, 3: b4, 4-7: b5, 8: loss
constexpr int NPART = 12 * 1024;

__global__ __launch_bounds__(64 * TRAIN_WAVES) void k_gnn_train(GnnArgs A)
{
    __shared__ bf16x8 Wl[NPACK];
    __shared__ __align__(16) float bias[2 * D + NO];
    // edge operands of the wavefronts' tiles, then the sums of the wavefronts
    __shared__ bf16x8 edges[TRAIN_WAVES][EDGE_SLOTS * 64];
    float4* red = reinterpret_cast<float4*>(edges);   // [TRAIN_WAVES][512]
    const int l = lane_id(), c = l & 31, h = l >> 5, wave = threadIdx.x >> 6;
    for (int e = threadIdx.x; e < NPACK; e += blockDim.x) Wl[e] = A.Wp[e];
    for (int e = threadIdx.x; e < 2 * D + NO; e += blockDim.x)
        bias[e] = A.W[e < D ? O_B3 + e : (e < 2 * D ? O_B4 + e - D : O_B5 + e - 2 * D)];
    __syncthreads();
    // identity operands: node form -> feature form in one product per k-step
    Op2 I;
    bf16x8 I8;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        const int k = h * 8 + q;
        I.k[0][q] = (__bf16)(k == c ? 1.0f : 0.0f);
        I.k[1][q] = (__bf16)(k + 16 == c ? 1.0f : 0.0f);
        I8[q] = (__bf16)(k < 4 && k + 8 == c ? 1.0f : 0.0f);   // to rows 8-11
    }
    auto flip = [&](const Op2& x) { return round_feat(mfma(x.k[1], I.k[1], mfma(x.k[0], I.k[0], zero16()))); };
    // acc += x^T y over the 32 nodes, both in feature form
    auto outer = [&](f32x16& acc, const Op2& x, const Op2& y) {
        acc = mfma(x.k[0], y.k[0], acc);
        acc = mfma(x.k[1], y.k[1], acc);
    };
    // d where the activation is positive (both in result order)
    auto gate = [&](f32x16& d, const Op2& act) {
#pragma unroll
        for (int v = 0; v < 16; ++v) d[v] = (float)act.k[v >> 3][v & 7] > 0.0f ? d[v] : 0.0f;
    };
    auto keep_order = [] { asm volatile("" ::: "memory"); };
    auto total = [&](const f32x16& d) {
        float s = 0.0f;
#pragma unroll
        for (int v = 0; v < 16; ++v) s += d[v];
        return s;
    };
    f32x16 acc[12];
#pragma unroll
    for (int t = 0; t < 12; ++t) acc[t] = zero16();
    f32x16 &g1 = acc[0], &g2 = acc[1], *g3 = &acc[2], *g4 = &acc[6], &g5 = acc[10], &gs = acc[11];

    // consecutive tiles to a workgroup; workgroups b, b + 8, .. share an XCD
    // and take consecutive ranges
    const int nt = (A.G.n + 31) / 32, ng = gridDim.x;
    const int per = (ng + 7) / 8, full = ng - (per - 1) * 8, x = blockIdx.x & 7;
    const int lb = (x < full ? x * per : full * per + (x - full) * (per - 1)) + (blockIdx.x >> 3);
    const int t0 = (int)((int64_t)nt * lb / ng), t1 = (int)((int64_t)nt * (lb + 1) / ng);
#pragma unroll 1
    for (int tile = t0 + wave; tile < t1; tile += TRAIN_WAVES) {
        keep_order();   // (the weights are read from LDS again, not held in registers)
        const int i = tile * 32 + c;
        const Layers L = forward_tile(A.G, A.inv_out, Wl, bias, bias + D, i, [&](const bf16x8& o, int s) {
            if (s < EDGE_SLOTS) edges[wave][s * 64 + l] = o;
        });
        // ---- loss and dL/dy (lower half-wave: outputs of node i)
        bf16x8 dy;
#pragma unroll
        for (int q = 0; q < 8; ++q) dy[q] = (__bf16)0.0f;
        if (h == 0 && i < A.G.n) {
            const float wgt = A.tw[i];
            const float4 tg = reinterpret_cast<const float4*>(A.tgt)[i];
            const float t[NO] = {tg.x, tg.y, tg.z, tg.w};
#pragma unroll
            for (int q = 0; q < NO; ++q) {
                const float err = L.y[q] + bias[2 * D + q] - t[q] * A.inv_out[q];
                gs[8] += A.cw[q] * wgt * err * err;
                const float d = 2.0f * A.cw[q] * wgt * err * A.inv_count;
                gs[4 + q] += d;
                dy[q] = (__bf16)d;
            }
        }
        // ---- W5, dz4 = (dy W5^T) [H4 > 0]
        Op2 dz[2], dzf[2];   // node form, feature form
        {
            const Op2 a = round_feat(mfma(dy, I.k[0], zero16())), b = round_feat(mfma(dy, I8, zero16()));
            const Op2 hf[2] = {flip(L.h4[0]), flip(L.h4[1])};
            outer(g5, a, hf[0]);
            outer(g5, b, hf[1]);
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const bf16x8 w = Wl[P_B5 + t * 64 + l];
                f32x16 d = mfma(w, dy, zero16());
                gate(d, swap_order(L.h4[t]));
                dz[t] = round_node(d);
                d = mfma(dy, w, zero16());
                gate(d, hf[t]);
                gs[2 + t] += total(d);
                dzf[t] = round_feat(d);
            }
        }
        // ---- W4, dz3 = (dz4 W4^T) [H3 > 0]
        {
            const Op2 hf[2] = {flip(L.h3[0]), flip(L.h3[1])};
#pragma unroll
            for (int t = 0; t < 4; ++t) outer(g4[t], hf[t >> 1], dzf[t & 1]);
            Op2 d3[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                f32x16 d = zero16(), df = zero16();
#pragma unroll
                for (int ks = 0; ks < 4; ++ks) {
                    const bf16x8 w = Wl[P_B4 + (t * 4 + ks) * 64 + l];
                    d = mfma(w, dz[ks >> 1].k[ks & 1], d);
                    df = mfma(dz[ks >> 1].k[ks & 1], w, df);
                }
                gate(d, swap_order(L.h3[t]));
                d3[t] = round_node(d);
                gate(df, hf[t]);
                gs[t] += total(df);
                dzf[t] = round_feat(df);
            }
            dz[0] = d3[0];
            dz[1] = d3[1];
        }
        // ---- W3, message gradient dm, W2, and d hsum = (dm W2^T) / 16
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const Op2 xf = flip(L.x0[t]);
            outer(g3[2 * t], xf, dzf[0]);
            outer(g3[2 * t + 1], xf, dzf[1]);
        }
        f32x16 dh = zero16();
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) dh = mfma(Wl[P_B3 + ks * 64 + l], dz[ks >> 1].k[ks & 1], dh);
        const Op2 dm = round_node(dh);
        outer(g2, flip(L.hs), flip(dm));
        dh = mfma(dm.k[0], Wl[P_B2 + l], zero16());
        dh = mfma(dm.k[1], Wl[P_B2 + 64 + l], dh);
#pragma unroll
        for (int v = 0; v < 16; ++v) dh[v] *= EDGE_NORM;
        keep_order();
        // ---- W1: sum over edges of e^T (dh [z > 0])
        const bf16x8 w1 = Wl[P_W1 + l];
        auto edge = [&](const bf16x8& o) {
            f32x16 z = mfma(o, w1, zero16());
            const Op2 ef = round_feat(mfma(o, I.k[0], zero16()));
#pragma unroll
            for (int v = 0; v < 16; ++v) z[v] = z[v] > 0.0f ? dh[v] : 0.0f;
            outer(g1, ef, round_feat(z));
        };
        // (the slot past an odd degree holds zeros)
#pragma unroll 1
        for (int s = 0; s < min(L.maxdeg, EDGE_SLOTS); s += 2) {
            const bf16x8 o1 = edges[wave][s * 64 + l], o2 = edges[wave][(s + 1) * 64 + l];
            edge(o1);
            edge(o2);
        }
        if (L.maxdeg > EDGE_SLOTS)
            for_edge_pairs(A.G, i, EDGE_SLOTS, [&](const bf16x8& o1, const bf16x8& o2, int) {
                edge(o1);
                edge(o2);
            });
    }
    // single values: over the halves, outputs and loss over the wavefront
#pragma unroll
    for (int v = 0; v < 9; ++v) {
        float s = gs[v];
        s += __shfl_xor(s, 32);
        if (v >= 4) {
#pragma unroll
            for (int o = 16; o > 0; o >>= 1) s += __shfl_xor(s, o);
        }
        gs[v] = s;
    }
    float4* out = A.part + (size_t)blockIdx.x * (NPART / 4);
    __syncthreads();   // (red: the edge operands are done)
#pragma unroll
    for (int ch = 0; ch < 6; ++ch) {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const f32x16& a = acc[2 * ch + (q >> 2)];
            const int v = 4 * (q & 3);
            red[wave * 512 + q * 64 + l] = make_float4(a[v], a[v + 1], a[v + 2], a[v + 3]);
        }
        __syncthreads();
        for (int e = threadIdx.x; e < 512; e += blockDim.x) {
            float4 s = red[e];
#pragma unroll
            for (int w = 1; w < TRAIN_WAVES; ++w) {
                const float4 a = red[w * 512 + e];
                s.x += a.x; s.y += a.y; s.z += a.z; s.w += a.w;
            }
            out[ch * 512 + e] = s;
        }
        __syncthreads();
    }
}

// The parameter at element p of a workgroup's gradient tiles (-1: none, -2: the loss).
__device__ __forceinline__ int param_at(int p)
{
    const int t = p >> 10, q = (p >> 8) & 3, l = (p >> 2) & 63, e = p & 3;
    const int row = q * 8 + (l >> 5) * 4 + e, col = l & 31;
    if (t == 0) return row < FE ? O_W1 + row * HE + col : -1;
    if (t == 1) return O_W2 + row * HE + col;
    if (t < 10) {
        const int m = (t - 2) & 3;
        return (t < 6 ? O_W3 : O_W4) + ((m >> 1) * 32 + row) * D + (m & 1) * 32 + col;
    }
    if (t == 10) return (row & 7) < NO && row < 16 ? O_W5 + ((row >> 3) * 32 + col) * NOP + (row & 7) : -1;
    const int v = q * 4 + e;
    if (l >= 32 || v > 8 || (v >= 4 && l > 0)) return -1;
    return v < 2 ? O_B3 + v * 32 + l : (v < 4 ? O_B4 + (v - 2) * 32 + l : (v < 8 ? O_B5 + v - 4 : -2));
}

struct AdamArgs {
    float *W, *m, *v;
    __bf16* Wp;      // packed weights, kept in step with W
    float lr, b1, b2, eps, c1, c2, clip;
};

// Sums the gradients of np workgroups.  gW != nullptr: stores them; otherwise
// one step of Adam (Kingma & Ba 2015) on the FP32 master weights.  64 elements
// per workgroup of 16 wavefronts, each summing every 16th workgroup's.
__global__ __launch_bounds__(1024) void k_gnn_update(const float* part, int np, float* gW, float* loss, AdamArgs U)
{
    __shared__ float s[16][64];
    const int l = threadIdx.x & 63, r = threadIdx.x >> 6, p = blockIdx.x * 64 + l;
    float g = 0.0f;
#pragma unroll 4
    for (int b = r; b < np; b += 16) g += part[(size_t)b * NPART + p];
    s[r][l] = g;
    __syncthreads();
    if (r > 0) return;
#pragma unroll
    for (int q = 1; q < 16; ++q) g += s[q][l];
    const int i = param_at(p);
    if (i == -2) *loss = g;
    if (i < 0) return;
    if (gW) {
        gW[i] = g;
        return;
    }
    const float gi = fminf(fmaxf(g, -U.clip), U.clip);
    const float mi = U.b1 * U.m[i] + (1.0f - U.b1) * gi;
    const float vi = U.b2 * U.v[i] + (1.0f - U.b2) * gi * gi;
    U.m[i] = mi;
    U.v[i] = vi;
    const float w = U.W[i] - U.lr * (mi * U.c1) / (sqrtf(vi * U.c2) + U.eps);
    U.W[i] = w;
    pack_places(i, [&](int e) { U.Wp[e] = (__bf16)w; });
}

__global__ void k_gnn_pack(const float* W, __bf16* Wp)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < NPARAM) pack_places(i, [&](int e) { Wp[e] = (__bf16)W[i]; });
}

// ------------------------------------------------------------------------
// Graph and features of one phase, in cell order: node = off + t for the
// particle a = order[t].  Neighbours: same-phase pairs with r < 2h (the
// exact predicate of the step), at most DEG (nd counts the kept ones).
// ------------------------------------------------------------------------
struct GatherOut {
    float* nf;
    float* raw;
    int* nb;
    int* nd;
    int n_nodes;       // nodes of both phases: the slot stride of nb
    float* tw;         // [n]
    int* node_of_id;   // [n of the phase] (phase-local ids)
    int* overflow;     // [1]
};

// nl_cell = nullptr: candidates are the rows of the particle's current cell (a
// cell list of the current positions on grid g).  Otherwise the cell list and
// record order are those of the neighbour lists (grid g is their grid, and the
// state is in cell order): the candidates are the particle's index list IL
// (windows of pb particles), tested with the current positions; a list that
// overflowed walks its rows.  The index list is what the coarse step reads
// next; with masks and the order looked up per candidate this took 36 us for
// 258k particles.
__device__ __forceinline__ void gnn_gather_body(int blk, DPhase P, Grid g, KParams K, double thr, int uni, int off,
                                                int phase, Scales S, GatherOut O, IdxList IL, int pb,
                                                const int* nl_cell)
{
    const int t = blk * blockDim.x + threadIdx.x;
    if (t >= P.n) return;
    const bool listed = nl_cell != nullptr;
    const int a = listed ? t : P.order[t];
    const int node = off + t;
    const double x = P.x[a], y = P.y[a], h = P.hsml[a];
    const double rho0 = phase == 0 ? K.w_rho0 : K.s_rho0;
    const bool virt = P.itype[a] < 0;
    const double kdt = S.kdt;
    float nf[FN];
    nf[0] = 1.0f;
    nf[1] = (float)phase;
    nf[2] = virt ? 1.0f : 0.0f;
    nf[3] = (float)(P.ax[a] * S.inv_a);
    nf[4] = (float)(P.ay[a] * S.inv_a);
    nf[5] = (float)(P.vx[a] * S.inv_v);
    nf[6] = (float)(P.vy[a] * S.inv_v);
    nf[7] = (float)((P.rho[a] - rho0) / rho0 * S.inv_r);
    nf[8] = (float)(P.drho[a] * kdt / rho0 * S.inv_r);
    nf[9] = (float)P.vof[a];
    if (phase == 1) {
        nf[10] = (float)(P.sxx[a] * S.inv_s);
        nf[11] = (float)(P.sxy[a] * S.inv_s);
        nf[12] = (float)(P.syy[a] * S.inv_s);
        nf[13] = (float)(P.p[a] * S.inv_s);
    } else {
        nf[10] = nf[11] = nf[12] = nf[13] = 0.0f;
    }
    nf[14] = nf[15] = 0.0f;
    // the rates the state holds (of the step before): k_gnn_delta turns them
    // into the rate-change features once the coarse step has evaluated the
    // rates of this state
    nf[FR] = (float)P.ax[a];
    nf[FR + 1] = (float)P.ay[a];
    nf[FR + 2] = (float)P.drho[a];
#pragma unroll
    for (int f = FR + 3; f < FN; ++f) nf[f] = 0.0f;
    // rows of 16 and 12 floats, written as 16-byte vectors
    float4* nf4 = reinterpret_cast<float4*>(O.nf + (size_t)node * FN);
#pragma unroll
    for (int q = 0; q < FN / 4; ++q) nf4[q] = make_float4(nf[4 * q], nf[4 * q + 1], nf[4 * q + 2], nf[4 * q + 3]);
    float4* rw4 = reinterpret_cast<float4*>(O.raw + (size_t)node * RAW);
    rw4[0] = make_float4((float)x, (float)y, nf[5], nf[6]);
    rw4[1] = make_float4(nf[7], nf[3], nf[4], (float)h);
    rw4[2] = make_float4(nf[2], 0.0f, 0.0f, 0.0f);
    O.tw[node] = virt ? 0.0f : 1.0f;
    O.node_of_id[P.id[a]] = node;
    // neighbours (cell order of the same phase), in ascending k
    int cnt = 0;
    int* nb = O.nb + node;   // slot s at nb[s * n_nodes]
    const size_t ns = (size_t)O.n_nodes;
    // candidates in groups of four: the position loads of all four, then the
    // predicates in candidate order
    auto group = [&](int k0, int k1, int k2, int k3) {
        const int kq[4] = {k0, k1, k2, k3};
        int bq[4];
        double xq[4], yq[4], hq[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) bq[q] = kq[q] < 0 || listed ? kq[q] : P.order[kq[q]];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int b = bq[q] >= 0 ? bq[q] : a;
            xq[q] = P.x[b];
            yq[q] = P.y[b];
            hq[q] = uni ? h : P.hsml[b];
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int k = kq[q];
            if (bq[q] < 0 || k == t) continue;
            const double dx = x - xq[q], dy = y - yq[q];
            double dr;
            {
#pragma clang fp contract(off)
                dr = dx * dx + dy * dy;
            }
            if (!pred(uni != 0, thr, dr, h, hq[q], K)) continue;
            if (cnt < DEG) nb[(size_t)cnt * ns] = off + k;
            ++cnt;
        }
    };
    const int nc = listed ? IL.cnt[t] : -1;
    if (nc >= 0) {
        const Ranges3 rec = window_ranges(IL.win + (size_t)(t / pb) * WIN_INTS);
        const unsigned short* li = IL.li + t;
        const size_t row = (size_t)P.n;
#pragma unroll 1
        for (int j = 0; j < nc; j += 4, li += 4 * row) {
            int kq[4];   // (the lists are padded: loads past the end stay inside)
#pragma unroll
            for (int q = 0; q < 4; ++q) kq[q] = li[q * row];
#pragma unroll
            for (int q = 0; q < 4; ++q) kq[q] = j + q < nc ? rec(kq[q]) : -1;
            group(kq[0], kq[1], kq[2], kq[3]);
        }
    } else {
        int cx, cy;
        if (listed) {
            const int key = nl_cell[t];
            cy = key / g.ncx;
            cx = key - cy * g.ncx;
        } else {
            clamped_cell(g, x, y, cx, cy);
        }
        const Rows R = block_rows_at(g, P.cell_start, cx, cy);
#pragma unroll 1
        for (int r = 0; r < 3; ++r) {
            const int k0 = r == 0 ? R.k0[0] : (r == 1 ? R.k0[1] : R.k0[2]);
            const int k1 = r == 0 ? R.k1[0] : (r == 1 ? R.k1[1] : R.k1[2]);
#pragma unroll 1
            for (int kb = k0; kb < k1; kb += 4) {
                int kq[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) kq[q] = kb + q < k1 ? kb + q : -1;
                group(kq[0], kq[1], kq[2], kq[3]);
            }
        }
    }
    if (cnt > DEG) atomicOr(O.overflow, 1);
    O.nd[node] = min(cnt, DEG);   // (slots past the degree are never read)
}

__global__ void k_gnn_gather(DPhase P, Grid g, KParams K, double thr, int uni, int off, int phase, Scales S,
                             GatherOut O, IdxList IL, int pb, const int* nl_cell)
{
    gnn_gather_body(blockIdx.x, P, g, K, thr, uni, off, phase, S, O, IL, pb, nl_cell);
}

// Rate-change features: after the coarse step P holds the rates evaluated at
// the state the advance starts from, and features FR..FR+2 hold the rates of
// the evaluation `gap` steps of dt before it.  Over K steps of dt a rate r
// changing at dr/dt moves the fine result from the coarse one by about
// K (K - 1) / 2 dt^2 dr/dt: with dr/dt ~ (r_new - r_old) / (gap dt) the
// features become coef (r_new - r_old), coef = K (K - 1) / 2 dt / gap, in the
// units of the correction (velocity, density).
__device__ __forceinline__ void gnn_delta_body(int blk, DPhase P, const int* node_of_id, float* nf, double coef)
{
    const int a = blk * blockDim.x + threadIdx.x;
    if (a >= P.n) return;
    float* f = nf + (size_t)node_of_id[P.id[a]] * FN + FR;
    f[0] = (float)((P.ax[a] - (double)f[0]) * coef);
    f[1] = (float)((P.ay[a] - (double)f[1]) * coef);
    f[2] = (float)((P.drho[a] - (double)f[2]) * coef);
}

__global__ void k_gnn_delta(DPhase P, const int* node_of_id, float* nf, double coef)
{
    gnn_delta_body(blockIdx.x, P, node_of_id, nf, coef);
}

// Targets: fine state (K plain steps, current) minus coarse state (one step
// of K dt, snapshot C), by particle id, in physical units.
__global__ void k_gnn_target(DPhase P, const int* node_of_id, DPhase C, const int* slot_of_id_c, float* tgt)
{
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= P.n) return;
    const int id = P.id[a];
    const int node = node_of_id[id];
    const int b = slot_of_id_c[id];
    float* tg = tgt + (size_t)node * NO;
    tg[0] = (float)(P.vx[a] - C.vx[b]);
    tg[1] = (float)(P.vy[a] - C.vy[b]);
    tg[2] = (float)(P.rho[a] - C.rho[b]);
    tg[3] = 0.0f;
}

// The network's correction of the coarse step (real particles).
__device__ __forceinline__ void gnn_correct_body(int blk, DPhase P, KParams K, const int* node_of_id, const float* y,
                                                 Scales S, int phase)
{
    const int a = blk * blockDim.x + threadIdx.x;
    if (a >= P.n) return;
    if (P.itype[a] <= 0) return;
    const int node = node_of_id[P.id[a]];
    const float* yy = y + (size_t)node * NO;
    const double cvx = (double)yy[0] * S.out[0] * S.gain[0];
    const double cvy = (double)yy[1] * S.out[1] * S.gain[1];
    const double crh = (double)yy[2] * S.out[2] * S.gain[2];
    P.vx[a] = P.vx[a] + cvx;
    P.vy[a] = P.vy[a] + cvy;
    P.x[a] = P.x[a] + 0.5 * (double)S.kdt * cvx;
    P.y[a] = P.y[a] + 0.5 * (double)S.kdt * cvy;
    P.rho[a] = P.rho[a] + crh;
    if (phase == 1) P.vof[a] = P.rho[a] / K.s_rho0;
}

__global__ void k_gnn_correct(DPhase P, KParams K, const int* node_of_id, const float* y, Scales S, int phase)
{
    gnn_correct_body(blockIdx.x, P, K, node_of_id, y, S, phase);
}

// out[0]: max (as float bits: non-negative floats order as their bits);
// sq[0] += sum of squares, sq[1] += count.  One atomic per block.
__global__ __launch_bounds__(256) void k_rho_err(DPhase A, DPhase B, const int* slot_of_id_b, unsigned int* out,
                                                 double* sq)
{
    __shared__ float smax[4];
    __shared__ double ssum[4], scnt[4];
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    float e = 0.0f;
    double e2 = 0.0, c = 0.0;
    if (a < A.n && A.itype[a] > 0) {
        const int b = slot_of_id_b[A.id[a]];
        const double ed = fabs(A.rho[a] - B.rho[b]) / fabs(B.rho[b]);
        e = (float)ed;
        e2 = ed * ed;
        c = 1.0;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        e = fmaxf(e, __shfl_xor(e, o));
        e2 += __shfl_xor(e2, o);
        c += __shfl_xor(c, o);
    }
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        smax[w] = e;
        ssum[w] = e2;
        scnt[w] = c;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        const int nw = (blockDim.x + 63) >> 6;
        for (int i = 1; i < nw; ++i) {
            e = fmaxf(e, smax[i]);
            e2 += ssum[i];
            c += scnt[i];
        }
        atomicMax(out, __float_as_uint(e));
        unsafeAtomicAdd(&sq[0], e2);
        unsafeAtomicAdd(&sq[1], c);
    }
}

// Flags a state a learned advance has broken: a non-finite or non-positive
// density, a non-finite velocity, or a particle outside the cell grid.
__device__ __forceinline__ void sanity_body(int blk, DPhase P, Grid g, int* flag)
{
    const int a = blk * blockDim.x + threadIdx.x;
    if (a >= P.n) return;
    const double x = P.x[a], y = P.y[a], r = P.rho[a];
    const bool ok = x >= g.x0 && x <= g.x1 && y >= g.y0 && y <= g.y1 && r > 0.0 && r < 1.0e300 &&
                    P.vx[a] == P.vx[a] && P.vy[a] == P.vy[a];
    if (!ok) atomicOr(flag, 1);
}

__global__ void k_sanity(DPhase P, Grid g, int* flag)
{
    sanity_body(blockIdx.x, P, g, flag);
}

// Least-squares gain of each output channel over one sample (real nodes):
// acc[o] += sum w y_o t_o / out_o, acc[NO + o] += sum w y_o^2.  The gain
// sum(y t) / sum(y^2) scales the applied correction so that it removes
// as much of the target as the network's prediction explains.
__global__ __launch_bounds__(256) void k_gnn_fit(const float* y, const float* tgt, const float* tw, int n,
                                                 Scales S, double* acc)
{
    __shared__ double part[4][2 * NO];
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    double v[2 * NO];
#pragma unroll
    for (int o = 0; o < NO; ++o) {
        const bool ok = i < n && tw[i] > 0.0f;
        const double yo = ok ? (double)y[(size_t)i * NO + o] : 0.0;
        const double to = ok ? (double)tgt[(size_t)i * NO + o] / (double)S.out[o] : 0.0;
        v[o] = yo * to;
        v[NO + o] = yo * yo;
    }
#pragma unroll
    for (int q = 0; q < 2 * NO; ++q)
        for (int off = 32; off > 0; off >>= 1) v[q] += __shfl_down(v[q], off, 64);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0)
        for (int q = 0; q < 2 * NO; ++q) part[w][q] = v[q];
    __syncthreads();
    if (threadIdx.x < 2 * NO) {
        const double sum = part[0][threadIdx.x] + part[1][threadIdx.x] + part[2][threadIdx.x] + part[3][threadIdx.x];
        atomicAdd(&acc[threadIdx.x], sum);
    }
}

// The state of a phase copied back from a snapshot (A.s* -> A.d*) when the
// sanity flag is set: a learned advance that broke the state is undone on
// the device, before any later kernel reads it.  Posts the flag.
__device__ __forceinline__ void restore_if_body(int blk, const int* flag, PermArgs A, int n, FlagPost post)
{
    post_flag(post, blk);
    if (*flag == 0) return;
    const int i = blk * blockDim.x + threadIdx.x;
    if (i >= n) return;
    // (constant indices into the argument arrays: a runtime-indexed loop
    // would copy them to scratch memory)
#pragma unroll
    for (int q = 0; q < PERM_MAXD; ++q)
        if (q < A.nd) A.dd[q][i] = A.sd[q][i];
#pragma unroll
    for (int q = 0; q < PERM_MAXI; ++q)
        if (q < A.ni) A.di[q][i] = A.si[q][i];
}

__global__ void k_restore_if(const int* flag, PermArgs A, int n, FlagPost post)
{
    restore_if_body(blockIdx.x, flag, A, n, post);
}

__global__ void k_slot_of_id(DPhase P, int* slot_of_id)
{
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a < P.n) slot_of_id[P.id[a]] = a;
}

}  // namespace gnn
