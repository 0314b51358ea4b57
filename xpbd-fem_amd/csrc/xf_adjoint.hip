// xf_adjoint.hip -- gfx950 kernels of the adjoint (reverse mode) of the
// substep: gradients of a trajectory loss with respect to per-tet log mu.
// No reference counterpart (the reference has no adjoint).
//
// Precision follows the forward: FP64 node state and adjoint state, FP32
// element arithmetic; per-tet gradients are summed in FP32 over a checkpoint
// window and added to an FP64 accumulator at the window boundary. Every
// forward expression is differentiated as written, clamps included. The
// operation order matches the CPU oracle's adjoint of the same precision.
//
// FP64 element model (xf_scene_adjoint_fp64): the same rollout and adjoint
// with every element, contact and settings product in double (element
// constants and settings widened from their FP32 values, inverse masses kept
// in FP32 as the reference stores them), per-tet window sums in double: the
// trajectory and gradient of the FP64 model rather than of the reference's
// FP32 element arithmetic.
//
// Scope: simultaneous MixedSel / YeohSkinFast (energy 4, 7 or per-body 0),
// pins, ground contact. Sphere contact is not differentiated.
#include <hip/hip_runtime.h>

#include "xf_adj.h"
#include "xf_device.h"
#include "xf_element.h"

namespace {

struct TetData {
    float Qi[3][3], QQ[3], QR[3], comp0, comp1, a;
    uint32_t body;
};

template <bool AUX>
__device__ __forceinline__ TetData load_tet(uint32_t i, const float4* tg0, const float4* tg1, const float4* tg2,
                                            const float4* tg3, const float4* taux, float comp1_u, float a_u) {
    TetData t;
    float4 q0 = tg0[i], q1 = tg1[i], q2 = tg2[i], q3 = tg3[i];
    t.Qi[0][0] = q0.x; t.Qi[0][1] = q0.y; t.Qi[0][2] = q0.z;
    t.Qi[1][0] = q0.w; t.Qi[1][1] = q1.x; t.Qi[1][2] = q1.y;
    t.Qi[2][0] = q1.z; t.Qi[2][1] = q1.w; t.Qi[2][2] = q2.x;
    t.QQ[0] = q2.y; t.QQ[1] = q2.z; t.QQ[2] = q2.w;
    t.QR[0] = q3.x; t.QR[1] = q3.y; t.QR[2] = q3.z;
    t.comp0 = q3.w;
    t.comp1 = comp1_u;
    t.a = a_u;
    t.body = 0;
    if constexpr (AUX) {
        float4 ax = taux[i];
        t.comp1 = ax.x;
        t.a = ax.y;
        t.body = __float_as_uint(ax.z);
    }
    return t;
}

}  // namespace

// Reverse of the projection of the tet at schedule position i. tape holds
// each tet's 4 node positions before its projection (12 doubles per
// schedule position) for this substep; W holds the inverse masses (.w);
// gacc accumulates d(loss)/d(log comp0) per schedule position. R: element
// precision (float, or double for the FP64 element model: constants
// widened from their FP32 values).
template <bool AUX, class R>
__device__ __forceinline__ void reverse_one(uint32_t i, const uint4* __restrict__ tidx, const float4* __restrict__ tg0,
                                            const float4* __restrict__ tg1, const float4* __restrict__ tg2,
                                            const float4* __restrict__ tg3, const float4* __restrict__ taux,
                                            const double* __restrict__ tape, const double4* __restrict__ W,
                                            double4* __restrict__ Xb, R* __restrict__ gacc,
                                            const XfBodyParams* __restrict__ bodies, float comp1_u, float a_u,
                                            float dt) {
    uint4 id = tidx[i];
    TetData t = load_tet<AUX>(i, tg0, tg1, tg2, tg3, taux, comp1_u, a_u);
    const XfBodyParams& bp = bodies[t.body];
    R C[3], Qi[3][3], QQ[3], QR[3];
#pragma unroll
    for (int c = 0; c < 3; c++) {
        C[c] = (R)bp.yeoh[c];
        QQ[c] = (R)t.QQ[c];
        QR[c] = (R)t.QR[c];
#pragma unroll
        for (int r = 0; r < 3; r++) Qi[c][r] = (R)t.Qi[c][r];
    }
    const double* tp = tape + 12 * (size_t)i;
    double x[4][3];
#pragma unroll
    for (int n = 0; n < 4; n++)
#pragma unroll
        for (int r = 0; r < 3; r++) x[n][r] = tp[3 * n + r];
    uint32_t nid[4] = {id.x, id.y, id.z, id.w};
    float w[4];
    double xb[4][3];
#pragma unroll
    for (int n = 0; n < 4; n++) {
        w[n] = (float)W[nid[n]].w;
        double4 b = Xb[nid[n]];
        xb[n][0] = b.x;
        xb[n][1] = b.y;
        xb[n][2] = b.z;
    }
    R gl = adjoint_tet<R>(bp.energy == 7, C, x, w, Qi, QQ, QR, (R)t.comp0, (R)t.comp1, (R)t.a, (R)dt, xb);
    gacc[i] = gacc[i] + gl;
#pragma unroll
    for (int n = 0; n < 4; n++) Xb[nid[n]] = make_double4(xb[n][0], xb[n][1], xb[n][2], 0.0);
}

// reverse_one on four lanes (adjoint_quad): lane q holds component q of the
// four nodes, lane 3 nothing.
template <bool AUX, class R>
__device__ __forceinline__ void reverse_quad(uint32_t i, uint32_t q, const uint4* __restrict__ tidx,
                                             const float4* __restrict__ tg0, const float4* __restrict__ tg1,
                                             const float4* __restrict__ tg2, const float4* __restrict__ tg3,
                                             const float4* __restrict__ taux, const double* __restrict__ tape,
                                             const double4* __restrict__ W, double4* __restrict__ Xb,
                                             R* __restrict__ gacc, const XfBodyParams* __restrict__ bodies,
                                             float comp1_u, float a_u, float dt) {
    const uint4 id = tidx[i];
    BlockTet t;
    t.q0 = tg0[i];
    t.q1 = tg1[i];
    t.q2 = tg2[i];
    t.q3 = tg3[i];
    t.ax = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if constexpr (AUX) t.ax = taux[i];
    t.loc = make_uint2(0u, 0u);
    const uint32_t nid[4] = {id.x, id.y, id.z, id.w}, c = min(q, 2u);
    const double* tp = tape + 12 * (size_t)i + c;
    double x[4], xb[4];
    float w[4];
#pragma unroll
    for (int n = 0; n < 4; n++) {
        x[n] = tp[3 * n];
        w[n] = (float)W[nid[n]].w;
        xb[n] = reinterpret_cast<const double*>(Xb + nid[n])[c];
    }
    const R g = gacc[i];
    const TetMaterial m = tet_material<AUX>(t.ax, comp1_u, a_u);
    const XfBodyParams& bp = bodies[m.body];
    const R C[3] = {(R)bp.yeoh[0], (R)bp.yeoh[1], (R)bp.yeoh[2]};
    const R gl = adjoint_quad<R>(quad_tet<R>(t), q, bp.energy == 7, C, x, w, (R)m.comp1, (R)m.a, (R)dt, xb);
    if (q == 0u) gacc[i] = g + gl;
#pragma unroll
    for (int n = 0; n < 4; n++) reinterpret_cast<double*>(Xb + nid[n])[q] = q < 3u ? xb[n] : 0.0;
}

// Projection of the tet at schedule position i in element precision R
// (xf::solve_mixed_sim: the simultaneous MixedSel / YeohSkinFast solve of
// solve_tet in xf_kernels.hip, constants widened for R = double); REC
// records its four node positions before the projection into tape (12
// doubles per schedule position).
template <bool AUX, class R, bool REC>
__device__ __forceinline__ void project_one(uint32_t i, const uint4* __restrict__ tidx, const float4* __restrict__ tg0,
                                            const float4* __restrict__ tg1, const float4* __restrict__ tg2,
                                            const float4* __restrict__ tg3, const float4* __restrict__ taux,
                                            double4* __restrict__ X, double* __restrict__ tape,
                                            const XfBodyParams* __restrict__ bodies, float comp1_u, float a_u,
                                            float dt) {
    uint4 id = tidx[i];
    TetData t = load_tet<AUX>(i, tg0, tg1, tg2, tg3, taux, comp1_u, a_u);
    const XfBodyParams& bp = bodies[t.body];
    R C[3], Qi[3][3], QQ[3], QR[3];
#pragma unroll
    for (int c = 0; c < 3; c++) {
        C[c] = (R)bp.yeoh[c];
        QQ[c] = (R)t.QQ[c];
        QR[c] = (R)t.QR[c];
#pragma unroll
        for (int r = 0; r < 3; r++) Qi[c][r] = (R)t.Qi[c][r];
    }
    double4 na = X[id.x], nb = X[id.y], nc = X[id.z], nd = X[id.w];
    double x[4][3] = {{na.x, na.y, na.z}, {nb.x, nb.y, nb.z}, {nc.x, nc.y, nc.z}, {nd.x, nd.y, nd.z}};
    float w[4] = {(float)na.w, (float)nb.w, (float)nc.w, (float)nd.w};
    if constexpr (REC) {
        double* tp = tape + 12 * (size_t)i;
#pragma unroll
        for (int n = 0; n < 4; n++)
#pragma unroll
            for (int r = 0; r < 3; r++) tp[3 * n + r] = x[n][r];
    }
    xf::solve_mixed_sim<R>(bp.energy == 7, C, x, w, Qi, QQ, QR, (R)t.comp0, (R)t.comp1, (R)t.a, (R)dt);
    X[id.x] = make_double4(x[0][0], x[0][1], x[0][2], na.w);
    X[id.y] = make_double4(x[1][0], x[1][1], x[1][2], nb.w);
    X[id.z] = make_double4(x[2][0], x[2][1], x[2][2], nc.w);
    X[id.w] = make_double4(x[3][0], x[3][1], x[3][2], nd.w);
}

// One launch of two independent sweeps of the pipelined reverse pass:
// workgroups [0, rblocks) record colour [rbegin, rbegin + rcount) of a
// window replay (on X, into tape_rec); the rest take the reverse of colour
// [vbegin, vbegin + vcount) of the later window (tape_rev, inverse masses
// from W, adjoint Xb, gacc). The two touch disjoint arrays.
template <bool AUX, class R, bool QUAD>
__global__ __launch_bounds__(64) void xf_adj_pair(
    uint32_t rbegin, uint32_t rcount, uint32_t rblocks, double4* __restrict__ X, double* __restrict__ tape_rec,
    uint32_t vbegin, uint32_t vcount, const double* __restrict__ tape_rev, const double4* __restrict__ W,
    double4* __restrict__ Xb, R* __restrict__ gacc, const uint4* __restrict__ tidx, const float4* __restrict__ tg0,
    const float4* __restrict__ tg1, const float4* __restrict__ tg2, const float4* __restrict__ tg3,
    const float4* __restrict__ taux, const XfBodyParams* __restrict__ bodies, float comp1_u, float a_u, float dt) {
    if (QUAD && blockIdx.x >= rblocks) {
        const uint32_t k = (blockIdx.x - rblocks) * 16u + (threadIdx.x >> 2);
        if (k < vcount)
            reverse_quad<AUX, R>(vbegin + k, threadIdx.x & 3u, tidx, tg0, tg1, tg2, tg3, taux, tape_rev, W, Xb, gacc,
                                 bodies, comp1_u, a_u, dt);
        return;
    }
    if (blockIdx.x < rblocks) {
        uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
        if (k < rcount)
            project_one<AUX, R, true>(rbegin + k, tidx, tg0, tg1, tg2, tg3, taux, X, tape_rec, bodies, comp1_u, a_u,
                                      dt);
    } else {
        uint32_t k = (blockIdx.x - rblocks) * blockDim.x + threadIdx.x;
        if (k < vcount)
            reverse_one<AUX, R>(vbegin + k, tidx, tg0, tg1, tg2, tg3, taux, tape_rev, W, Xb, gacc, bodies, comp1_u,
                                a_u, dt);
    }
}

// ---------------------------------------------- FP64 element model forward
//
// Geo3d::Substep (Geo.cpp:305-356) with the element, contact and settings
// arithmetic in double, as the oracle's f64 variant: predict, colour
// launches of the simultaneous MixedSel / YeohSkinFast projection
// (xf::solve_mixed_sim<double>), then pins, ground contact and velocity.

// Prediction from V (Geo.cpp:307-312): v += g dt, v *= 1 - drag, O = X,
// X += v dt, with g dt and 1 - drag formed in double. Thread 0 advances the
// scene clock by dt (the substep's end time; not read by this model).
__global__ __launch_bounds__(256) void xf_predict64(uint32_t n, double4* __restrict__ X, double4* __restrict__ O,
                                                    const double4* __restrict__ V,
                                                    const XfBodyParams* __restrict__ bodies, float dt,
                                                    float* __restrict__ clock) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0 && clock != nullptr) {
        clock[0] = clock[0] + dt;
        uint32_t* tick = reinterpret_cast<uint32_t*>(clock) + 1;
        tick[0] = tick[0] + 1u;
    }
    if (i >= n) return;
    double4 xi = X[i], oi = O[i], vi = V[i];
    const XfBodyParams& p = bodies[(uint32_t)oi.w >> 1];
    double x[3] = {xi.x, xi.y, xi.z}, v[3] = {vi.x, vi.y, vi.z};
    predict64_one(p, x, v);
    O[i] = make_double4(xi.x, xi.y, xi.z, oi.w);
    X[i] = make_double4(x[0], x[1], x[2], xi.w);
}

// One colour of the FP64 projection; REC: records each tet's four node
// positions before its projection into tape (12 doubles per schedule
// position), as xf_project_record does for the FP32 model.
template <bool AUX, bool REC>
__global__ __launch_bounds__(64) void xf_project64(uint32_t begin, uint32_t count, const uint4* __restrict__ tidx,
                                                   const float4* __restrict__ tg0, const float4* __restrict__ tg1,
                                                   const float4* __restrict__ tg2, const float4* __restrict__ tg3,
                                                   const float4* __restrict__ taux, double4* __restrict__ X,
                                                   double* __restrict__ tape, const XfBodyParams* __restrict__ bodies,
                                                   float comp1_u, float a_u, float dt) {
    uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < count)
        project_one<AUX, double, REC>(begin + k, tidx, tg0, tg1, tg2, tg3, taux, X, tape, bodies, comp1_u, a_u, dt);
}

// End of an FP64 substep (finish64_one).
// xs_out / oo_out (nullable): X after the sweep and O are copied there first.
__global__ __launch_bounds__(256) void xf_finish64(uint32_t n, double4* __restrict__ X, const double4* __restrict__ O,
                                                   double4* __restrict__ V, const XfBodyParams* __restrict__ bodies,
                                                   double4* __restrict__ xs_out, double4* __restrict__ oo_out) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double4 xi = X[i], oi = O[i];
    if (xs_out) {
        xs_out[i] = xi;
        oo_out[i] = oi;
    }
    const uint32_t flags = (uint32_t)oi.w;
    const XfBodyParams& p = bodies[flags >> 1];
    double x[3] = {xi.x, xi.y, xi.z}, v[3];
    const double o[3] = {oi.x, oi.y, oi.z};
    finish64_one(p, flags, o, x, v);
    X[i] = make_double4(x[0], x[1], x[2], xi.w);
    V[i] = make_double4(v[0], v[1], v[2], 0.0);
}

// Reverse of the node steps around one substep boundary, per node:
// START: the prediction of the later substep (node_start_one, from Ob);
// END: then the end of the earlier substep (node_end_one, recorded xs / o,
// loss at xloss when it ends a loss frame), writing Ob for its sweep.
template <class R, bool START, bool END>
__global__ __launch_bounds__(256) void xf_adj_nodes(uint32_t n, const double4* __restrict__ O,
                                                    const double4* __restrict__ xs, const double4* __restrict__ o,
                                                    double4* __restrict__ Xb, double4* __restrict__ Vb,
                                                    double4* __restrict__ Ob, const XfBodyParams* __restrict__ bodies,
                                                    const double4* __restrict__ xloss,
                                                    const double4* __restrict__ target,
                                                    const double* __restrict__ lw) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t flags = (uint32_t)O[i].w;
    const XfBodyParams& p = bodies[flags >> 1];
    const double4 xb4 = Xb[i], vb4 = Vb[i];
    double xb[3] = {xb4.x, xb4.y, xb4.z}, vb[3] = {vb4.x, vb4.y, vb4.z};
    if constexpr (START) {
        const double4 o4 = Ob[i];
        const double ob[3] = {o4.x, o4.y, o4.z};
        node_start_one<R>(p, xb, ob, vb);
    }
    if constexpr (END) {
        double ob[3];
        node_end_one<R>(i, flags, p, xs, o, xloss, target, lw, xb, vb, ob);
        Ob[i] = make_double4(ob[0], ob[1], ob[2], 0.0);
    }
    Xb[i] = make_double4(xb[0], xb[1], xb[2], 0.0);
    if constexpr (START) Vb[i] = make_double4(vb[0], vb[1], vb[2], 0.0);
}

// Window boundary: glog += gacc (the window sum in element precision into
// the FP64 total); gacc = 0.
template <class R>
__global__ __launch_bounds__(256) void xf_adj_flush(uint32_t t, R* __restrict__ gacc, double* __restrict__ glog) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= t) return;
    glog[i] += (double)gacc[i];
    gacc[i] = R(0.0);
}

// Zero-fill of a double4 array (adjoint state reset).
__global__ __launch_bounds__(256) void xf_zero_d4(uint32_t n, double4* __restrict__ a) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = make_double4(0.0, 0.0, 0.0, 0.0);
}

// Zero-fill of n 32-bit words (gradient accumulators; a kernel rather than
// a memset so that the caller's stream may be under graph capture).
__global__ __launch_bounds__(256) void xf_zero_u32(uint32_t n, uint32_t* __restrict__ a) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = 0u;
}

// Loss targets as the caller passes them (3 doubles a node, n entries over
// all loss substeps) to the double4 layout of the node state.
__global__ __launch_bounds__(256) void xf_expand_targets(uint32_t n, const double* __restrict__ raw,
                                                         double4* __restrict__ out) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = make_double4(raw[3 * (size_t)i], raw[3 * (size_t)i + 1], raw[3 * (size_t)i + 2], 0.0);
}

// Per-node weight of the loss gradient, 2 / (nodes of the node's body); the
// body id is O.w >> 1.
__global__ __launch_bounds__(256) void xf_loss_weights(uint32_t n, const double4* __restrict__ O,
                                                       const XfBodyParams* __restrict__ bodies,
                                                       double* __restrict__ lw) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint32_t body = (uint32_t)O[i].w >> 1;
    lw[i] = 2.0 / (double)bodies[body].n_nodes;
}

// Squared-error sum of one body at one loss substep: wave (j, b) adds
// |x - target|^2 over the body's nodes in node order, component by
// component, into e[j * nb + b]. The lanes form the squares of 64 nodes at a
// time and one lane adds them, in the order of a serial loop, while the
// others load the next (one thread that also loaded took 0.2 us a node, its
// two dependent loads; 425 nodes 91 us).
__global__ __launch_bounds__(64) void xf_body_sq_err(uint32_t n_loss, uint32_t nb, uint32_t n,
                                                     const double4* __restrict__ xloss,
                                                     const double4* __restrict__ tgt,
                                                     const XfBodyParams* __restrict__ bodies,
                                                     double* __restrict__ e) {
    __shared__ double sq[2][3 * 64];
    const uint32_t k = blockIdx.x, lane = threadIdx.x;
    if (k >= n_loss * nb) return;
    const uint32_t j = k / nb, b = k % nb;
    const XfBodyParams& bp = bodies[b];
    const uint32_t cnt = bp.n_nodes;
    const double4* x = xloss + (size_t)n * j + bp.node_base;
    const double4* t = tgt + (size_t)n * j + bp.node_base;
    double acc = 0.0;
    for (uint32_t i0 = 0, half = 0; i0 < cnt; i0 += 64, half ^= 1u) {
        const uint32_t i = i0 + lane;
        if (i < cnt) {
            const double4 xi = x[i], ti = t[i];
            const double d0 = xi.x - ti.x, d1 = xi.y - ti.y, d2 = xi.z - ti.z;
            sq[half][3 * lane] = d0 * d0;
            sq[half][3 * lane + 1] = d1 * d1;
            sq[half][3 * lane + 2] = d2 * d2;
        }
        __syncthreads();
        if (lane == 0) {
            const uint32_t m = 3u * min(64u, cnt - i0);
#pragma unroll 8
            for (uint32_t q = 0; q < m; q++) acc += sq[half][q];
        }
    }
    if (lane == 0) e[k] = acc;
}

// L = sum over loss substeps, then bodies, of e / n_b, and each body's share,
// in that order by one thread: out[0] = L, out[1 + b] = body b's terms.
__global__ __launch_bounds__(64) void xf_loss_total(uint32_t n_loss, uint32_t nb, const double* __restrict__ e,
                                                    const XfBodyParams* __restrict__ bodies,
                                                    double* __restrict__ out) {
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    for (uint32_t b = 0; b < nb; b++) out[1 + b] = 0.0;
    double L = 0.0;
    for (uint32_t j = 0; j < n_loss; j++)
        for (uint32_t b = 0; b < nb; b++) {
            double v = e[(size_t)j * nb + b] / (double)bodies[b].n_nodes;
            L += v;
            out[1 + b] += v;
        }
    out[0] = L;
}

// Gradient in the caller's order: schedule position p holds the tet whose
// output slot is tout[p]; dL/dlog mu = -glog.
__global__ __launch_bounds__(256) void xf_grad_out(uint32_t t, const double* __restrict__ glog,
                                                   const uint32_t* __restrict__ tout, double* __restrict__ g) {
    uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < t) g[tout[p]] = -glog[p];
}

// Copy of two double4 arrays of n entries (the replay's per-substep
// snapshot of X and O) in one launch.
__global__ __launch_bounds__(256) void xf_copy2_d4(uint32_t n, double4* __restrict__ d0,
                                                   const double4* __restrict__ s0, double4* __restrict__ d1,
                                                   const double4* __restrict__ s1) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        d0[i] = s0[i];
        d1[i] = s1[i];
    }
}

// ------------------------------------------------------ launch wrappers

// Record of colour [rbegin, rbegin + rcount) and reverse of colour
// [vbegin, vbegin + vcount) in one launch (xf_adj_pair); either count may
// be 0. fp64: the FP64 element model (gacc then holds doubles). quad: four lanes per tet of the reverse.
extern "C" hipError_t xf_launch_adj_pair(hipStream_t s, bool aux, bool fp64, bool quad, uint32_t rbegin, uint32_t rcount,
                                         double4* X, double* tape_rec, uint32_t vbegin, uint32_t vcount,
                                         const double* tape_rev, const double4* W, double4* Xb, void* gacc,
                                         const uint4* tidx, const float4* tg0, const float4* tg1, const float4* tg2,
                                         const float4* tg3, const float4* taux, const XfBodyParams* bodies,
                                         float comp1_u, float a_u, float dt) {
    const uint32_t rblocks = (rcount + 63) / 64, vblocks = quad ? (vcount + 15) / 16 : (vcount + 63) / 64;
    if (rblocks + vblocks == 0) return hipSuccess;
    dim3 grid(rblocks + vblocks), block(64);
#define XF_PAIR(A, R, G)                                                                                         \
    hipLaunchKernelGGL((quad ? xf_adj_pair<A, R, true> : xf_adj_pair<A, R, false>), grid, block, 0, s, rbegin,   \
                       rcount, rblocks, X, tape_rec, vbegin, vcount, tape_rev, W, Xb, static_cast<R*>(G), tidx, tg0, \
                       tg1, tg2, tg3, taux, bodies, comp1_u, a_u, dt)
    if (fp64) {
        if (aux) XF_PAIR(true, double, gacc);
        else XF_PAIR(false, double, gacc);
    } else {
        if (aux) XF_PAIR(true, float, gacc);
        else XF_PAIR(false, float, gacc);
    }
#undef XF_PAIR
    return hipGetLastError();
}

// start / end: the reverse of the later substep's prediction and of the
// earlier substep's end (xs, o, xloss, target, lw are read only with end).
extern "C" hipError_t xf_launch_adj_nodes(hipStream_t s, bool fp64, bool start, bool end, uint32_t n,
                                          const double4* O, const double4* xs, const double4* o, double4* Xb,
                                          double4* Vb, double4* Ob, const XfBodyParams* bodies,
                                          const double4* xloss, const double4* target, const double* lw) {
    if (n == 0 || (!start && !end)) return hipSuccess;
    dim3 grid((n + 255) / 256), block(256);
#define XF_NODES(R, S, E)                                                                                    \
    hipLaunchKernelGGL((xf_adj_nodes<R, S, E>), grid, block, 0, s, n, O, xs, o, Xb, Vb, Ob, bodies, xloss, \
                       target, lw)
    if (fp64) {
        if (start && end) XF_NODES(double, true, true);
        else if (start) XF_NODES(double, true, false);
        else XF_NODES(double, false, true);
    } else {
        if (start && end) XF_NODES(float, true, true);
        else if (start) XF_NODES(float, true, false);
        else XF_NODES(float, false, true);
    }
#undef XF_NODES
    return hipGetLastError();
}

extern "C" hipError_t xf_launch_adj_flush(hipStream_t s, bool fp64, uint32_t t, void* gacc, double* glog) {
    if (t == 0) return hipSuccess;
    if (fp64)
        hipLaunchKernelGGL(xf_adj_flush<double>, dim3((t + 255) / 256), dim3(256), 0, s, t, static_cast<double*>(gacc),
                           glog);
    else
        hipLaunchKernelGGL(xf_adj_flush<float>, dim3((t + 255) / 256), dim3(256), 0, s, t, static_cast<float*>(gacc),
                           glog);
    return hipGetLastError();
}

extern "C" hipError_t xf_launch_predict64(hipStream_t s, uint32_t n, double4* X, double4* O, const double4* V,
                                          const XfBodyParams* bodies, float dt, float* clock) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(xf_predict64, dim3((n + 255) / 256), dim3(256), 0, s, n, X, O, V, bodies, dt, clock);
    return hipGetLastError();
}

extern "C" hipError_t xf_launch_project64(hipStream_t s, bool aux, bool rec, uint32_t begin, uint32_t count,
                                          const uint4* tidx, const float4* tg0, const float4* tg1, const float4* tg2,
                                          const float4* tg3, const float4* taux, double4* X, double* tape,
                                          const XfBodyParams* bodies, float comp1_u, float a_u, float dt) {
    if (count == 0) return hipSuccess;
    dim3 grid((count + 63) / 64), block(64);
#define XF_P64(A, RC)                                                                                              \
    hipLaunchKernelGGL((xf_project64<A, RC>), grid, block, 0, s, begin, count, tidx, tg0, tg1, tg2, tg3, taux, X, \
                       tape, bodies, comp1_u, a_u, dt)
    if (aux) {
        if (rec) XF_P64(true, true);
        else XF_P64(true, false);
    } else {
        if (rec) XF_P64(false, true);
        else XF_P64(false, false);
    }
#undef XF_P64
    return hipGetLastError();
}

extern "C" hipError_t xf_launch_finish64(hipStream_t s, uint32_t n, double4* X, const double4* O, double4* V,
                                         const XfBodyParams* bodies, double4* xs_out, double4* oo_out) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(xf_finish64, dim3((n + 255) / 256), dim3(256), 0, s, n, X, O, V, bodies, xs_out, oo_out);
    return hipGetLastError();
}

extern "C" hipError_t xf_launch_copy2_d4(hipStream_t s, uint32_t n, double4* d0, const double4* s0, double4* d1,
                                         const double4* s1) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(xf_copy2_d4, dim3((n + 255) / 256), dim3(256), 0, s, n, d0, s0, d1, s1);
    return hipGetLastError();
}

extern "C" hipError_t xf_launch_zero_d4(hipStream_t s, uint32_t n, double4* a) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(xf_zero_d4, dim3((n + 255) / 256), dim3(256), 0, s, n, a);
    return hipGetLastError();
}

extern "C" hipError_t xf_launch_zero_u32(hipStream_t s, uint32_t n, uint32_t* a) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(xf_zero_u32, dim3((n + 255) / 256), dim3(256), 0, s, n, a);
    return hipGetLastError();
}

extern "C" hipError_t xf_launch_expand_targets(hipStream_t s, uint32_t n, const double* raw, double4* out) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(xf_expand_targets, dim3((n + 255) / 256), dim3(256), 0, s, n, raw, out);
    return hipGetLastError();
}

extern "C" hipError_t xf_launch_loss_weights(hipStream_t s, uint32_t n, const double4* O, const XfBodyParams* bodies,
                                             double* lw) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(xf_loss_weights, dim3((n + 255) / 256), dim3(256), 0, s, n, O, bodies, lw);
    return hipGetLastError();
}

extern "C" hipError_t xf_launch_loss(hipStream_t s, uint32_t n_loss, uint32_t nb, uint32_t n, const double4* xloss,
                                     const double4* tgt, const XfBodyParams* bodies, double* e, double* out) {
    uint32_t terms = n_loss * nb;
    if (terms == 0) return hipSuccess;
    hipLaunchKernelGGL(xf_body_sq_err, dim3(terms), dim3(64), 0, s, n_loss, nb, n, xloss, tgt, bodies, e);
    hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
    hipLaunchKernelGGL(xf_loss_total, dim3(1), dim3(64), 0, s, n_loss, nb, e, bodies, out);
    return hipGetLastError();
}

extern "C" hipError_t xf_launch_grad_out(hipStream_t s, uint32_t t, const double* glog, const uint32_t* tout,
                                         double* g) {
    if (t == 0) return hipSuccess;
    hipLaunchKernelGGL(xf_grad_out, dim3((t + 255) / 256), dim3(256), 0, s, t, glog, tout, g);
    return hipGetLastError();
}
