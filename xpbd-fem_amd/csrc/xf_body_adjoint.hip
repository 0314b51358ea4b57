// xf_body_adjoint.hip -- checkpoint windows of the adjoint of small bodies on
// gfx950: one workgroup per body rolls a window forward (recording what the
// reverse needs) or reverses one, with the body's nodes (or their adjoints)
// in LDS and a workgroup barrier between colours, where the launches per
// colour (xf_adjoint.hip) have a kernel boundary. The two kinds of workgroup
// share a launch: window w - 1 is replayed while window w is reversed. The
// same operations on the same values in the same order, so the same bits.
//
// What bounds it: a colour phase of the reverse is one dependent chain, about
// 600 VALU instructions on quads (FP32 elements) against 1,070 on one lane,
// plus the LDS round trip and the barrier; the tape (96 bytes a tet and
// substep) streams beside it, read one phase ahead (holding it in cache gains
// nothing). Adjoint of 200 substeps, forward, replay and reverse together, per
// colour phase: 16x4x4 beam (64 tets a colour) 2.61 us against 7.22 with
// launches per colour, 16x8x8 (256) 4.58 against 7.99, 24x10x8 (480) 6.44
// against 8.52; FP64 element model 3.60 / 8.91 and 5.60 / 9.22.
#include <hip/hip_runtime.h>

#include "xf_adj.h"
#include "xf_body.h"
#include "xf_tet.h"

namespace {

// Phases of at most this many tets run on quads, larger ones with one lane per
// tet. 64 tets are a wave on each SIMD; FP32 reverse phases take 128 (two
// waves on each, about as long as one lane per tet, and the greedy colourings'
// larger colours are mostly in that range: 16x4x4 beam 55 us a substep against
// 58 with two rounds of 64), on workgroups of 512 threads when there are such.
constexpr uint32_t kRollQuadTets = 64;
template <class R>
constexpr uint32_t kReverseQuadTets = sizeof(R) == 4 ? 128u : 64u;
template <class R>
constexpr uint32_t kMaxThreads = sizeof(R) == 4 ? 512u : 256u;

// (first schedule position, count) of each colour, by scalar loads (the
// constant address space: nothing writes them during a launch)
typedef const __attribute__((address_space(4))) uint32_t* Records;

__device__ __forceinline__ void local_nodes(const uint2& l, uint32_t id[4]) {
    id[0] = l.x & 0xFFFFu;
    id[1] = l.x >> 16;
    id[2] = l.y & 0xFFFFu;
    id[3] = l.y >> 16;
}

// `A.roll_len` substeps of one body from (x0, v0). REC: each tet's node
// positions before its projection go to the tape (12 doubles per schedule
// position and substep), X after the sweep and O of every node to xs / oo;
// else the end state goes to x1 / v1. R: element precision (float: the step of
// xf_body_steps; double: the FP64 element model).
template <class R, bool AUX, bool REC>
__device__ __forceinline__ void roll_window(const XfBodyWindowArgs& A, const XfBodyWindowData& D, uint32_t body,
                                            double4* lds) {
    const uint32_t tid = threadIdx.x, threads = blockDim.x, last = A.ntet - 1u;
    const XfBodyParams p = D.bodies[body];
    const uint32_t n = p.n_nodes, nb = p.node_base;
    const Records rec = (Records)(D.rec + (size_t)body * 2 * A.ncol);
    const R C[3] = {(R)p.yeoh[0], (R)p.yeoh[1], (R)p.yeoh[2]};
    const bool yf = p.energy == 7u;
    const NodeLds<32> xs{reinterpret_cast<double2*>(lds)};
    const NodeLds<32> os{xs.base + 2u * A.nmax};
    auto load = [&](uint32_t c) {
        const uint32_t first = rec[2 * c], cnt = rec[2 * c + 1];
        return load_block_tet<AUX>(min(first + (cnt <= kRollQuadTets ? tid >> 2 : tid), last), D.loc, D.tg0, D.tg1,
                                   D.tg2, D.tg3, D.taux);
    };
    auto solve = [&](const BlockTet& t, double* tape) {
        uint32_t id[4];
        local_nodes(t.loc, id);
        double x[4][3];
        float w[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const double4 v = xs.get(id[k]);
            x[k][0] = v.x;
            x[k][1] = v.y;
            x[k][2] = v.z;
            w[k] = (float)v.w;
        }
        if constexpr (REC)
#pragma unroll
            for (int k = 0; k < 4; k++)
#pragma unroll
                for (int r = 0; r < 3; r++) tape[3 * k + r] = x[k][r];
        const TetMaterial m = tet_material<AUX>(t.ax, A.comp1, A.a);
        const QuadTet<R> e = quad_tet<R>(t);
        xf::solve_mixed_sim<R>(yf, C, x, w, e.Qi, e.QQ, e.QR, e.comp0, (R)m.comp1, (R)m.a, (R)A.dt);
#pragma unroll
        for (int k = 0; k < 4; k++) xs.put_xyz(id[k], x[k][0], x[k][1], x[k][2]);
    };
    auto quad = [&](const BlockTet& t, double* tape) {
        const uint32_t q = tid & 3u;
        const QuadNodes<32> nodes(xs, t.loc, q);
        double x[4], xn[4];
        float w[4];
        nodes.get(x, w);
        if constexpr (REC)
            if (q != 3u)
#pragma unroll
                for (int k = 0; k < 4; k++) tape[3 * k + q] = x[k];
        const TetMaterial m = tet_material<AUX>(t.ax, A.comp1, A.a);
        quad_solve<R>(quad_tet<R>(t), q, x, w, yf, C, (R)m.comp1, (R)m.a, (R)A.dt, xn);
        nodes.put(q, xn);
    };

    BlockTet ta = load(0), tb;
    for (uint32_t i = tid; i < n; i += threads) {
        const uint32_t k = xf_body_slot(i);
        const double4 xi = D.x0[nb + i], vi = D.v0[nb + i];
        const double flags = D.O[nb + i].w;
        double x[3] = {xi.x, xi.y, xi.z}, v[3] = {vi.x, vi.y, vi.z};
        if constexpr (sizeof(R) == 4) {
            double4 xn, on;
            predict(p, v, x, &xn, &on, xi.w, flags);
            xs.put(k, xn);
            os.put(k, on);
        } else {
            os.put(k, make_double4(x[0], x[1], x[2], flags));
            predict64_one(p, x, v);
            xs.put(k, make_double4(x[0], x[1], x[2], xi.w));
        }
    }
    __syncthreads();
    for (uint32_t s = 0; s < A.roll_len; s++) {
        double* const tape = REC ? D.tape_rec + 12 * (size_t)A.ntet * s : nullptr;
        auto phase = [&](uint32_t c, const BlockTet& t) {
            const uint32_t first = rec[2 * c], cnt = rec[2 * c + 1];
            if (cnt == 0u) return;
            if (cnt <= kRollQuadTets) {
                if ((tid >> 2) < cnt) quad(t, tape + 12 * (size_t)(first + (tid >> 2)));
            } else {
                if (tid < cnt) solve(t, tape + 12 * (size_t)(first + tid));
                for (uint32_t k = tid + threads; k < cnt; k += threads)
                    solve(load_block_tet<AUX>(first + k, D.loc, D.tg0, D.tg1, D.tg2, D.tg3, D.taux),
                          tape + 12 * (size_t)(first + k));
            }
            __syncthreads();
        };
        for (uint32_t c = 0; c < A.ncol; c += 2) {
            tb = load(c + 1u);
            phase(c, ta);
            ta = load(c + 2u < A.ncol ? c + 2u : 0u);
            phase(c + 1u, tb);
        }
        const bool more = s + 1u < A.roll_len;
        for (uint32_t i = tid; i < n; i += threads) {
            const uint32_t k = xf_body_slot(i);
            const double4 xi = xs.get(k), oi = os.get(k);
            if constexpr (REC) {
                D.xs_rec[(size_t)A.N * s + nb + i] = xi;
                D.oo_rec[(size_t)A.N * s + nb + i] = oi;
            }
            double x[3] = {xi.x, xi.y, xi.z}, v[3];
            const double o[3] = {oi.x, oi.y, oi.z};
            if constexpr (sizeof(R) == 4) {
                const double w = lock_contact(p, (uint32_t)oi.w, 0.0f, xi.w, o, x);
                const double invdt = (double)p.invdt;
#pragma unroll
                for (int r = 0; r < 3; r++) v[r] = (x[r] - o[r]) * invdt;
                if (more) {
                    double4 xn, on;
                    predict(p, v, x, &xn, &on, w, oi.w);
                    xs.put(k, xn);
                    os.put(k, on);
                }
            } else {
                finish64_one(p, (uint32_t)oi.w, o, x, v);
                if (!REC && !more) {
                    D.x1[nb + i] = make_double4(x[0], x[1], x[2], xi.w);
                    D.v1[nb + i] = make_double4(v[0], v[1], v[2], 0.0);
                } else if (more) {
                    os.put(k, make_double4(x[0], x[1], x[2], oi.w));
                    predict64_one(p, x, v);
                    xs.put(k, make_double4(x[0], x[1], x[2], xi.w));
                }
            }
        }
        __syncthreads();
    }
}

// Reverse of the window of A.rev_len substeps that ends after substep
// A.rev_end, for one body: Xb, Vb in and out, glog += the window's gradients.
template <class R, bool AUX>
__device__ __forceinline__ void reverse_window(const XfBodyWindowArgs& A, const XfBodyWindowData& D, uint32_t body,
                                               double4* lds) {
    const uint32_t tid = threadIdx.x, threads = blockDim.x, last = A.ntet - 1u;
    const XfBodyParams p = D.bodies[body];
    const uint32_t n = p.n_nodes, nb = p.node_base;
    const Records rec = (Records)(D.rec + (size_t)body * 2 * A.ncol);
    const R C[3] = {(R)p.yeoh[0], (R)p.yeoh[1], (R)p.yeoh[2]};
    const bool yf = p.energy == 7u;
    R* const gacc = static_cast<R*>(D.gacc);
    // Xb with the inverse mass, and Ob
    const NodeLds<32> bs{reinterpret_cast<double2*>(lds)};
    const NodeLds<32> os{bs.base + 2u * A.nmax};
    uint32_t jl = A.n_loss;
    // END of substep s of the window (0 the first) for every node, with the
    // loss injected when it ends a loss frame; START: after the reverse of
    // the prediction of the substep after it
    auto nodes = [&](bool start, bool end, uint32_t s) {
        const double4 *xl = nullptr, *tg = nullptr;
        if (end && jl > 0u && D.loss_at[jl - 1u] == A.rev_end - A.rev_len + s + 1u) {
            jl--;
            xl = D.xloss + (size_t)A.N * jl + nb;
            tg = D.target + (size_t)A.N * jl + nb;
        }
        for (uint32_t i = tid; i < n; i += threads) {
            const uint32_t k = xf_body_slot(i);
            const uint32_t flags = (uint32_t)D.O[nb + i].w;
            double xb[3], vb[3], w;
            if (start) {
                const double4 x4 = bs.get(k), o4 = os.get(k);
                const double ob[3] = {o4.x, o4.y, o4.z};
                xb[0] = x4.x;
                xb[1] = x4.y;
                xb[2] = x4.z;
                w = x4.w;
                node_start_one<R>(p, xb, ob, vb);
            } else {
                const double4 x4 = D.Xb[nb + i], v4 = D.Vb[nb + i];
                xb[0] = x4.x;
                xb[1] = x4.y;
                xb[2] = x4.z;
                vb[0] = v4.x;
                vb[1] = v4.y;
                vb[2] = v4.z;
                w = D.W[nb + i].w;
            }
            if (end) {
                double ob[3];
                node_end_one<R>(i, flags, p, D.xs_rev + (size_t)A.N * s + nb, D.oo_rev + (size_t)A.N * s + nb, xl, tg,
                                D.lw + nb, xb, vb, ob);
                os.put(k, make_double4(ob[0], ob[1], ob[2], 0.0));
                bs.put(k, make_double4(xb[0], xb[1], xb[2], w));
            } else {
                D.Xb[nb + i] = make_double4(xb[0], xb[1], xb[2], 0.0);
                D.Vb[nb + i] = make_double4(vb[0], vb[1], vb[2], 0.0);
            }
        }
    };
    // a tet's element data with its recorded positions (quads: this lane's
    // component, lane 3 any) and its gradient sum
    struct RevTet {
        BlockTet t;
        double x[4][3];  // quads: x[k][0]
        R g;
    };
    auto load_at = [&](uint32_t i, const double* tape, bool quads) {
        RevTet r;
        r.t = load_block_tet<AUX>(i, D.loc, D.tg0, D.tg1, D.tg2, D.tg3, D.taux);
        const double* tp = tape + 12 * (size_t)i;
        if (quads) {
            const uint32_t q = min(tid & 3u, 2u);
#pragma unroll
            for (int k = 0; k < 4; k++) r.x[k][0] = tp[3 * k + q];
        } else {
#pragma unroll
            for (int k = 0; k < 4; k++)
#pragma unroll
                for (int c = 0; c < 3; c++) r.x[k][c] = tp[3 * k + c];
        }
        r.g = gacc[i];
        return r;
    };
    auto load = [&](uint32_t c, const double* tape) {
        const uint32_t first = rec[2 * c], cnt = rec[2 * c + 1];
        const bool quads = cnt <= kReverseQuadTets<R>;
        return load_at(min(first + (quads ? tid >> 2 : tid), last), tape, quads);
    };
    auto quad = [&](const RevTet& r, uint32_t i) {
        const uint32_t q = tid & 3u;
        const QuadNodes<32> node(bs, r.t.loc, q);
        double xb[4];
        float w[4];
        node.get(xb, w);
        const double x[4] = {r.x[0][0], r.x[1][0], r.x[2][0], r.x[3][0]};
        const TetMaterial m = tet_material<AUX>(r.t.ax, A.comp1, A.a);
        const R gl = adjoint_quad<R>(quad_tet<R>(r.t), q, yf, C, x, w, (R)m.comp1, (R)m.a, (R)A.dt, xb);
        node.put(q, xb);
        if (q == 0u) gacc[i] = r.g + gl;
    };
    auto lane = [&](const RevTet& r, uint32_t i) {
        uint32_t id[4];
        local_nodes(r.t.loc, id);
        double xb[4][3];
        float w[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const double4 v = bs.get(id[k]);
            xb[k][0] = v.x;
            xb[k][1] = v.y;
            xb[k][2] = v.z;
            w[k] = (float)v.w;
        }
        const TetMaterial m = tet_material<AUX>(r.t.ax, A.comp1, A.a);
        const QuadTet<R> e = quad_tet<R>(r.t);
        const R gl = adjoint_tet<R>(yf, C, r.x, w, e.Qi, e.QQ, e.QR, e.comp0, (R)m.comp1, (R)m.a, (R)A.dt, xb);
#pragma unroll
        for (int k = 0; k < 4; k++) bs.put_xyz(id[k], xb[k][0], xb[k][1], xb[k][2]);
        gacc[i] = r.g + gl;
    };
    auto tape_of = [&](uint32_t s) { return D.tape_rev + 12 * (size_t)A.ntet * s; };

    RevTet ta = load(A.ncol - 1u, tape_of(A.rev_len - 1u)), tb;
    nodes(false, true, A.rev_len - 1u);
    __syncthreads();
    for (uint32_t s = A.rev_len; s-- > 0u;) {
        const double* const tape = tape_of(s);
        const double* const next = tape_of(s > 0u ? s - 1u : 0u);
        auto phase = [&](uint32_t c, const RevTet& r) {
            const uint32_t first = rec[2 * c], cnt = rec[2 * c + 1];
            if (cnt == 0u) return;
            if (cnt <= kReverseQuadTets<R>) {
                if ((tid >> 2) < cnt) quad(r, first + (tid >> 2));
            } else {
                if (tid < cnt) lane(r, first + tid);
                for (uint32_t k = tid + threads; k < cnt; k += threads)
                    lane(load_at(first + k, tape, false), first + k);
            }
            __syncthreads();
        };
        for (uint32_t c = A.ncol; c > 0u; c -= 2u) {
            tb = load(c - 2u, tape);
            phase(c - 1u, ta);
            const bool end = c == 2u;
            ta = load(end ? A.ncol - 1u : c - 3u, end ? next : tape);
            phase(c - 2u, tb);
        }
        nodes(true, s > 0u, s > 0u ? s - 1u : 0u);
        __syncthreads();
    }
    // the window's gradients into the total
    for (uint32_t c = 0; c < A.ncol; c++) {
        const uint32_t first = rec[2 * c], cnt = rec[2 * c + 1];
        for (uint32_t k = tid; k < cnt; k += threads) {
            D.glog[first + k] += (double)gacc[first + k];
            gacc[first + k] = R(0.0);
        }
    }
}

template <class R, bool AUX>
__global__ __launch_bounds__(kMaxThreads<R>) void xf_body_windows(XfBodyWindowArgs A, XfBodyWindowData D) {
    extern __shared__ double4 xf_window_nodes[];
    if (blockIdx.x < A.replays) roll_window<R, AUX, true>(A, D, blockIdx.x, xf_window_nodes);
    else reverse_window<R, AUX>(A, D, blockIdx.x - A.replays, xf_window_nodes);
}

// Rollout in the FP64 element model.
template <bool AUX>
__global__ __launch_bounds__(kMaxThreads<double>) void xf_body_roll64(XfBodyWindowArgs A, XfBodyWindowData D) {
    extern __shared__ double4 xf_window_nodes[];
    roll_window<double, AUX, false>(A, D, blockIdx.x, xf_window_nodes);
}

template <class K>
hipError_t launch(K fn, uint32_t grid, uint32_t threads, size_t lds, size_t lds_limit, hipStream_t s,
                  const XfBodyWindowArgs* a, const XfBodyWindowData* d) {
    if (a->ncol % 2 || a->ntet == 0 || lds > lds_limit) return hipErrorInvalidValue;
    if (grid == 0) return hipSuccess;
    if (lds > 65536) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(fn, dim3(grid), dim3(threads), lds, s, *a, *d);
    return hipGetLastError();
}

}  // namespace

extern "C" size_t xf_body_lds_bytes(uint32_t n);

// One replay and one reverse of a window (either may be absent: replays /
// reverses 0). fp64: the FP64 element model.
extern "C" hipError_t xf_launch_body_windows(hipStream_t s, bool aux, bool fp64, size_t lds_limit,
                                             const XfBodyWindowArgs* a, const XfBodyWindowData* d) {
    const uint32_t grid = a->replays + a->reverses;
    const size_t lds = xf_body_lds_bytes(a->nmax);
    if ((a->replays && a->roll_len == 0) || (a->reverses && a->rev_len == 0)) return hipErrorInvalidValue;
    // quads of a phase take 4 threads a tet; one lane per tet goes round
    const uint32_t threads = !fp64 && a->cmax > 64 ? kMaxThreads<float> : 256u;
    if (fp64)
        return aux ? launch(xf_body_windows<double, true>, grid, threads, lds, lds_limit, s, a, d)
                   : launch(xf_body_windows<double, false>, grid, threads, lds, lds_limit, s, a, d);
    return aux ? launch(xf_body_windows<float, true>, grid, threads, lds, lds_limit, s, a, d)
               : launch(xf_body_windows<float, false>, grid, threads, lds, lds_limit, s, a, d);
}

// roll_len substeps of the FP64 element model for every body, (x0, v0) to
// (x1, v1), which may be the same arrays.
extern "C" hipError_t xf_launch_body_roll64(hipStream_t s, bool aux, size_t lds_limit, const XfBodyWindowArgs* a,
                                            const XfBodyWindowData* d) {
    if (a->roll_len == 0) return hipSuccess;
    const size_t lds = xf_body_lds_bytes(a->nmax);
    return aux ? launch(xf_body_roll64<true>, a->nbodies, kMaxThreads<double>, lds, lds_limit, s, a, d)
               : launch(xf_body_roll64<false>, a->nbodies, kMaxThreads<double>, lds, lds_limit, s, a, d);
}
