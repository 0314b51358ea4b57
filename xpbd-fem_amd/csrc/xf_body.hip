// xf_body.hip -- whole step calls of small bodies on gfx950: one workgroup
// per body runs the prediction, every colour phase, every pass and the node
// phase of all substeps of a call with the body's nodes in LDS, a workgroup
// barrier between phases where the per-colour launches have a kernel
// boundary. Colours in order, tets of a colour sharing no node: the same
// operations on the same values as the per-colour launches, so the same bits.
//
// What bounds it: a phase is one dependent element chain plus an LDS round
// trip and a barrier, where a colour launch has a kernel boundary and two
// dependent loads from beyond L2 before the chain starts. Per colour phase,
// node phase included, beam with greedy colours: 12x4x4 cells (1,152 tets,
// phases on quads) 0.89 us against 2.68 with launches per colour, 16x8x8
// (phases of up to 305 tets) 1.56 against 3.15, 24x10x8 (up to 564 tets, the
// whole LDS) 2.13 against 3.26.
#include <hip/hip_runtime.h>

#include "xf_body.h"
#include "xf_tet.h"

namespace {

// A phase of at most this many tets runs on quads (four waves, one per SIMD);
// a larger one has waves for every SIMD with one lane per tet.
constexpr uint32_t kBodyQuadTets = 64;

struct BodyTet {
    BlockTet t;
    float2 dm;  // surface area, position in the body's sweep order (PASSES)
};

// PASSES: volume and damping passes as A.vpasses and A.post say, material
// from the per-tet slots. DAMP: bodies may damp inside the projection.
template <int E, bool SIM, bool AUX, bool DAMP, bool PASSES>
__global__ __launch_bounds__(512) void xf_body_steps(
    XfBodyArgs A, const uint32_t* __restrict__ recs, const uint2* __restrict__ loc, const float4* __restrict__ tg0,
    const float4* __restrict__ tg1, const float4* __restrict__ tg2, const float4* __restrict__ tg3,
    const float4* __restrict__ taux, const float2* __restrict__ tdmp, double4* __restrict__ Xs,
    const double4* __restrict__ Os, double4* __restrict__ Vs, const XfBodyParams* __restrict__ bodies,
    float* __restrict__ clock) {
    extern __shared__ double4 xf_body_nodes[];
    constexpr bool HQ = SIM && !DAMP && (E == 0 || E == 4 || E == 7);
    const uint32_t tid = threadIdx.x, bs = blockDim.x, last = A.ntet - 1u;
    const XfBodyParams p = bodies[blockIdx.x];  // a copy: in scalar registers over the LDS writes of the phases
    const uint32_t n = p.n_nodes;
    double4* const X = Xs + p.node_base;
    const double4* const O = Os + p.node_base;
    double4* const V = Vs + p.node_base;
    const uint32_t* rec = recs + (size_t)blockIdx.x * 2 * A.ncol;
    const float C[3] = {p.yeoh[0], p.yeoh[1], p.yeoh[2]};
    const bool yf = E == 7 || (E == 0 && p.energy == 7u);
    // X with the inverse mass, and O with the flags (V while a pass damps it)
    const NodeLds<32> xs{reinterpret_cast<double2*>(xf_body_nodes)};
    const NodeLds<32> os{xs.base + 2u * A.nmax};

    auto load_tet = [&](uint32_t i) {
        BodyTet b;
        b.t = load_block_tet<AUX>(i, loc, tg0, tg1, tg2, tg3, taux);
        b.dm = make_float2(0.0f, 0.0f);
        if constexpr (PASSES) b.dm = tdmp[i];
        return b;
    };
    auto load = [&](uint32_t c, bool project) {
        const uint32_t first = rec[2 * c], cnt = rec[2 * c + 1];
        return load_tet(min(first + (HQ && project && cnt <= kBodyQuadTets ? tid >> 2 : tid), last));
    };
    auto nodes4 = [](const uint2& l, uint32_t id[4]) {
        id[0] = l.x & 0xFFFFu;
        id[1] = l.x >> 16;
        id[2] = l.y & 0xFFFFu;
        id[3] = l.y >> 16;
    };
    auto get3 = [](const auto& s, const uint32_t id[4], double x[4][3], float w[4]) {
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const double4 v = s.get(id[k]);
            x[k][0] = v.x;
            x[k][1] = v.y;
            x[k][2] = v.z;
            w[k] = (float)v.w;
        }
    };
    auto put3 = [](const auto& s, const uint32_t id[4], const double x[4][3]) {
#pragma unroll
        for (int k = 0; k < 4; k++) s.put_xyz(id[k], x[k][0], x[k][1], x[k][2]);
    };
    auto project = [&](const BodyTet& b) {
        uint32_t id[4];
        double x[4][3];
        float w[4];
        nodes4(b.t.loc, id);
        get3(xs, id, x, w);
        const TetMaterial m = tet_material<AUX>(b.t.ax, A.comp1, A.a);
        const float Qi[3][3] = {{b.t.q0.x, b.t.q0.y, b.t.q0.z},
                                {b.t.q0.w, b.t.q1.x, b.t.q1.y},
                                {b.t.q1.z, b.t.q1.w, b.t.q2.x}};
        const float QQ[3] = {b.t.q2.y, b.t.q2.z, b.t.q2.w};
        const float QR[3] = {b.t.q3.x, b.t.q3.y, b.t.q3.z};
        if constexpr (DAMP) {
            double o[4][3];
            float unused[4];
            get3(os, id, o, unused);
            solve_tet<E, SIM, true>(yf, C, x, w, Qi, QQ, QR, b.t.q3.w, m.comp1, m.a, A.dt, o, p.damping, p.rtype);
        } else {
            solve_tet<E, SIM>(yf, C, x, w, Qi, QQ, QR, b.t.q3.w, m.comp1, m.a, A.dt);
        }
        put3(xs, id, x);
    };
    auto quad = [&](const BodyTet& b) {
        const TetMaterial m = tet_material<AUX>(b.t.ax, A.comp1, A.a);
        block_tet_quad<32>(b.t, tid & 3u, xs, yf, C, m.comp1, m.a, A.dt);
    };
    // One sweep over the colours. ta holds colour 0's tets on entry (loaded
    // with the lanes of this sweep) and on return (with those of the next
    // one): element data is loaded one phase ahead, over the sweep's end too.
    BodyTet ta, tb;
    auto sweep = [&](bool proj, bool next_proj, auto solve) {
        auto phase = [&](uint32_t c, const BodyTet& b) {
            const uint32_t first = rec[2 * c], cnt = rec[2 * c + 1];
            if (cnt == 0u) return;
            if (HQ && proj && cnt <= kBodyQuadTets) {
                if ((tid >> 2) < cnt) quad(b);
            } else {
                if (tid < cnt) solve(b);
                for (uint32_t k = tid + bs; k < cnt; k += bs) solve(load_tet(first + k));
            }
            __syncthreads();
        };
        for (uint32_t c = 0; c < A.ncol; c += 2) {
            const bool end = c + 2u >= A.ncol;
            tb = load(c + 1u, proj);
            phase(c, ta);
            ta = load(end ? 0u : c + 2u, end ? next_proj : proj);
            phase(c + 1u, tb);
        }
    };

    ta = load(0, true);
    for (uint32_t i = tid; i < n; i += bs) {
        const uint32_t k = xf_body_slot(i);
        const double4 xi = X[i], oi = O[i], vi = V[i];
        double v[3] = {vi.x, vi.y, vi.z};
        const double x[3] = {xi.x, xi.y, xi.z};
        double4 xn, on;
        predict(p, v, x, &xn, &on, xi.w, oi.w);
        xs.put(k, xn);
        os.put(k, on);
    }
    __syncthreads();
    float t_end = A.time;
    for (uint32_t s = 0; s < A.substeps; s++) {
        t_end = t_end + A.dt;
        const bool more = s + 1u < A.substeps;
        const bool passes = PASSES && (A.vpasses != 0u || A.post != 0u);
        sweep(true, !passes, project);
        if constexpr (PASSES) {
            for (uint32_t v = 0; v < A.vpasses; v++)
                sweep(false, v + 1u >= A.vpasses && A.post == 0u, [&](const BodyTet& b) {
                    if (v >= p.volume_passes) return;
                    uint32_t id[4];
                    double x[4][3];
                    float w[4];
                    nodes4(b.t.loc, id);
                    get3(xs, id, x, w);
                    volume_solve(b.t.q0, b.t.q1, b.t.q2, x, w, b.t.ax.w, A.dt);
                    put3(xs, id, x);
                });
        }
        const bool keep_v = PASSES && A.post != 0u;  // the damping passes work on stored velocities
        const double invdt = (double)p.invdt;
        for (uint32_t i = tid; i < n; i += bs) {
            const uint32_t k = xf_body_slot(i);
            const double4 xi = xs.get(k), oi = os.get(k);
            double x[3] = {xi.x, xi.y, xi.z}, v[3];
            const double o[3] = {oi.x, oi.y, oi.z};
            const double w = lock_contact(p, (uint32_t)oi.w, t_end, xi.w, o, x);
#pragma unroll
            for (int r = 0; r < 3; r++) v[r] = (x[r] - o[r]) * invdt;
            if (keep_v) {
                xs.put(k, make_double4(x[0], x[1], x[2], w));
                os.put_xyz(k, v[0], v[1], v[2]);
            } else if (more) {
                double4 xn, on;
                predict(p, v, x, &xn, &on, w, oi.w);
                xs.put(k, xn);
                os.put(k, on);
            } else {
                X[i] = make_double4(x[0], x[1], x[2], w);
                V[i] = make_double4(v[0], v[1], v[2], 0.0);
            }
        }
        __syncthreads();
        if constexpr (PASSES) {
            if (!keep_v) continue;
            const uint32_t tick = A.tick + s;
            auto on_v = [&](const BodyTet& b, auto damp) {
                uint32_t id[4];
                double x[4][3], v[4][3];
                float w[4], unused[4];
                nodes4(b.t.loc, id);
                get3(xs, id, x, w);
                get3(os, id, v, unused);
                damp(x, v, w);
                put3(os, id, v);
            };
            if (A.post & 1u)
                sweep(false, !(A.post & 2u), [&](const BodyTet& b) {
                    if (!damps_post(p, b.dm, tick)) return;
                    on_v(b, [&](const double x[4][3], double v[4][3], const float w[4]) {
                        damp_solve<E>(p, b.t.q0, b.t.q1, b.t.q2, b.t.q3, b.t.ax.x, b.t.ax.y, x, v, w, A.dt);
                    });
                });
            if (A.post & 2u)
                sweep(false, true, [&](const BodyTet& b) {
                    if (!damps_pbd(p, b.dm, tick)) return;
                    on_v(b, [&](const double x[4][3], double v[4][3], const float w[4]) {
                        pbd_solve(p, b.dm.x, x, v, w);
                    });
                });
            for (uint32_t i = tid; i < n; i += bs) {
                const uint32_t k = xf_body_slot(i);
                const double4 xi = xs.get(k), vi = os.get(k);
                double v[3] = {vi.x, vi.y, vi.z};
                const double x[3] = {xi.x, xi.y, xi.z};
                if (more) {
                    double4 xn, on;
                    predict(p, v, x, &xn, &on, xi.w, vi.w);
                    xs.put(k, xn);
                    os.put(k, on);
                } else {
                    X[i] = xi;
                    V[i] = make_double4(v[0], v[1], v[2], 0.0);
                }
            }
            __syncthreads();
        }
    }
    if (blockIdx.x == 0 && tid == 0) {
        clock[0] = t_end;
        reinterpret_cast<uint32_t*>(clock)[1] = A.tick + A.substeps;
    }
}

typedef void (*XfBodyFn)(XfBodyArgs, const uint32_t*, const uint2*, const float4*, const float4*, const float4*,
                         const float4*, const float4*, const float2*, double4*, const double4*, double4*,
                         const XfBodyParams*, float*);

// With passes or damping inside the projection the material comes from the
// per-tet slots (taux) whether or not it is uniform.
template <int E>
XfBodyFn pick_body(bool sim, bool aux, bool damp, bool passes) {
    if constexpr (E == 0 || E == 4 || E == 7)
        if (sim && !damp && !passes) {
            if constexpr (E == 0) return xf_body_steps<E, true, true, false, false>;
            else return aux ? xf_body_steps<E, true, true, false, false> : xf_body_steps<E, true, false, false, false>;
        }
    if (sim) return damp ? xf_body_steps<E, true, true, true, true> : xf_body_steps<E, true, true, false, true>;
    if constexpr (E == 0) return nullptr;
    else return damp ? xf_body_steps<E, false, true, true, true> : xf_body_steps<E, false, true, false, true>;
}

}  // namespace

// LDS bytes of a body of n slots: X and O, 32 bytes each.
extern "C" size_t xf_body_lds_bytes(uint32_t n) { return (size_t)64 * n; }

// Whether the launch reads the per-tet material slots even if the material is
// uniform.
extern "C" bool xf_body_needs_slots(int energy, bool sim, bool damp, bool passes) {
    return !((energy == 0 || energy == 4 || energy == 7) && sim && !damp && !passes);
}

// Host-callable: one step call of nbodies bodies (energy 3..7, or 0 for
// per-body MixedSel / YeohSkinFast), `threads` per workgroup.
extern "C" hipError_t xf_launch_body(hipStream_t s, int energy, bool sim, bool aux, bool damp, uint32_t threads,
                                     uint32_t nbodies, size_t lds_limit, const XfBodyArgs* args,
                                     const XfBodyData* d) {
    const bool passes = args->vpasses != 0 || args->post != 0;
    XfBodyFn fn = nullptr;
    switch (energy) {
        case 0: fn = pick_body<0>(sim, aux, damp, passes); break;
        case 3: fn = pick_body<3>(sim, aux, damp, passes); break;
        case 4: fn = pick_body<4>(sim, aux, damp, passes); break;
        case 5: fn = pick_body<5>(sim, aux, damp, passes); break;
        case 6: fn = pick_body<6>(sim, aux, damp, passes); break;
        case 7: fn = pick_body<7>(sim, aux, damp, passes); break;
        default: break;
    }
    const size_t lds = xf_body_lds_bytes(args->nmax);
    if (fn == nullptr || threads < 4 * kBodyQuadTets || threads > 512 || threads % 64 || args->ncol % 2 ||
        args->ntet == 0 || lds > lds_limit)
        return hipErrorInvalidValue;
    if (xf_body_needs_slots(energy, sim, damp, passes) && d->taux == nullptr) return hipErrorInvalidValue;
    if (nbodies == 0 || args->substeps == 0) return hipSuccess;
    if (lds > 65536) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(fn, dim3(nbodies), dim3(threads), lds, s, *args, d->rec, d->loc, d->tg0, d->tg1, d->tg2,
                       d->tg3, d->taux, d->tdmp, d->X, d->O, d->V, d->bodies, d->clock);
    return hipGetLastError();
}
