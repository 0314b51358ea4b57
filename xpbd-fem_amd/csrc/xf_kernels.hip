// xf_kernels.hip -- gfx950 kernels of the small-step XPBD substep.
//
// One tetrahedron per lane. Tets of one colour share no node, so a colour
// is swept by one launch with plain (non-atomic) gathers and scatters;
// colours run in order, which equals the reference's serial Gauss-Seidel
// sweep (GeoLinear3d::Constrain, Geo.cpp:774-788) over the colour-major
// order. Node kernels fuse pin + collisions + velocity with the next
// substep's prediction (Geo.cpp:305-344).
//
// Node state is FP64 and element arithmetic FP32, as in the reference
// (dvec3 X, O, V in Geo.h:61-64; P = Vec(X_i - X_3) in Fem.cpp:453; deltas
// added back as Dvec in Xpbd.h:212), in the reference's operation order,
// compiled with -ffp-contract=off and IEEE division/sqrt: a serial sweep of
// the same colour order on the CPU reproduces the result bit-for-bit.
//
// The file is compiled twice. As itself it holds every kernel and launcher
// of this part of the library. xf_blocks_contract.hip includes it inside
// namespace xf_contract with XF_BLOCKS_ONLY defined, compiled with
// -ffp-contract=fast: that copy keeps only the sweep-block launcher, named
// XF_BLOCKS_LAUNCH, whose kernels then fuse multiplies and adds (v_fma) and
// no longer round like the reference.
#include <hip/hip_runtime.h>

#include "xf_device.h"
#include "xf_element.h"
#include "xf_sched.h"
#include "xf_tet.h"

#ifndef XF_BLOCKS_LAUNCH
#define XF_BLOCKS_LAUNCH xf_launch_blocks
#endif

using xf::colour_grid;
using xf::colour_slot;

// ---------------------------------------------------------------- kernels

#ifndef XF_BLOCKS_ONLY
// Volume pass `pass` over one colour: tets [begin, begin+count).
__global__ __launch_bounds__(256) void xf_volume_colour(uint32_t begin, uint32_t count, uint32_t slabs, uint32_t pass,
                                                        const uint4* __restrict__ tidx,
                                                        const float4* __restrict__ tg0,
                                                        const float4* __restrict__ tg1,
                                                        const float4* __restrict__ tg2,
                                                        const float4* __restrict__ taux, double4* __restrict__ X,
                                                        const XfBodyParams* __restrict__ bodies, float dt) {
    uint32_t i = colour_slot(begin, count, slabs);
    if (i == xf::kNoSlot) return;
    volume_one(i, pass, tidx, tg0, tg1, tg2, taux, X, bodies, dt);
}
#endif  // XF_BLOCKS_ONLY

// Projects one colour: tets [begin, begin+count) of the sweep order.
// AUX: per-tet (comp1, a, body) from taux; otherwise comp1/a are uniform and
// the body is 0. The first colour launch of a substep also advances the
// simulation clock (clock != nullptr); no other kernel of the colour sweep
// reads it.
// Rayleigh post damping (Geo.cpp:797-802) of one colour.
template <int E, bool AUX>
__global__ __launch_bounds__(256) void xf_damp_colour(uint32_t begin, uint32_t count, uint32_t slabs,
                                                      const uint4* __restrict__ tidx,
                                                      const float4* __restrict__ tg0, const float4* __restrict__ tg1,
                                                      const float4* __restrict__ tg2, const float4* __restrict__ tg3,
                                                      const float4* __restrict__ taux, const float2* __restrict__ tdmp,
                                                      const double4* __restrict__ X, double4* __restrict__ V,
                                                      const XfBodyParams* __restrict__ bodies, float comp1_u,
                                                      float a_u, float dt, const float* __restrict__ clock) {
    if constexpr (E == 30) return;  // no constraint on tets, nothing to damp
    uint32_t i = colour_slot(begin, count, slabs);
    if (i == xf::kNoSlot) return;
    uint32_t tick = reinterpret_cast<const uint32_t*>(clock)[1] - 1u;
    damp_one<E, AUX>(i, tidx, tg0, tg1, tg2, tg3, taux, tdmp, X, V, bodies, comp1_u, a_u, dt, tick);
}

// PBD damping (Geo.cpp:806-809) of one colour.
template <bool AUX>
__global__ __launch_bounds__(256) void xf_pbd_colour(uint32_t begin, uint32_t count, uint32_t slabs,
                                                     const uint4* __restrict__ tidx,
                                                     const float4* __restrict__ taux, const float2* __restrict__ tdmp,
                                                     const double4* __restrict__ X, double4* __restrict__ V,
                                                     const XfBodyParams* __restrict__ bodies,
                                                     const float* __restrict__ clock) {
    uint32_t i = colour_slot(begin, count, slabs);
    if (i == xf::kNoSlot) return;
    uint32_t tick = reinterpret_cast<const uint32_t*>(clock)[1] - 1u;
    pbd_one<AUX>(i, tidx, taux, tdmp, X, V, bodies, tick);
}

template <int E, bool SIM, bool AUX, bool DAMP>
__global__ __launch_bounds__(256) void xf_project_colour(
    uint32_t begin, uint32_t count, uint32_t slabs, const uint4* __restrict__ tidx, const float4* __restrict__ tg0,
    const float4* __restrict__ tg1, const float4* __restrict__ tg2, const float4* __restrict__ tg3,
    const float4* __restrict__ taux, double4* __restrict__ X, const double4* __restrict__ O,
    const XfBodyParams* __restrict__ bodies, float comp1_u, float a_u, float dt, float* __restrict__ clock) {
    if (clock != nullptr && blockIdx.x == 0 && threadIdx.x == 0) {
        clock[0] = clock[0] + dt;
        uint32_t* tick = reinterpret_cast<uint32_t*>(clock) + 1;
        tick[0] = tick[0] + 1u;
    }
    if constexpr (E == 30) return;  // CubeNeo / CubeSkin: no constraint on tets (Fem.cpp:567-760)
    uint32_t i = colour_slot(begin, count, slabs);
    if (i == xf::kNoSlot) return;

    uint4 id = tidx[i];
    float4 q0 = tg0[i], q1 = tg1[i], q2 = tg2[i], q3 = tg3[i];
    double4 na = X[id.x], nb = X[id.y], nc = X[id.z], nd = X[id.w];
    float4 ax = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if constexpr (AUX) ax = taux[i];

    double x[4][3] = {{na.x, na.y, na.z}, {nb.x, nb.y, nb.z}, {nc.x, nc.y, nc.z}, {nd.x, nd.y, nd.z}};
    float w[4] = {(float)na.w, (float)nb.w, (float)nc.w, (float)nd.w};
    project_loaded<E, SIM, AUX, DAMP>(q0, q1, q2, q3, ax, id, x, w, O, bodies, comp1_u, a_u, dt);

    X[id.x] = make_double4(x[0][0], x[0][1], x[0][2], na.w);
    X[id.y] = make_double4(x[1][0], x[1][1], x[1][2], nb.w);
    X[id.z] = make_double4(x[2][0], x[2][1], x[2][2], nc.w);
    X[id.w] = make_double4(x[3][0], x[3][1], x[3][2], nd.w);
}

// Sweep-block projection: workgroup s of one launch colour sweeps block s
// through all of its phases. The block's nodes live in LDS for the whole
// launch; phases are separated by workgroup barriers and the nodes are
// written back at the end. Blocks of one launch colour share no node, so the
// launch equals the serial sweep of its blocks one after another, each phase
// by phase. Each lane holds one tet of the current phase and loads its
// element data for the next phase before solving the current one.
// rec: per block, nph (first schedule position, count) pairs. bnode: per
// block, nmax global node ids (xf::kNoNode past the block's nodes). tloc: per
// schedule position, the tet's four block-local node indices, 16 bits each
// (x: corners 0 | 1 << 16, y: corners 2 | 3 << 16). The first launch colour
// of a substep advances the simulation clock (clock != nullptr).
template <uint32_t NS>
__device__ __forceinline__ void write_nodes(uint32_t tid, uint32_t bs, uint32_t n, const uint32_t* __restrict__ bn,
                                            double4* __restrict__ X, NodeLds<NS> xs) {
    for (uint32_t k0 = tid; k0 < n; k0 += kStage * bs) {
        uint32_t g[kStage];
#pragma unroll
        for (uint32_t u = 0; u < kStage; u++) g[u] = bn[min(k0 + u * bs, n - 1u)];
#pragma unroll
        for (uint32_t u = 0; u < kStage; u++) {
            const uint32_t k = k0 + u * bs;
            if (k < n && g[u] != xf::kNoNode) X[g[u]] = xs.get(k);
        }
    }
}

// ntet: tets in the schedule. Element loads are issued by every lane for
// every phase pair, at clamped in-range positions (lanes without a tet, and
// the phase after the last, load data they do not use), so that the loads in
// flight are the same on every path and the wait before a phase covers
// exactly that phase's loads. OVER: some block has more tets in a phase than
// the workgroup has lanes (lanes then load and solve further tets in turn).
// FIN: the launch is the substep's last; its workgroups end the substep and
// predict the next one for every node of the scene (the node phase, fused).
// fextra holds per workgroup nmax + fmax node ids (xf::kNoNode padded): its
// block nodes as in bnode, then fmax nodes that no block of this launch
// colour touches. All are staged in LDS with their O and finished from there
// after the last phase. No other workgroup of the launch reads or writes
// those nodes, and O is not read by the projection (FIN excludes DAMP).
// ncu: compute units; pwaves: wavefronts of the largest phase, at most 4.
// tend: the clock, read for the end time of the substep (advanced by an
// earlier launch). fsingle: the scene has one body.
// PF: register sets of element data, loaded PF - 1 phases ahead. One lane per
// tet: 2 (a phase lasts 1.2 us, longer than a load, and the chain needs the
// registers). Quads: 3 (a phase lasts 0.7 us, less than a load from beyond L2:
// 1.43 against 1.44 ms per frame of the 96x24x24 beam with 2, 1.49 with 4).
template <int E, bool SIM, bool AUX, bool DAMP, bool OVER, bool FIN, bool QUAD = false, uint32_t NS = 32>
__global__ __launch_bounds__(256) void xf_project_blocks(
    uint32_t nph, uint32_t nmax, uint32_t ntet, const uint32_t* __restrict__ rec, const uint32_t* __restrict__ bnode,
    const uint2* __restrict__ tloc, const uint4* __restrict__ tidx, const float4* __restrict__ tg0,
    const float4* __restrict__ tg1, const float4* __restrict__ tg2, const float4* __restrict__ tg3,
    const float4* __restrict__ taux, double4* __restrict__ X, double4* __restrict__ O,
    const XfBodyParams* __restrict__ bodies, float comp1_u, float a_u, float dt, float* __restrict__ clock,
    const uint32_t* __restrict__ fextra, uint32_t fmax, const float* __restrict__ tend, uint32_t fsingle, uint32_t ncu, uint32_t pwaves) {
    static_assert(!(FIN && (DAMP || E == 30)), "the fused node phase needs a projection that leaves O unread");
    static_assert(!QUAD || (SIM && !DAMP && (E == 0 || E == 4 || E == 7)),
                  "quad lanes take the simultaneous MixedSel / YeohSkinFast projection without damping");
    if (clock != nullptr && blockIdx.x == 0 && threadIdx.x == 0) {
        clock[0] = clock[0] + dt;
        uint32_t* tick = reinterpret_cast<uint32_t*>(clock) + 1;
        tick[0] = tick[0] + 1u;
    }
    if constexpr (E == 30) return;  // CubeNeo / CubeSkin: no constraint on tets (Fem.cpp:567-760)
    extern __shared__ double4 xf_block_nodes[];
    const NodeLds<NS> xs{reinterpret_cast<double2*>(xf_block_nodes)};
    const uint32_t tid = threadIdx.x, bs = blockDim.x, last = ntet - 1u;
    const uint32_t* r = rec + (size_t)blockIdx.x * 2 * nph;
    const uint32_t* bn = bnode + (size_t)blockIdx.x * nmax;
    const uint32_t jl = nph - 1u;
    // FIN: LDS holds ftot nodes (the block nodes, then the extra nodes, NS
    // bytes each), then their O, then their ids
    const uint32_t ftot = FIN ? nmax + fmax : 0u;
    double4* os = FIN ? reinterpret_cast<double4*>(xs.base + (NS / 16u) * ftot) : nullptr;
    uint32_t* fs = FIN ? reinterpret_cast<uint32_t*>(os + ftot) : nullptr;
    // QUAD: four lanes per tet (block_tet_quad), bs / 4 tets at a time; else
    // one lane per tet. Where few workgroups share a compute unit (NS 48), the
    // lanes are turned by whole wavefronts so that their busy ones do not share
    // a SIMD: of the g-th workgroup of a compute unit, wavefront k was seen on
    // SIMD (k + g) mod 4, and its first tets go to the wavefront on SIMD pwaves
    // * g mod 4, pwaves wavefronts having tets in the largest phase. 269
    // workgroups of 128-tet phases on 256 compute units (64 mixed boxes): those
    // that share one took 22.6 us where the others took 15; without sharing
    // SIMDs a substep of four such launches takes 85 us, 107 before. 128x36x36
    // beam, 128-tet slots: 1.95 ms per frame, 2.35 before.
    constexpr bool TURN = NS == 48 && !QUAD;
    const uint32_t turned = TURN ? (tid + 64u * (blockIdx.x / ncu) * (5u - pwaves)) % bs : tid;
    const uint32_t lt = QUAD ? tid >> 2 : turned, per = QUAD ? bs >> 2 : bs;
    constexpr uint32_t PF = QUAD ? 3 : 2;
    // AUX: the material (ax), and with it the body, of a lane's tet is loaded
    // two phases ahead and the body's energy term one, so that neither is
    // waited for behind the element data
    auto at = [&](uint32_t j) { return min(r[2 * j] + lt, last); };
    auto load = [&](uint32_t j) {
        return load_block_tet<false>(at(j), tloc, tg0, tg1, tg2, tg3, taux);
    };
    auto load_ax = [&](uint32_t j) { return AUX ? taux[at(j)] : make_float4(0.0f, 0.0f, 0.0f, 0.0f); };
    struct Term {
        float C[3];
        uint32_t energy;
    };
    auto term = [&](const float4& ax) {
        const XfBodyParams& bp = bodies[tet_material<AUX>(ax, comp1_u, a_u).body];
        return Term{{bp.yeoh[0], bp.yeoh[1], bp.yeoh[2]}, bp.energy};
    };
    auto solve = [&](const BlockTet& t, const Term& p, uint32_t i) {
        if constexpr (DAMP) {
            lds_tet_damped<E, SIM, AUX, NS>(t, tidx[i], xs, O, bodies, comp1_u, a_u, dt);
        } else {
            const TetMaterial m = tet_material<AUX>(t.ax, comp1_u, a_u);
            const bool yf = E == 7 || (E == 0 && p.energy == 7u);
            if constexpr (QUAD) block_tet_quad<NS>(t, tid & 3u, xs, yf, p.C, m.comp1, m.a, dt);
            else lds_tet<E, SIM, NS>(t, xs, yf, p.C, m.comp1, m.a, dt);
        }
    };
    // each lane's first tet of the phase is t; with OVER, lanes go on to the
    // tets beyond the workgroup's lanes
    auto phase = [&](uint32_t j, BlockTet& t, const float4& ax, const Term& p) {
        const uint32_t b = r[2 * j], cnt = r[2 * j + 1];
        t.ax = ax;
        if (lt < cnt) solve(t, p, b + lt);
        if constexpr (OVER)
            for (uint32_t k = lt + per; k < cnt; k += per) {
                const BlockTet o = load_block_tet<AUX>(b + k, tloc, tg0, tg1, tg2, tg3, taux);
                solve(o, term(o.ax), b + k);
            }
        __syncthreads();
    };
    float4 ax = load_ax(0), ax_next = load_ax(min(1u, jl));
    Term tm = term(ax);
    BlockTet t[PF];
    t[0] = load(0);
    if constexpr (FIN) {
        // nodes, their O and their ids staged for the end of the substep
        const uint32_t* fl = fextra + (size_t)blockIdx.x * ftot;
        for (uint32_t k = tid; k < ftot; k += bs) {
            uint32_t g = fl[k];
            fs[k] = g;
            if (g != xf::kNoNode) {
                xs.put(k, X[g]);
                os[k] = O[g];
            }
        }
    } else {
        stage_nodes(tid, bs, nmax, bn, X, xs);
    }
    __syncthreads();
    // element data of phase j + PF - 1 loaded before solving phase j (set
    // j mod PF), so that the wait before a phase covers only that phase's loads
#pragma unroll
    for (uint32_t k = 1; k + 1 < PF; k++) t[k] = load(min(k, jl));
    for (uint32_t j = 0; j < nph; j += PF) {
#pragma unroll
        for (uint32_t k = 0; k < PF; k++) {
            const Term tm_next = term(ax_next);
            const float4 ax_after = load_ax(min(j + k + 2, jl));
            t[(k + PF - 1) % PF] = load(min(j + k + PF - 1, jl));
            if (k == 0 || j + k < nph) phase(j + k, t[k], ax, tm);
            ax = ax_next;
            ax_next = ax_after;
            tm = tm_next;
        }
    }
    if constexpr (FIN) {
        // (single-body scenes read the body's parameters once)
        const float t_end = tend[0];
        auto finish_all = [&](auto body_of) {
            for (uint32_t k = tid; k < ftot; k += bs) {
                uint32_t g = fs[k];
                if (g != xf::kNoNode) {
                    double4 oi = os[k];
                    finish_predict(xs.get(k), oi, g, X, O, body_of((uint32_t)oi.w), t_end);
                }
            }
        };
        if (fsingle)
            finish_all([&](uint32_t) -> const XfBodyParams& { return bodies[0]; });
        else
            finish_all([&](uint32_t flags) -> const XfBodyParams& { return bodies[flags >> 1]; });
    } else {
        write_nodes(tid, bs, nmax, bn, X, xs);
    }
}

#ifndef XF_BLOCKS_ONLY
// First prediction of a step call from the stored velocity (Xo: X, or the
// other node array of the tile launches).
__global__ __launch_bounds__(256) void xf_predict(uint32_t n, const double4* X, double4* Xo, double4* __restrict__ O,
                                                  const double4* __restrict__ V,
                                                  const XfBodyParams* __restrict__ bodies) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double4 xi = X[i];
    double4 oi = O[i];
    double4 vi = V[i];
    const XfBodyParams& p = bodies[(uint32_t)oi.w >> 1];
    double v[3] = {vi.x, vi.y, vi.z};
    double x[3] = {xi.x, xi.y, xi.z};
    predict(p, v, x, &Xo[i], &O[i], xi.w, oi.w);
}

// End of a substep: pin (Geo.cpp:318-322), collisions, velocity
// (Geo.cpp:342-344); then, if PREDICT, the next substep's prediction,
// else the velocity is stored. clock holds the end time of the substep.
// SINGLE: the scene has one body, whose parameters every node reads (loaded
// once per wave, alongside the node loads, instead of through the node's
// body id).
// SNAP: X after the sweep and O are first copied to xs_out / oo_out (the
// adjoint's replay records them for the reverse of the contact pass).
template <bool PREDICT, bool SINGLE, bool SNAP>
__global__ __launch_bounds__(256) void xf_finish(uint32_t n, double4* __restrict__ X, double4* __restrict__ O,
                                                 double4* __restrict__ V, const XfBodyParams* __restrict__ bodies,
                                                 const float* __restrict__ clock, double4* __restrict__ xs_out,
                                                 double4* __restrict__ oo_out) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double4 xi = X[i];
    double4 oi = O[i];
    if constexpr (SNAP) {
        xs_out[i] = xi;
        oo_out[i] = oi;
    }
    uint32_t flags = (uint32_t)oi.w;
    const XfBodyParams& p = bodies[SINGLE ? 0u : flags >> 1];
    double x[3] = {xi.x, xi.y, xi.z};
    double o[3] = {oi.x, oi.y, oi.z};
    const double w = lock_contact(p, flags, clock[0], xi.w, o, x);
    double v[3];
    double invdt = (double)p.invdt;
#pragma unroll
    for (int r = 0; r < 3; r++) v[r] = (x[r] - o[r]) * invdt;
    if constexpr (PREDICT) {
        predict(p, v, x, &X[i], &O[i], w, oi.w);
    } else {
        X[i] = make_double4(x[0], x[1], x[2], w);
        V[i] = make_double4(v[0], v[1], v[2], 0.0);
    }
}

// Nodes held at kinematic targets (Settings_LockRight, Geo.cpp:324-331):
// after the sweep, X = O = target and the inverse mass becomes 0.
__global__ __launch_bounds__(256) void xf_kinematic(uint32_t n, const uint32_t* __restrict__ idx,
                                                    const double4* __restrict__ target, double4* __restrict__ X,
                                                    double4* __restrict__ O) {
    uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    uint32_t i = idx[k];
    double4 t = target[k];
    X[i] = make_double4(t.x, t.y, t.z, 0.0);
    O[i] = make_double4(t.x, t.y, t.z, O[i].w);
}

// The manipulation constraint of Geo3d::Substep (Geo.cpp:334-339): m holds
// the target point and, in w, the bits of the node id (xf::kNoNode: none).
// X += (target - X) * w / (max(1e-6, w) + 1.8 / dt^2), in FP32 as there.
__global__ __launch_bounds__(64) void xf_manip(const float4* __restrict__ m, float dt, double4* __restrict__ X) {
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    const float4 t = m[0];
    const uint32_t i = __float_as_uint(t.w);
    if (i == xf::kNoNode) return;
    double4 xi = X[i];
    float w = (float)xi.w;
    float s = w / (fmaxf(0.000001f, w) + 1.8f / (dt * dt));
    float d0 = (t.x - (float)xi.x) * s, d1 = (t.y - (float)xi.y) * s, d2 = (t.z - (float)xi.z) * s;
    X[i] = make_double4(xi.x + (double)d0, xi.y + (double)d1, xi.z + (double)d2, xi.w);
}

// Forward projection of one colour that also records each tet's 4 node
// positions before the projection into tape (12 doubles per schedule
// position), for the adjoint's replay of a checkpoint window.
template <int E, bool AUX>
__global__ __launch_bounds__(256) void xf_project_record(
    uint32_t begin, uint32_t count, const uint4* __restrict__ tidx, const float4* __restrict__ tg0,
    const float4* __restrict__ tg1, const float4* __restrict__ tg2, const float4* __restrict__ tg3,
    const float4* __restrict__ taux, double4* __restrict__ X, double* __restrict__ tape,
    const XfBodyParams* __restrict__ bodies, float comp1_u, float a_u, float dt, float* __restrict__ clock) {
    if (clock != nullptr && blockIdx.x == 0 && threadIdx.x == 0) {
        clock[0] = clock[0] + dt;
        uint32_t* tick = reinterpret_cast<uint32_t*>(clock) + 1;
        tick[0] = tick[0] + 1u;
    }
    uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= count) return;
    uint32_t i = begin + k;
    uint4 id = tidx[i];
    float4 q0 = tg0[i], q1 = tg1[i], q2 = tg2[i], q3 = tg3[i];
    double4 na = X[id.x], nb = X[id.y], nc = X[id.z], nd = X[id.w];
    float comp1 = comp1_u, a = a_u;
    uint32_t body = 0;
    if constexpr (AUX) {
        float4 ax = taux[i];
        comp1 = ax.x;
        a = ax.y;
        body = __float_as_uint(ax.z);
    }
    const XfBodyParams& bp = bodies[body];
    float C[3] = {bp.yeoh[0], bp.yeoh[1], bp.yeoh[2]};
    bool yeohFast = bp.energy == 7;
    float Qi[3][3] = {{q0.x, q0.y, q0.z}, {q0.w, q1.x, q1.y}, {q1.z, q1.w, q2.x}};
    float QQ[3] = {q2.y, q2.z, q2.w};
    float QR[3] = {q3.x, q3.y, q3.z};
    double x[4][3] = {{na.x, na.y, na.z}, {nb.x, nb.y, nb.z}, {nc.x, nc.y, nc.z}, {nd.x, nd.y, nd.z}};
    float w[4] = {(float)na.w, (float)nb.w, (float)nc.w, (float)nd.w};
    double* tp = tape + 12 * (size_t)i;
#pragma unroll
    for (int n = 0; n < 4; n++)
#pragma unroll
        for (int r = 0; r < 3; r++) tp[3 * n + r] = x[n][r];
    solve_tet<E, true>(yeohFast, C, x, w, Qi, QQ, QR, q3.w, comp1, a, dt);
    X[id.x] = make_double4(x[0][0], x[0][1], x[0][2], na.w);
    X[id.y] = make_double4(x[1][0], x[1][1], x[1][2], nb.w);
    X[id.z] = make_double4(x[2][0], x[2][1], x[2][2], nc.w);
    X[id.w] = make_double4(x[3][0], x[3][1], x[3][2], nd.w);
}

// ------------------------------------------------------ persistent frame

namespace {

// Spin bound of one grid-barrier wait (each spin sleeps ~2 x 64 cycles): far
// beyond any real barrier wait, small enough that a stalled grid gives up
// within a fraction of a second.
constexpr uint32_t kBarrierSpinLimit = 1u << 21;

// Grid barrier of a co-resident grid (cooperative launch). `arrive` counts
// block arrivals since the launch (zeroed by the host before it); barrier k
// waits for k * gridDim.x arrivals. On a spin timeout the error flag is set
// and every block returns false from its next barrier, so all blocks leave
// the kernel.
__device__ __forceinline__ bool grid_barrier(uint32_t* arrive, uint32_t target, uint32_t* err) {
    __shared__ uint32_t ok;
    __syncthreads();
    if (threadIdx.x == 0) {
        __threadfence();
        __hip_atomic_fetch_add(arrive, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        uint32_t spins = 0, good = 1;
        while (__hip_atomic_load(arrive, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < target) {
            if (__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u || ++spins > kBarrierSpinLimit) {
                __hip_atomic_fetch_or(err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                good = 0;
                break;
            }
            __builtin_amdgcn_s_sleep(2);
        }
        __threadfence();
        ok = good;
    }
    __syncthreads();
    return ok != 0u;
}

template <int E, bool SIM, bool AUX, bool DAMP>
__device__ __forceinline__ void project_one(uint32_t i, const uint4* __restrict__ tidx, const float4* __restrict__ tg0,
                                            const float4* __restrict__ tg1, const float4* __restrict__ tg2,
                                            const float4* __restrict__ tg3, const float4* __restrict__ taux,
                                            double4* __restrict__ X, const double4* __restrict__ O,
                                            const XfBodyParams* __restrict__ bodies, float comp1_u, float a_u,
                                            float dt) {
    uint4 id = tidx[i];
    float4 q0 = tg0[i], q1 = tg1[i], q2 = tg2[i], q3 = tg3[i];
    double4 na = X[id.x], nb = X[id.y], nc = X[id.z], nd = X[id.w];
    float comp1 = comp1_u, a = a_u;
    uint32_t body = 0;
    if constexpr (AUX) {
        float4 ax = taux[i];
        comp1 = ax.x;
        a = ax.y;
        body = __float_as_uint(ax.z);
    }
    const XfBodyParams& bp = bodies[body];
    float C[3] = {bp.yeoh[0], bp.yeoh[1], bp.yeoh[2]};
    bool yeohFast = bp.energy == 7;
    float Qi[3][3] = {{q0.x, q0.y, q0.z}, {q0.w, q1.x, q1.y}, {q1.z, q1.w, q2.x}};
    float QQ[3] = {q2.y, q2.z, q2.w};
    float QR[3] = {q3.x, q3.y, q3.z};
    double x[4][3] = {{na.x, na.y, na.z}, {nb.x, nb.y, nb.z}, {nc.x, nc.y, nc.z}, {nd.x, nd.y, nd.z}};
    float w[4] = {(float)na.w, (float)nb.w, (float)nc.w, (float)nd.w};
    if constexpr (DAMP) {
        double4 oa = O[id.x], ob = O[id.y], oc = O[id.z], od = O[id.w];
        double o[4][3] = {{oa.x, oa.y, oa.z}, {ob.x, ob.y, ob.z}, {oc.x, oc.y, oc.z}, {od.x, od.y, od.z}};
        solve_tet<E, SIM, true>(yeohFast, C, x, w, Qi, QQ, QR, q3.w, comp1, a, dt, o, bp.damping, bp.rtype);
    } else {
        solve_tet<E, SIM>(yeohFast, C, x, w, Qi, QQ, QR, q3.w, comp1, a, dt);
    }
    X[id.x] = make_double4(x[0][0], x[0][1], x[0][2], na.w);
    X[id.y] = make_double4(x[1][0], x[1][1], x[1][2], nb.w);
    X[id.z] = make_double4(x[2][0], x[2][1], x[2][2], nc.w);
    X[id.w] = make_double4(x[3][0], x[3][1], x[3][2], nd.w);
}

// End of substep + next prediction for one node (the xf_finish body).
__device__ __forceinline__ void finish_one(uint32_t i, bool predict_next, double4* __restrict__ X,
                                           double4* __restrict__ O, double4* __restrict__ V,
                                           const XfBodyParams* __restrict__ bodies, float t_end) {
    double4 xi = X[i];
    double4 oi = O[i];
    uint32_t flags = (uint32_t)oi.w;
    const XfBodyParams& p = bodies[flags >> 1];
    double x[3] = {xi.x, xi.y, xi.z};
    double o[3] = {oi.x, oi.y, oi.z};
    const double w = lock_contact(p, flags, t_end, xi.w, o, x);
    double v[3];
    double invdt = (double)p.invdt;
#pragma unroll
    for (int r = 0; r < 3; r++) v[r] = (x[r] - o[r]) * invdt;
    if (predict_next) {
        predict(p, v, x, &X[i], &O[i], w, oi.w);
    } else {
        X[i] = make_double4(x[0], x[1], x[2], w);
        V[i] = make_double4(v[0], v[1], v[2], 0.0);
    }
}

// Prediction of one node from its stored velocity (the xf_predict body).
__device__ __forceinline__ void predict_one(uint32_t i, double4* __restrict__ X, double4* __restrict__ O,
                                            const double4* __restrict__ V, const XfBodyParams* __restrict__ bodies) {
    double4 xi = X[i];
    double4 oi = O[i];
    double4 vi = V[i];
    const XfBodyParams& p = bodies[(uint32_t)oi.w >> 1];
    double v[3] = {vi.x, vi.y, vi.z};
    double x[3] = {xi.x, xi.y, xi.z};
    predict(p, v, x, &X[i], &O[i], xi.w, oi.w);
}

}  // namespace

// A whole step call (`substeps` substeps) in one cooperative launch: the
// first prediction, then per substep every colour phase, `vpasses` rounds of
// volume colour phases and the fused finish/predict node phase, with a grid
// barrier after each phase. With post damping (post bit 0: Rayleigh post
// pass, bit 1: PBD pass) the node phase stores the velocity instead, the
// damping colour phases follow, and then a separate prediction phase. Work is
// spread over the grid by global thread index (grid-stride loops). The
// results equal the per-colour launches bit-for-bit: each tet and node runs
// the same code on the same inputs in the same phase order.
template <int E, bool SIM, bool AUX, bool DAMP>
__global__ __launch_bounds__(256) void xf_frame_persistent(
    uint32_t substeps, uint32_t ncol, uint32_t vpasses, uint32_t post, const uint32_t* __restrict__ colour_begin,
    uint32_t n_nodes, const uint4* __restrict__ tidx, const float4* __restrict__ tg0, const float4* __restrict__ tg1,
    const float4* __restrict__ tg2, const float4* __restrict__ tg3, const float4* __restrict__ taux,
    const float2* __restrict__ tdmp, double4* __restrict__ X, double4* __restrict__ O, double4* __restrict__ V,
    const XfBodyParams* __restrict__ bodies, float comp1_u, float a_u, float dt, float* __restrict__ clock,
    uint32_t* __restrict__ arrive, uint32_t* __restrict__ err) {
    const uint32_t nthreads = gridDim.x * blockDim.x;
    const uint32_t gid = blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t* tickw = reinterpret_cast<uint32_t*>(clock) + 1;
    uint32_t target = 0;
    for (uint32_t i = gid; i < n_nodes; i += nthreads) predict_one(i, X, O, V, bodies);
    target += gridDim.x;
    if (!grid_barrier(arrive, target, err)) return;
    for (uint32_t s = 0; s < substeps; s++) {
        for (uint32_t c = 0; c < ncol; c++) {
            if (c == 0 && gid == 0) {
                clock[0] = clock[0] + dt;
                tickw[0] = tickw[0] + 1u;
            }
            uint32_t begin = colour_begin[c], count = colour_begin[c + 1] - begin;
            for (uint32_t k = gid; k < count; k += nthreads)
                project_one<E, SIM, AUX, DAMP>(begin + k, tidx, tg0, tg1, tg2, tg3, taux, X, O, bodies, comp1_u, a_u,
                                               dt);
            target += gridDim.x;
            if (!grid_barrier(arrive, target, err)) return;
        }
        for (uint32_t pass = 0; pass < vpasses; pass++)
            for (uint32_t c = 0; c < ncol; c++) {
                uint32_t begin = colour_begin[c], count = colour_begin[c + 1] - begin;
                for (uint32_t k = gid; k < count; k += nthreads)
                    volume_one(begin + k, pass, tidx, tg0, tg1, tg2, taux, X, bodies, dt);
                target += gridDim.x;
                if (!grid_barrier(arrive, target, err)) return;
            }
        float t_end = clock[0];
        bool next = s + 1 < substeps;
        if (post == 0u) {
            for (uint32_t i = gid; i < n_nodes; i += nthreads) finish_one(i, next, X, O, V, bodies, t_end);
            if (next) {
                target += gridDim.x;
                if (!grid_barrier(arrive, target, err)) return;
            }
            continue;
        }
        for (uint32_t i = gid; i < n_nodes; i += nthreads) finish_one(i, false, X, O, V, bodies, t_end);
        target += gridDim.x;
        if (!grid_barrier(arrive, target, err)) return;
        uint32_t tick = tickw[0] - 1u;
        for (uint32_t kind = 0; kind < 2; kind++) {
            if (!(post & (1u << kind))) continue;
            for (uint32_t c = 0; c < ncol; c++) {
                uint32_t begin = colour_begin[c], count = colour_begin[c + 1] - begin;
                for (uint32_t k = gid; k < count; k += nthreads) {
                    if (kind == 0)
                        damp_one<E, AUX>(begin + k, tidx, tg0, tg1, tg2, tg3, taux, tdmp, X, V, bodies, comp1_u, a_u,
                                         dt, tick);
                    else
                        pbd_one<AUX>(begin + k, tidx, taux, tdmp, X, V, bodies, tick);
                }
                target += gridDim.x;
                if (!grid_barrier(arrive, target, err)) return;
            }
        }
        if (next) {
            for (uint32_t i = gid; i < n_nodes; i += nthreads) predict_one(i, X, O, V, bodies);
            target += gridDim.x;
            if (!grid_barrier(arrive, target, err)) return;
        }
    }
}

// State of n nodes between the scene's double4 records and packed triples in
// pinned host memory, where the kernel reads or writes them itself: one launch
// and one wait in place of two staged copies, a repacking loop and their
// waits. A workgroup's 256 records pass through LDS, so that the accesses over
// PCIe are whole lines. Bound by the launch and the wait on small bodies, by
// PCIe and the host's own copy on large ones (the state of the 96x24x24 beam,
// 2.9 MB: 0.34 -> 0.14 ms). x, v: nullptr to leave one out.
__global__ __launch_bounds__(256) void xf_pack_state(uint32_t n, const double4* __restrict__ X,
                                                     const double4* __restrict__ V, double* __restrict__ x,
                                                     double* __restrict__ v) {
    __shared__ double row[3 * 256];
    const uint32_t i0 = blockIdx.x * 256u, i = i0 + threadIdx.x, m = 3u * min(256u, n - i0);
    auto pack = [&](const double4* __restrict__ src, double* __restrict__ dst) {
        if (i < n) {
            const double4 a = src[i];
            row[3 * threadIdx.x] = a.x;
            row[3 * threadIdx.x + 1] = a.y;
            row[3 * threadIdx.x + 2] = a.z;
        }
        __syncthreads();
        for (uint32_t k = threadIdx.x; k < m; k += 256u) dst[3 * (size_t)i0 + k] = row[k];
        __syncthreads();
    };
    if (x) pack(X, x);
    if (v) pack(V, v);
}

// The other way: x replaces the positions of X (inverse masses stay) and of O
// (flags stay), v the velocities.
__global__ __launch_bounds__(256) void xf_unpack_state(uint32_t n, const double* __restrict__ x,
                                                       const double* __restrict__ v, double4* __restrict__ X,
                                                       double4* __restrict__ O, double4* __restrict__ V) {
    __shared__ double row[3 * 256];
    const uint32_t i0 = blockIdx.x * 256u, i = i0 + threadIdx.x, m = 3u * min(256u, n - i0);
    const uint32_t t = 3 * threadIdx.x;
    auto fetch = [&](const double* __restrict__ src) {
        __syncthreads();
        for (uint32_t k = threadIdx.x; k < m; k += 256u) row[k] = src[3 * (size_t)i0 + k];
        __syncthreads();
    };
    if (x) {
        fetch(x);
        if (i < n) {
            X[i] = make_double4(row[t], row[t + 1], row[t + 2], X[i].w);
            O[i] = make_double4(row[t], row[t + 1], row[t + 2], O[i].w);
        }
    }
    if (v) {
        fetch(v);
        if (i < n) V[i] = make_double4(row[t], row[t + 1], row[t + 2], 0.0);
    }
}

// Counts nodes whose position is not finite.
__global__ __launch_bounds__(256) void xf_count_nonfinite(uint32_t n, const double4* __restrict__ X,
                                                          uint32_t* __restrict__ count) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    bool bad = false;
    if (i < n) {
        double4 xi = X[i];
        bad = !(isfinite(xi.x) && isfinite(xi.y) && isfinite(xi.z));
    }
    unsigned long long m = __ballot(bad);
    if ((threadIdx.x & 63u) == 0 && m != 0ull) atomicAdd(count, (uint32_t)__popcll(m));
}

// ------------------------------------------------------ launch wrappers

typedef void (*XfProjectFn)(uint32_t, uint32_t, uint32_t, const uint4*, const float4*, const float4*, const float4*,
                            const float4*, const float4*, double4*, const double4*, const XfBodyParams*, float, float, float,
                            float*);


namespace {
template <int E, bool SIM>
XfProjectFn pick_aux_damp(bool aux, bool damp) {
    if (aux) return damp ? xf_project_colour<E, SIM, true, true> : xf_project_colour<E, SIM, true, false>;
    return damp ? xf_project_colour<E, SIM, false, true> : xf_project_colour<E, SIM, false, false>;
}
template <int E>
XfProjectFn pick_aux(bool sim, bool aux, bool damp) {
    return sim ? pick_aux_damp<E, true>(aux, damp) : pick_aux_damp<E, false>(aux, damp);
}
}  // namespace

// Host-callable: launch one projection kernel. energy 3..7, or 0 for
// per-body MixedSel/YeohSkinFast dispatch. damp: some body damps inside
// the projection (O is then read).
extern "C" hipError_t xf_launch_project(hipStream_t s, int energy, bool sim, bool aux, bool damp, uint32_t block,
                                        uint32_t slabs, uint32_t begin, uint32_t count, const uint4* tidx,
                                        const float4* tg0,
                                        const float4* tg1, const float4* tg2, const float4* tg3, const float4* taux,
                                        double4* X, const double4* O, const XfBodyParams* bodies, float comp1_u,
                                        float a_u, float dt, float* clock) {
    XfProjectFn fn = nullptr;
    switch (energy) {
        case 0: fn = pick_aux<0>(sim, aux, damp); break;
        case 3: fn = pick_aux<3>(sim, aux, damp); break;
        case 4: fn = pick_aux<4>(sim, aux, damp); break;
        case 5: fn = pick_aux<5>(sim, aux, damp); break;
        case 6: fn = pick_aux<6>(sim, aux, damp); break;
        case 7: fn = pick_aux<7>(sim, aux, damp); break;
        case 20: fn = pick_aux<20>(sim, aux, damp); break;
        case 22: fn = pick_aux<22>(sim, aux, damp); break;
        case 30: fn = pick_aux<30>(sim, aux, damp); break;
        default: return hipErrorInvalidValue;
    }
    if (count == 0) return hipSuccess;
    hipLaunchKernelGGL(fn, dim3(colour_grid(count, block, slabs)), dim3(block), 0, s, begin, count, slabs, tidx, tg0,
                       tg1, tg2, tg3, taux, X, O, bodies, comp1_u, a_u, dt, clock);
    return hipGetLastError();
}
#endif  // XF_BLOCKS_ONLY

typedef void (*XfBlocksFn)(uint32_t, uint32_t, uint32_t, const uint32_t*, const uint32_t*, const uint2*,
                           const uint4*, const float4*, const float4*, const float4*, const float4*, const float4*,
                           double4*, double4*, const XfBodyParams*, float, float, float, float*, const uint32_t*,
                           uint32_t, const float*, uint32_t, uint32_t, uint32_t);

namespace {
template <int E, bool OVER>
XfBlocksFn pick_blocks_quad(bool aux, bool fin) {
    if constexpr (E == 0 || E == 4 || E == 7) {
        if (fin)
            return aux ? xf_project_blocks<E, true, true, false, OVER, true, true>
                       : xf_project_blocks<E, true, false, false, OVER, true, true>;
        return aux ? xf_project_blocks<E, true, true, false, OVER, false, true>
                   : xf_project_blocks<E, true, false, false, OVER, false, true>;
    }
    return nullptr;
}
template <int E, bool SIM, bool OVER>
XfBlocksFn pick_blocks_ad(bool aux, bool damp, bool fin) {
    if (fin) {
        if constexpr (E == 30) return nullptr;
        else if (damp) return nullptr;
        else return aux ? xf_project_blocks<E, SIM, true, false, OVER, true>
                        : xf_project_blocks<E, SIM, false, false, OVER, true>;
    }
    if (aux)
        return damp ? xf_project_blocks<E, SIM, true, true, OVER, false> : xf_project_blocks<E, SIM, true, false, OVER, false>;
    return damp ? xf_project_blocks<E, SIM, false, true, OVER, false> : xf_project_blocks<E, SIM, false, false, OVER, false>;
}
// 48-byte nodes: the simultaneous MixedSel / YeohSkinFast projection without
// damping, no phase beyond the workgroup's lanes; else nullptr (the launch
// keeps 32-byte nodes)
template <int E, bool QUAD>
XfBlocksFn pick_blocks_wide_aux(bool aux, bool fin) {
    if (fin)
        return aux ? xf_project_blocks<E, true, true, false, false, true, QUAD, 48>
                   : xf_project_blocks<E, true, false, false, false, true, QUAD, 48>;
    return aux ? xf_project_blocks<E, true, true, false, false, false, QUAD, 48>
               : xf_project_blocks<E, true, false, false, false, false, QUAD, 48>;
}
template <int E>
XfBlocksFn pick_blocks_wide(bool sim, bool aux, bool damp, bool over, bool fin, bool quad) {
    if constexpr (E == 0 || E == 4 || E == 7) {
        if (!sim || damp || over) return nullptr;
        return quad ? pick_blocks_wide_aux<E, true>(aux, fin) : pick_blocks_wide_aux<E, false>(aux, fin);
    }
    return nullptr;
}
template <int E>
XfBlocksFn pick_blocks(bool sim, bool aux, bool damp, bool over, bool fin, bool quad) {
    if (quad) {
        if (!sim || damp) return nullptr;
        return over ? pick_blocks_quad<E, true>(aux, fin) : pick_blocks_quad<E, false>(aux, fin);
    }
    if (over)
        return sim ? pick_blocks_ad<E, true, true>(aux, damp, fin) : pick_blocks_ad<E, false, true>(aux, damp, fin);
    return sim ? pick_blocks_ad<E, true, false>(aux, damp, fin) : pick_blocks_ad<E, false, false>(aux, damp, fin);
}
}  // namespace

#ifndef XF_BLOCKS_ONLY
// LDS bytes of a sweep-block workgroup: its nodes in FP64, ns (32 or 48)
// bytes each.
extern "C" size_t xf_block_lds_bytes(uint32_t nmax, uint32_t ns) { return (size_t)ns * nmax; }

// LDS bytes of a workgroup of the launch that ends the substep: its nodes and
// extra nodes, each with O (32 B) and id (4 B).
extern "C" size_t xf_block_fin_lds_bytes(uint32_t nmax, uint32_t fmax, uint32_t ns) {
    return ((size_t)ns + 36) * ((size_t)nmax + fmax);
}
#else
extern "C" size_t xf_block_lds_bytes(uint32_t nmax, uint32_t ns);
extern "C" size_t xf_block_fin_lds_bytes(uint32_t nmax, uint32_t fmax, uint32_t ns);
#endif

// Host-callable: one sweep-block launch (nslot workgroups of `threads`);
// rec / bnode point at the launch colour's first block; pmax: the most tets
// of one block in one phase. fin: the launch also ends the substep and
// predicts the next for every node (fextra: per workgroup its nmax block
// nodes and fmax extra nodes; tend: the clock, not advanced by this launch;
// single_body: the scene has one body); not with damp or energy 30. quad:
// four lanes per tet (simultaneous MixedSel / YeohSkinFast without damping,
// energies 0, 4 and 7; anything else is hipErrorInvalidValue). ncu: the
// device's compute units. lds_limit:
// the device's LDS bytes per workgroup (more than 64 KiB is granted to the
// kernel with hipFuncAttributeMaxDynamicSharedMemorySize). wide: the launch
// may keep 48 bytes per node in LDS (NodeLds) where a 48-byte kernel exists
// for it and its LDS fits; *nstride (if not null) receives the bytes per
// node used.
extern "C" hipError_t XF_BLOCKS_LAUNCH(hipStream_t s, int energy, bool sim, bool aux, bool damp, uint32_t threads,
                                       uint32_t nslot, uint32_t nph, uint32_t nmax, uint32_t ntet, uint32_t pmax,
                                       const uint32_t* rec,
                                       const uint32_t* bnode, const uint2* tloc, const uint4* tidx,
                                       const float4* tg0, const float4* tg1, const float4* tg2, const float4* tg3,
                                       const float4* taux, double4* X, double4* O,
                                       const XfBodyParams* bodies, float comp1_u, float a_u, float dt,
                                       float* clock, bool fin, const uint32_t* fextra, uint32_t fmax,
                                       const float* tend, bool single_body, bool quad, uint32_t ncu, size_t lds_limit,
                                       bool wide, uint32_t* nstride) {
    XfBlocksFn fn = nullptr;
    const bool over = pmax > (quad ? threads / 4 : threads);
    uint32_t ns = 32;
    if (wide && (fin ? xf_block_fin_lds_bytes(nmax, fmax, 48) : xf_block_lds_bytes(nmax, 48)) <= lds_limit) {
        switch (energy) {
            case 0: fn = pick_blocks_wide<0>(sim, aux, damp, over, fin, quad); break;
            case 4: fn = pick_blocks_wide<4>(sim, aux, damp, over, fin, quad); break;
            case 7: fn = pick_blocks_wide<7>(sim, aux, damp, over, fin, quad); break;
            default: break;
        }
        if (fn != nullptr) ns = 48;
    }
    if (nstride != nullptr) *nstride = ns;
    if (fn == nullptr) switch (energy) {
        case 0: fn = pick_blocks<0>(sim, aux, damp, over, fin, quad); break;
        case 3: fn = pick_blocks<3>(sim, aux, damp, over, fin, quad); break;
        case 4: fn = pick_blocks<4>(sim, aux, damp, over, fin, quad); break;
        case 5: fn = pick_blocks<5>(sim, aux, damp, over, fin, quad); break;
        case 6: fn = pick_blocks<6>(sim, aux, damp, over, fin, quad); break;
        case 7: fn = pick_blocks<7>(sim, aux, damp, over, fin, quad); break;
        case 20: fn = pick_blocks<20>(sim, aux, damp, over, fin, quad); break;
        case 22: fn = pick_blocks<22>(sim, aux, damp, over, fin, quad); break;
        case 30: fn = pick_blocks<30>(sim, aux, damp, over, fin, quad); break;
        default: return hipErrorInvalidValue;
    }
    size_t lds = fin ? xf_block_fin_lds_bytes(nmax, fmax, ns) : xf_block_lds_bytes(nmax, ns);
    if (fn == nullptr || threads == 0 || threads > 256 || threads % 64 || nph == 0 || ntet == 0 || ncu == 0 ||
        lds > lds_limit)
        return hipErrorInvalidValue;
    if (fin && (tend == nullptr || clock != nullptr || fextra == nullptr)) return hipErrorInvalidValue;
    if (nslot == 0) return hipSuccess;
    if (lds > 65536) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(fn, dim3(nslot), dim3(threads), lds, s, nph, nmax, ntet, rec, bnode, tloc, tidx, tg0, tg1,
                       tg2, tg3, taux, X, O, bodies, comp1_u, a_u, dt, clock, fextra, fmax, tend,
                       single_body ? 1u : 0u, ncu, std::min(4u, (pmax + 63u) / 64u));
    return hipGetLastError();
}

#ifndef XF_BLOCKS_ONLY
typedef void (*XfDampFn)(uint32_t, uint32_t, uint32_t, const uint4*, const float4*, const float4*, const float4*,
                         const float4*, const float4*, const float2*, const double4*, double4*, const XfBodyParams*, float, float,
                         float, const float*);

namespace {
template <int E>
XfDampFn pick_damp(bool aux) {
    return aux ? xf_damp_colour<E, true> : xf_damp_colour<E, false>;
}
}  // namespace

// Rayleigh post damping of one colour (bodies with type Post/PostAmortized).
extern "C" hipError_t xf_launch_damp(hipStream_t s, int energy, bool aux, uint32_t block, uint32_t slabs,
                                     uint32_t begin, uint32_t count, const uint4* tidx, const float4* tg0, const float4* tg1,
                                     const float4* tg2, const float4* tg3, const float4* taux, const float2* tdmp,
                                     const double4* X, double4* V, const XfBodyParams* bodies, float comp1_u,
                                     float a_u, float dt, const float* clock) {
    XfDampFn fn = nullptr;
    switch (energy) {
        case 0: fn = pick_damp<0>(aux); break;
        case 3: fn = pick_damp<3>(aux); break;
        case 4: fn = pick_damp<4>(aux); break;
        case 5: fn = pick_damp<5>(aux); break;
        case 6: fn = pick_damp<6>(aux); break;
        case 7: fn = pick_damp<7>(aux); break;
        case 20: fn = pick_damp<20>(aux); break;
        case 22: fn = pick_damp<22>(aux); break;
        case 30: fn = pick_damp<30>(aux); break;
        default: return hipErrorInvalidValue;
    }
    if (count == 0) return hipSuccess;
    hipLaunchKernelGGL(fn, dim3(colour_grid(count, block, slabs)), dim3(block), 0, s, begin, count, slabs, tidx, tg0,
                       tg1, tg2, tg3, taux, tdmp, X, V, bodies, comp1_u, a_u, dt, clock);
    return hipGetLastError();
}

// PBD damping of one colour.
extern "C" hipError_t xf_launch_pbd(hipStream_t s, bool aux, uint32_t block, uint32_t slabs, uint32_t begin,
                                    uint32_t count,
                                    const uint4* tidx, const float4* taux, const float2* tdmp, const double4* X,
                                    double4* V, const XfBodyParams* bodies, const float* clock) {
    if (count == 0) return hipSuccess;
    uint32_t grid = colour_grid(count, block, slabs);
    if (aux)
        hipLaunchKernelGGL(xf_pbd_colour<true>, dim3(grid), dim3(block), 0, s, begin, count, slabs, tidx, taux, tdmp,
                           X, V, bodies, clock);
    else
        hipLaunchKernelGGL(xf_pbd_colour<false>, dim3(grid), dim3(block), 0, s, begin, count, slabs, tidx, taux, tdmp,
                           X, V, bodies, clock);
    return hipGetLastError();
}

extern "C" hipError_t xf_launch_volume(hipStream_t s, uint32_t block, uint32_t slabs, uint32_t begin, uint32_t count,
                                       uint32_t pass,
                                       const uint4* tidx, const float4* tg0, const float4* tg1, const float4* tg2,
                                       const float4* taux, double4* X, const XfBodyParams* bodies, float dt) {
    if (count == 0) return hipSuccess;
    hipLaunchKernelGGL(xf_volume_colour, dim3(colour_grid(count, block, slabs)), dim3(block), 0, s, begin, count,
                       slabs, pass, tidx, tg0, tg1, tg2, taux, X, bodies, dt);
    return hipGetLastError();
}

extern "C" hipError_t xf_launch_predict(hipStream_t s, uint32_t n, const double4* X, double4* Xo, double4* O,
                                        const double4* V, const XfBodyParams* bodies) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(xf_predict, dim3((n + 255) / 256), dim3(256), 0, s, n, X, Xo, O, V, bodies);
    return hipGetLastError();
}

extern "C" hipError_t xf_launch_finish(hipStream_t s, bool predict_next, bool single_body, uint32_t n, double4* X,
                                       double4* O, double4* V, const XfBodyParams* bodies, const float* clock) {
    if (n == 0) return hipSuccess;
    auto fn = predict_next ? (single_body ? xf_finish<true, true, false> : xf_finish<true, false, false>)
                           : (single_body ? xf_finish<false, true, false> : xf_finish<false, false, false>);
    hipLaunchKernelGGL(fn, dim3((n + 255) / 256), dim3(256), 0, s, n, X, O, V, bodies, clock, nullptr, nullptr);
    return hipGetLastError();
}

// xf_launch_finish that first copies X (after the sweep) and O to xs_out /
// oo_out.
extern "C" hipError_t xf_launch_finish_snap(hipStream_t s, bool predict_next, bool single_body, uint32_t n,
                                            double4* X, double4* O, double4* V, const XfBodyParams* bodies,
                                            const float* clock, double4* xs_out, double4* oo_out) {
    if (n == 0) return hipSuccess;
    auto fn = predict_next ? (single_body ? xf_finish<true, true, true> : xf_finish<true, false, true>)
                           : (single_body ? xf_finish<false, true, true> : xf_finish<false, false, true>);
    hipLaunchKernelGGL(fn, dim3((n + 255) / 256), dim3(256), 0, s, n, X, O, V, bodies, clock, xs_out, oo_out);
    return hipGetLastError();
}

extern "C" hipError_t xf_launch_kinematic(hipStream_t s, uint32_t n, const uint32_t* idx, const double4* target,
                                          double4* X, double4* O) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(xf_kinematic, dim3((n + 255) / 256), dim3(256), 0, s, n, idx, target, X, O);
    return hipGetLastError();
}

extern "C" hipError_t xf_launch_manip(hipStream_t s, const float4* target, float dt, double4* X) {
    hipLaunchKernelGGL(xf_manip, dim3(1), dim3(64), 0, s, target, dt, X);
    return hipGetLastError();
}

// x, v: device-visible pinned host memory (3 doubles a node; either nullptr).
extern "C" hipError_t xf_launch_pack_state(hipStream_t s, uint32_t n, const double4* X, const double4* V, double* x,
                                           double* v) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(xf_pack_state, dim3((n + 255) / 256), dim3(256), 0, s, n, X, V, x, v);
    return hipGetLastError();
}

extern "C" hipError_t xf_launch_unpack_state(hipStream_t s, uint32_t n, const double* x, const double* v, double4* X,
                                             double4* O, double4* V) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(xf_unpack_state, dim3((n + 255) / 256), dim3(256), 0, s, n, x, v, X, O, V);
    return hipGetLastError();
}

extern "C" hipError_t xf_launch_count_nonfinite(hipStream_t s, uint32_t n, const double4* X, uint32_t* count) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(xf_count_nonfinite, dim3((n + 255) / 256), dim3(256), 0, s, n, X, count);
    return hipGetLastError();
}

typedef void (*XfFrameFn)(uint32_t, uint32_t, uint32_t, uint32_t, const uint32_t*, uint32_t, const uint4*,
                          const float4*, const float4*, const float4*, const float4*, const float4*, const float2*,
                          double4*, double4*, double4*, const XfBodyParams*, float, float, float, float*, uint32_t*,
                          uint32_t*);

namespace {
template <int E, bool SIM>
XfFrameFn pick_frame_ad(bool aux, bool damp) {
    if (aux) return damp ? xf_frame_persistent<E, SIM, true, true> : xf_frame_persistent<E, SIM, true, false>;
    return damp ? xf_frame_persistent<E, SIM, false, true> : xf_frame_persistent<E, SIM, false, false>;
}
template <int E>
XfFrameFn pick_frame(bool sim, bool aux, bool damp) {
    return sim ? pick_frame_ad<E, true>(aux, damp) : pick_frame_ad<E, false>(aux, damp);
}
XfFrameFn frame_fn(int energy, bool sim, bool aux, bool damp) {
    switch (energy) {
        case 0: return pick_frame<0>(sim, aux, damp);
        case 3: return pick_frame<3>(sim, aux, damp);
        case 4: return pick_frame<4>(sim, aux, damp);
        case 5: return pick_frame<5>(sim, aux, damp);
        case 6: return pick_frame<6>(sim, aux, damp);
        case 7: return pick_frame<7>(sim, aux, damp);
        default: return nullptr;
    }
}
}  // namespace

// Largest co-resident grid of the persistent kernel at 256 threads per block.
extern "C" hipError_t xf_frame_max_blocks(int energy, bool sim, bool aux, bool damp, int* max_blocks) {
    XfFrameFn fn = frame_fn(energy, sim, aux, damp);
    if (!fn) return hipErrorInvalidValue;
    int dev = 0, per_cu = 0, cus = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e == hipSuccess) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void*)fn, 256, 0);
    if (e == hipSuccess) *max_blocks = per_cu * cus;
    return e;
}

extern "C" hipError_t xf_launch_frame(hipStream_t s, int energy, bool sim, bool aux, bool damp, uint32_t blocks,
                                      uint32_t substeps, uint32_t ncol, uint32_t vpasses, uint32_t post,
                                      const float2* tdmp, const uint32_t* colour_begin,
                                      uint32_t n_nodes, const uint4* tidx, const float4* tg0, const float4* tg1,
                                      const float4* tg2, const float4* tg3, const float4* taux, double4* X,
                                      double4* O, double4* V, const XfBodyParams* bodies, float comp1_u, float a_u,
                                      float dt, float* clock, uint32_t* arrive, uint32_t* err) {
    XfFrameFn fn = frame_fn(energy, sim, aux, damp);
    if (!fn) return hipErrorInvalidValue;
    // same order as the xf_frame_persistent parameters
    void* args[] = {&substeps, &ncol, &vpasses, &post, &colour_begin, &n_nodes, &tidx, &tg0,     &tg1, &tg2, &tg3,
                    &taux,     &tdmp, &X,       &O,    &V,            &bodies,  &comp1_u, &a_u, &dt,  &clock,
                    &arrive,   &err};
    return hipLaunchCooperativeKernel((const void*)fn, dim3(blocks), dim3(256), args, 0, s);
}

extern "C" hipError_t xf_launch_project_record(hipStream_t s, int energy, bool aux, uint32_t begin, uint32_t count,
                                               const uint4* tidx, const float4* tg0, const float4* tg1,
                                               const float4* tg2, const float4* tg3, const float4* taux, double4* X,
                                               double* tape, const XfBodyParams* bodies, float comp1_u, float a_u,
                                               float dt, float* clock) {
    if (count == 0) return hipSuccess;
    dim3 grid((count + 63) / 64), block(64);
#define XF_REC(E, A) hipLaunchKernelGGL((xf_project_record<E, A>), grid, block, 0, s, begin, count, tidx, tg0, tg1, \
                                        tg2, tg3, taux, X, tape, bodies, comp1_u, a_u, dt, clock)
    switch (energy) {
        case 0: if (aux) XF_REC(0, true); else XF_REC(0, false); break;
        case 4: if (aux) XF_REC(4, true); else XF_REC(4, false); break;
        case 7: if (aux) XF_REC(7, true); else XF_REC(7, false); break;
        default: return hipErrorInvalidValue;
    }
#undef XF_REC
    return hipGetLastError();
}
#endif  // XF_BLOCKS_ONLY
