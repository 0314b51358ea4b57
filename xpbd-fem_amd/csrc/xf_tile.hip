// xf_tile.hip -- several colours of a sweep in one launch on gfx950, a
// workgroup per tile of nodes (xf_tile.h).
//
// What bounds it: a launch per colour pays a kernel boundary and two dependent
// loads from beyond L2 for one element chain (3.5 us each on 4,096 tets, most
// of the chip idle). Here one launch pays them for a span of colours, whose
// chains follow each other out of LDS; the halo tets that neighbours project
// too run on lanes that would be idle. Per substep, launches per colour
// against tiles, one to a compute unit: 24x12x12 beam of 24 colours 85 us and
// 35 (spans of 4, 9 and 11 colours, 17 own nodes a tile and up to 1,033 in LDS,
// a tet projected 14.7 times), 64x16x16 90 and 44 (4 spans of 6, 74 own nodes
// and up to 712, 3.9 times), 96x24x24 125 and 66 (4, 6, 7 and 7 colours, 3.0
// times), 128x36x36 258 and 107, the same with 31 greedy colours 255 and 137;
// 64 mixed boxes 206 and 93. The element data of a tile's
// entries is stored in entry order: read from the schedule by position, 64x16x16
// took 50.7 us (a 16-byte quarter of a line per tet and array).
#include <hip/hip_runtime.h>

#include "xf_tet.h"
#include "xf_tile.h"

namespace {

// END: the span ends the sweep; the node phase follows on the own nodes.
template <int E, bool SIM, bool AUX, bool END>
__global__ __launch_bounds__(512) void xf_tile_span(XfTileArgs A, XfTileData D, uint32_t advance) {
    extern __shared__ double4 xf_tile_nodes[];
    constexpr bool HQ = SIM && (E == 0 || E == 4 || E == 7);
    const NodeLds<kTileNodeBytes> xs{reinterpret_cast<double2*>(xf_tile_nodes)};
    const uint32_t tid = threadIdx.x, bs = blockDim.x, last = A.nent - 1u, jl = A.nph - 1u;
    if (advance && blockIdx.x == 0 && tid == 0) {
        D.clock[0] = D.clock[0] + A.dt;
        uint32_t* tick = reinterpret_cast<uint32_t*>(D.clock) + 1;
        tick[0] = tick[0] + 1u;
    }
    const uint4 m = D.meta[blockIdx.x];
    const uint2* r = D.rec + (size_t)blockIdx.x * A.nph;
    const XfBodyParams p = D.bodies[m.w];  // a copy: in scalar registers before the phases
    const float C[3] = {p.yeoh[0], p.yeoh[1], p.yeoh[2]};
    const bool yf = E == 7 || (E == 0 && p.energy == 7u);
    const uint32_t* node = D.node + m.x;

    auto load = [&](uint32_t j) {
        const uint2 e = r[min(j, jl)];
        return load_block_tet<AUX>(min(e.x + (HQ && e.y <= kTileQuadTets ? tid >> 2 : tid), last), D.loc, D.tg0, D.tg1,
                                   D.tg2, D.tg3, D.taux);
    };
    auto project = [&](const BlockTet& t) {
        const TetMaterial mt = tet_material<AUX>(t.ax, A.comp1, A.a);
        lds_tet<E, SIM>(t, xs, yf, C, mt.comp1, mt.a, A.dt);
    };
    auto phase = [&](uint32_t j, const BlockTet& t) {
        const uint2 e = r[j];
        if (HQ && e.y <= kTileQuadTets) {
            if constexpr (HQ) {
                if ((tid >> 2) < e.y) {
                    const TetMaterial mt = tet_material<AUX>(t.ax, A.comp1, A.a);
                    block_tet_quad<kTileNodeBytes>(t, tid & 3u, xs, yf, C, mt.comp1, mt.a, A.dt);
                }
            }
        } else {
            if (tid < e.y) project(t);
            for (uint32_t k = tid + bs; k < e.y; k += bs)
                project(load_block_tet<AUX>(e.x + k, D.loc, D.tg0, D.tg1, D.tg2, D.tg3, D.taux));
        }
        __syncthreads();
    };

    // element data is loaded one phase ahead
    BlockTet ta = load(0), tb;
    stage_nodes(tid, bs, m.y, node, D.Xin, xs);
    const bool own = tid < m.z;
    const uint32_t g = own ? node[tid] : 0u;
    double4 oi = make_double4(0.0, 0.0, 0.0, 0.0);
    float t_end = 0.0f;
    if constexpr (END) {
        oi = D.O[g];
        t_end = D.clock[0];
    }
    __syncthreads();
    for (uint32_t j = 0; j < A.nph; j += 2) {
        tb = load(j + 1u);
        phase(j, ta);
        if (j + 1u < A.nph) {
            ta = load(j + 2u);
            phase(j + 1u, tb);
        }
    }
    auto store = [&](uint32_t i, const double4& xi, const double4& oi) {
        if constexpr (END) {
            if (A.end == 1u) {
                finish_predict(xi, oi, i, D.Xout, D.O, p, t_end);
            } else {
                double x[3] = {xi.x, xi.y, xi.z}, v[3];
                const double o[3] = {oi.x, oi.y, oi.z};
                const double w = lock_contact(p, (uint32_t)oi.w, t_end, xi.w, o, x);
                const double invdt = (double)p.invdt;
#pragma unroll
                for (int c = 0; c < 3; c++) v[c] = (x[c] - o[c]) * invdt;
                D.Xout[i] = make_double4(x[0], x[1], x[2], w);
                D.V[i] = make_double4(v[0], v[1], v[2], 0.0);
            }
        } else {
            D.Xout[i] = xi;
        }
    };
    if (own) store(g, xs.get(tid), oi);
    for (uint32_t k = tid + bs; k < m.z; k += bs) {
        const uint32_t i = node[k];
        store(i, xs.get(k), END ? D.O[i] : oi);
    }
}

// Element data and material of the tile entries, from the schedule's.
__global__ __launch_bounds__(256) void xf_tile_fill(uint32_t n, const uint32_t* __restrict__ pos,
                                                    const float4* __restrict__ tg0, const float4* __restrict__ tg1,
                                                    const float4* __restrict__ tg2, const float4* __restrict__ tg3,
                                                    const float4* __restrict__ taux, float4* __restrict__ e0,
                                                    float4* __restrict__ e1, float4* __restrict__ e2,
                                                    float4* __restrict__ e3, float4* __restrict__ eaux) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t k = pos[i];
    e0[i] = tg0[k];
    e1[i] = tg1[k];
    e2[i] = tg2[k];
    e3[i] = tg3[k];
    if (taux != nullptr) eaux[i] = taux[k];
}

typedef void (*XfTileFn)(XfTileArgs, XfTileData, uint32_t);

template <int E>
XfTileFn pick_tile(bool sim, bool aux, bool end) {
    if (sim) {
        if (E == 0 || aux) return end ? xf_tile_span<E, true, true, true> : xf_tile_span<E, true, true, false>;
        if constexpr (E != 0) return end ? xf_tile_span<E, true, false, true> : xf_tile_span<E, true, false, false>;
    }
    if constexpr (E != 0) {
        if (aux) return end ? xf_tile_span<E, false, true, true> : xf_tile_span<E, false, true, false>;
        return end ? xf_tile_span<E, false, false, true> : xf_tile_span<E, false, false, false>;
    }
    return nullptr;
}

}  // namespace

// Host-callable: one span of ntile tiles (energy 3..7, or 0 for per-body
// MixedSel / YeohSkinFast). nmax: most nodes of a tile; lanes: most tets of a
// colour, or own nodes.
extern "C" hipError_t xf_launch_tiles(hipStream_t s, int energy, bool sim, bool aux, uint32_t ntile, uint32_t nmax,
                                      uint32_t lanes, size_t lds_limit, bool advance, const XfTileArgs* args,
                                      const XfTileData* d) {
    XfTileFn fn = nullptr;
    const bool end = args->end != 0;
    switch (energy) {
        case 0: fn = pick_tile<0>(sim, aux, end); break;
        case 3: fn = pick_tile<3>(sim, aux, end); break;
        case 4: fn = pick_tile<4>(sim, aux, end); break;
        case 5: fn = pick_tile<5>(sim, aux, end); break;
        case 6: fn = pick_tile<6>(sim, aux, end); break;
        case 7: fn = pick_tile<7>(sim, aux, end); break;
        default: break;
    }
    const size_t lds = (size_t)nmax * kTileNodeBytes;
    const uint32_t threads = xf_tile_threads(lanes);
    if (fn == nullptr || lds > lds_limit || args->nph == 0 || args->nent == 0 ||
        ((aux || energy == 0) && d->taux == nullptr))
        return hipErrorInvalidValue;
    if (ntile == 0) return hipSuccess;
    if (lds > 65536) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(fn, dim3(ntile), dim3(threads), lds, s, *args, *d, advance ? 1u : 0u);
    return hipGetLastError();
}

// Host-callable: xf_tile_fill of n entries (tg, e: four arrays; taux and eaux
// null where the launches read no material slots).
extern "C" hipError_t xf_launch_tile_fill(hipStream_t s, uint32_t n, const uint32_t* pos, float4* const tg[4],
                                          const float4* taux, float4* const e[4], float4* eaux) {
    if (n == 0) return hipSuccess;
    if (taux != nullptr && eaux == nullptr) return hipErrorInvalidValue;
    hipLaunchKernelGGL(xf_tile_fill, dim3((n + 255) / 256), dim3(256), 0, s, n, pos, tg[0], tg[1], tg[2], tg[3], taux,
                       e[0], e[1], e[2], e[3], eaux);
    return hipGetLastError();
}
