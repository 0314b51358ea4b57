// xf_rings.hip -- gfx950 kernels of the vertex-ring ("continuous") energies:
// Energy_ContinuousPixar (8), Energy_ContinuousMixed (9) and
// Energy_ContinuousSkin (10). For these GeoLinear3d::Constrain sweeps vertex
// rings instead of tets (Geo.cpp:783-786): ring v gathers a volume-weighted
// I1 and J over the tets around v and their gradients on every ring node
// (SolveRing, Geo.cpp:148-188; CalculateElementEnergyAndGradients,
// Fem.cpp:941-973), then solves one or two coupled XPBD constraints over all
// of them (SolveSimplex, Geo.cpp:13-64; Xpbd.h:87-263).
//
// Rings of one colour share no node (the host colours the ring conflict
// graph), so a colour is one launch with plain gathers and scatters, and
// colours in order equal the reference's serial sweep over the colour-major
// ring order. Inside a launch a team of 16, 32, 64 or 128 lanes works on one
// ring, in LDS, in phases (no barrier between them for a team of one
// wavefront):
//   0  load the ring's FP64 node positions and its tets (the ring volume, a
//      sum of rest volumes, comes precomputed in the same order);
//   1  per ring tet (lanes in parallel): I1 and J of the tet and their
//      weighted gradient contributions at its 4 corners;
//   2  the contributions of each node's tets added in ring-tet order, a lane
//      per node and component (host-built incidence lists; phase 1 wrote them
//      in that order), beside two lanes that add the energy terms;
//   3  per ring node: SolveSimplex's scaling and the terms of the constraint
//      sums; then every lane adds the sums in ring-node order and forms the
//      Lagrange multipliers;
//   4  per ring node: the position (or velocity) update.
// Every sum keeps the reference's order (ring tets in OneRing order, ring
// nodes in OneRing order), compiled with -ffp-contract=off: a serial CPU
// sweep of the same ring order reproduces the result bit for bit.
//
// What bounds it: a colour holds few rings (376 of 24 tets on the 48x12x12
// beam) and each is one chain of instructions, four cycles apiece, on a
// wavefront that is alone on its SIMD. With 32 lanes a ring, a lane per node in
// phase 2 and workgroup barriers it took 14,200 cycles (a colour launch 7.15
// us): 2,900 in three dependent loads (now two: a ring's first kRingFirst nodes
// and tets are found by its index), 3,650 in phase 2 (the ring's own vertex has
// every tet: 24 times six values for one lane), 4,100 in scaling, terms and
// sums through LDS, 930 in multipliers formed by one lane. Now 9,800 with 32
// lanes (5.13 us), 8,900 with 64, 8,400 with 128 (4.63).
#include <hip/hip_runtime.h>

#include "xf_device.h"
#include "xf_element.h"
#include "xf_sched.h"

namespace {

// Floats per ring tet in LDS: five entries of six, four of the tet's I1 and J
// gradient contributions at its corners, at the corners' entries of the
// incidence lists, and one that starts with its weighted I1 and J.
constexpr uint32_t kTetFloats = 6 * 5;

// LDS of one ring team: entries [5 tmax][6] (corners in incidence-entry order,
// then the tets; reused for the terms of the constraint sums), positions
// [3][nmax] double, inverse masses [nmax], gradients [6][nmax] (g0 xyz, g1
// xyz), the nodes' incidence lists (first entry, end) [nmax], the two energy
// sums.
__host__ __device__ inline size_t ring_round16(size_t b) { return (b + 15) & ~(size_t)15; }
__host__ __device__ inline size_t ring_entry_bytes(uint32_t nmax, uint32_t tmax) {
    const size_t e = (size_t)tmax * kTetFloats, t = 5 * ring_round16(nmax);
    return ring_round16(4 * (e > t ? e : t));
}
__host__ __device__ inline size_t ring_team_bytes(uint32_t nmax, uint32_t tmax) {
    return ring_entry_bytes(nmax, tmax) + ring_round16(8 * 3 * (size_t)nmax + 4 * ((size_t)nmax * (1 + 6 + 1) + 2));
}

struct Team {
    double* xs;
    float *ws, *g, *c, *sc;
    uint32_t* seg;
    uint32_t nmax;
    __device__ double& x(uint32_t r, uint32_t n) const { return xs[r * nmax + n]; }
};

// LDS writes of a team's lanes before, reads after. The lanes of up to 64 are
// of one wavefront, whose LDS accesses complete in order: only the compiler is
// held. Every lane of a workgroup reaches every barrier.
template <uint32_t LANES>
__device__ __forceinline__ void team_sync() {
    if constexpr (LANES > 64u) {
        __syncthreads();
    } else {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
}

// A value that the lanes of a team share, in a scalar register where a team is
// of whole wavefronts (its loads and branches are then scalar too).
template <uint32_t LANES>
__device__ __forceinline__ uint32_t team_value(uint32_t v) {
    return LANES >= 64u ? (uint32_t)__builtin_amdgcn_readfirstlane((int)v) : v;
}

// a[0] + a[6] + a[12] + ... (n terms), in order from 0. Eight loads are in
// flight at a time, those past the last term in a remainder not used (they lie
// in the team's own LDS: up to 32 floats past its entries, where the nodes'
// part follows with 14 floats a node, four nodes and more); adding 0 in their
// place is exact, as the sum is never -0.
__device__ __forceinline__ float ordered_sum(const float* a, uint32_t n) {
    float s = 0.0f;
    for (; n >= 8u; n -= 8u, a += 48) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = a[6 * u];
#pragma unroll
        for (int u = 0; u < 8; u++) s = s + v[u];
    }
    if (n > 0u) {
        float v[7];
#pragma unroll
        for (int u = 0; u < 7; u++) v[u] = a[6 * u];
#pragma unroll
        for (uint32_t u = 0; u < 7; u++) s = s + (u < n ? v[u] : 0.0f);
    }
    return s;
}

using xf::adjdet;
using xf::dot3;

// Phase 1 for ring tet k (CalculateElementEnergyAndGradients for a linear
// tet, Fem.cpp:941-973): entry 4 nt + k holds w_t I1 and w_t J and, for corner
// j, its incidence entry w_t dI1/dx_j and w_t dJ/dx_j, with w_t = (V_t / 4) /
// V. The sums of phase 2 then read each node's entries, and the energies, at
// one stride. a, b, d: the tet's record. I, V: the I1 half, the J half.
template <bool I, bool V>
__device__ __forceinline__ void ring_tet(const Team& T, float4 a, float4 b, float4 d, uint32_t k, uint32_t nt) {
    const uint32_t bits = __float_as_uint(d.y), e01 = __float_as_uint(d.z), e23 = __float_as_uint(d.w);
    const uint32_t li[4] = {bits & 255u, (bits >> 8) & 255u, (bits >> 16) & 255u, bits >> 24};
    const uint32_t en[4] = {e01 & 0xFFFFu, e01 >> 16, e23 & 0xFFFFu, e23 >> 16};
    float P[3][3];
    for (int i = 0; i < 3; i++)
        for (uint32_t r = 0; r < 3; r++) P[i][r] = (float)(T.x(r, li[i]) - T.x(r, li[3]));
    const float ew = b.z;
    float* slot[4];
    for (int n = 0; n < 4; n++) slot[n] = T.c + 6 * en[n];
    float* sum = T.c + 6 * (4 * nt + k);
    if constexpr (I) {
        // CalculateIncompressibleNeoHookeanEnergyAndGradients (Fem.cpp:164-190)
        const float QQ[3] = {a.x, a.y, a.z}, QR[3] = {a.w, b.x, b.y};
        float I1 = 0.0f, gI[4][3];
        for (int i = 0; i < 3; i++) {
            I1 = I1 + QQ[i] * dot3(P[i], P[i]);
            for (int r = 0; r < 3; r++) gI[i][r] = (2.0f * QQ[i]) * P[i][r];
        }
        int q = 0;
        for (int i = 0; i < 3; i++)
            for (int j = i + 1; j < 3; j++) {
                I1 = I1 + QR[q] * dot3(P[i], P[j]);
                for (int r = 0; r < 3; r++) gI[i][r] = gI[i][r] + QR[q] * P[j][r];
                for (int r = 0; r < 3; r++) gI[j][r] = gI[j][r] + QR[q] * P[i][r];
                ++q;
            }
        for (int r = 0; r < 3; r++) gI[3][r] = ((0.0f - gI[0][r]) - gI[1][r]) - gI[2][r];
        sum[0] = ew * I1;
        for (int n = 0; n < 4; n++)
            for (int r = 0; r < 3; r++) slot[n][r] = ew * gI[n][r];
    }
    if constexpr (V) {
        // J of the tet from mat3 PP with rows P_i (Fem.cpp:960-970)
        float M[3][3], adj[3][3];
        for (int j = 0; j < 3; j++)
            for (int r = 0; r < 3; r++) M[j][r] = P[r][j];
        float det = adjdet(M, adj);
        float J = b.w * det;
        sum[1] = ew * J;
        const float sJ = d.x;
        for (int n = 0; n < 3; n++)
            for (int r = 0; r < 3; r++) slot[n][3 + r] = sJ * adj[n][r];
        for (int r = 0; r < 3; r++) slot[3][3 + r] = sJ * (((-adj[0][r]) - adj[1][r]) - adj[2][r]);
    }
}

// One colour of the ring sweep. POST = false: project positions
// (GeoLinear3d::Constrain), the first colour of a substep advancing the
// clock (clock != nullptr). POST = true: the Rayleigh post pass on V
// (GeoLinear3d::Damp, Geo.cpp:802-804) of bodies with type Post or
// PostAmortized and damping > 0, over the amortized eighth of the body's
// ring order when PostAmortized (damping x 8).
template <bool POST, uint32_t LANES>
__global__ __launch_bounds__(256) void xf_ring_colour(
    uint32_t begin, uint32_t count, uint32_t slabs, uint32_t nmax, uint32_t tmax, const uint4* __restrict__ rmeta,
    const uint4* __restrict__ rinfo, const uint2* __restrict__ rnode, const float4* __restrict__ rtet,
    const uint2* __restrict__ rnode_more, const float4* __restrict__ rtet_more, double4* __restrict__ X,
    const double4* __restrict__ O, double4* __restrict__ V, const XfBodyParams* __restrict__ bodies, float dt,
    float* __restrict__ clock) {
    extern __shared__ double2 xf_ring_lds[];
    if (!POST && clock != nullptr && blockIdx.x == 0 && threadIdx.x == 0) {
        clock[0] = clock[0] + dt;
        uint32_t* tick = reinterpret_cast<uint32_t*>(clock) + 1;
        tick[0] = tick[0] + 1u;
    }
    const uint32_t lane = threadIdx.x % LANES, team = threadIdx.x / LANES;
    Team T;
    T.nmax = nmax;
    T.c = reinterpret_cast<float*>(reinterpret_cast<char*>(xf_ring_lds) + team * ring_team_bytes(nmax, tmax));
    T.xs = reinterpret_cast<double*>(reinterpret_cast<char*>(T.c) + ring_entry_bytes(nmax, tmax));
    T.ws = reinterpret_cast<float*>(T.xs + 3 * nmax);
    T.g = T.ws + nmax;
    T.seg = reinterpret_cast<uint32_t*>(T.g + 6 * nmax);
    T.sc = reinterpret_cast<float*>(T.seg + nmax);

    // Phase 0. A lane's first node and tet are found by the ring's index, so
    // only the node's position waits for another load. A team without a ring
    // (colour tail, or a body the damping pass skips) loads the colour's first
    // and has nn = nt = 0.
    const uint32_t i = team_value<LANES>(xf::colour_slot(begin, count, slabs, LANES));
    const uint32_t ic = i == xf::kNoSlot ? begin : i;
    uint4 m = rmeta[ic];
    const uint4 info = rinfo[ic];
    uint2 nd = rnode[(size_t)ic * kRingFirst + min(lane, kRingFirst - 1u)];
    // with 128 lanes the second wavefront takes the J halves of the tets
    const uint32_t tl = LANES > 64u ? lane & 63u : lane, lf = min(tl, kRingFirst - 1u);
    const float4* tf = rtet + (size_t)ic * 3 * kRingFirst;
    float4 ta = tf[lf], tb = tf[kRingFirst + lf], td = tf[2 * kRingFirst + lf];
    double4 x0 = X[nd.x];
    const float volume = __uint_as_float(info.z);
    const XfBodyParams& bp = bodies[team_value<LANES>(info.x)];
    const uint32_t energy = bp.energy, rtype = bp.rtype;
    const float compliance = bp.compliance, C0 = bp.yeoh[0], C1 = bp.yeoh[1], C2 = bp.yeoh[2];
    float damp = bp.damping;
    if (i == xf::kNoSlot) {
        m = make_uint4(0, 0, 0, 0);
    } else {
        if (POST) {
            bool on = rtype >= 2u && damp > 0.0f;
            if (on && rtype == 3u) {
                uint32_t k8 = (reinterpret_cast<const uint32_t*>(clock)[1] - 1u) % 8u;
                uint32_t lo = bp.n_rings * k8 / 8u, hi = bp.n_rings * (k8 + 1u) / 8u;
                on = info.y >= lo && info.y < hi;
                damp = damp * 8.0f;
            }
            if (!on) m = make_uint4(0, 0, 0, 0);
        }
    }
    const uint32_t nn = team_value<LANES>(m.y), nt = team_value<LANES>(m.w);
    auto node_of = [&](uint32_t n) {
        return n < kRingFirst ? rnode[(size_t)ic * kRingFirst + n] : rnode_more[m.x + n - kRingFirst];
    };
    auto put_node = [&](uint32_t n, const uint2& d, const double4& x) {
        T.x(0, n) = x.x;
        T.x(1, n) = x.y;
        T.x(2, n) = x.z;
        T.ws[n] = (float)x.w;
        T.seg[n] = d.y;
    };
    if (lane < nn) {
        if (LANES > kRingFirst && lane >= kRingFirst) {
            nd = node_of(lane);
            x0 = X[nd.x];
        }
        put_node(lane, nd, x0);
    }
    for (uint32_t n = lane + LANES; n < nn; n += LANES) {
        const uint2 d = node_of(n);
        put_node(n, d, X[d.x]);
    }
    team_sync<LANES>();

    // Phase 1: per ring tet.
    for (uint32_t k = tl; k < nt; k += LANES > 64u ? 64u : LANES) {
        if (k >= kRingFirst) {
            const float4* t = rtet_more + 3 * (size_t)(m.z + k - kRingFirst);
            ta = t[0];
            tb = t[1];
            td = t[2];
        } else if (k != tl) {
            ta = tf[k];
            tb = tf[kRingFirst + k];
            td = tf[2 * kRingFirst + k];
        }
        if constexpr (LANES > 64u) {
            if (threadIdx.x & 64u) ring_tet<false, true>(T, ta, tb, td, k, nt);
            else ring_tet<true, false>(T, ta, tb, td, k, nt);
        } else {
            ring_tet<true, true>(T, ta, tb, td, k, nt);
        }
    }
    team_sync<LANES>();

    // Phase 2. Items 0 to 5: the components of the ring's own vertex, which is
    // a corner of every tet; 6 and 7: the energies; then node 1's components
    // and so on. The first eight lanes take one of the long ones each, the
    // others go on through the rest.
    if (nt > 0) {
        const uint32_t items = 6u * nn + 2u;
        for (uint32_t it = lane; it < items; it += lane < 8u ? items : LANES - 8u) {
            const bool energy_sum = it == 6u || it == 7u;
            const uint32_t q = it < 6u ? it : it - 2u, n = energy_sum ? 0u : q / 6u, r = energy_sum ? it - 6u : q - 6u * n;
            const uint32_t e = T.seg[n], e0 = energy_sum ? 4u * nt : e & 0xFFFFu, e1 = energy_sum ? 5u * nt : e >> 16;
            const float sum = ordered_sum(T.c + 6 * e0 + r, e1 - e0);
            (energy_sum ? T.sc : T.g + n)[r * (energy_sum ? 1u : nmax)] = sum;
        }
    }
    team_sync<LANES>();

    // Phase 3: SolveSimplex (Geo.cpp:13-64): constants and gradient scaling.
    float I1 = 0.0f, J = 0.0f, U0 = 0.0f, U1 = 0.0f, comp0 = 0.0f, comp1 = 0.0f;
    float sc = 1.0f, s1 = 0.0f;
    const float mu = bp.ring_mu, lambda = bp.ring_lambda, a = bp.ring_a;
    const bool two = energy != 8u, skin = energy == 10u;
    const bool damped_proj = !POST && damp > 0.0f && rtype < 2u;
    if (nt > 0) {
        I1 = T.sc[0];
        J = T.sc[1];
        if (!two) {
            comp0 = compliance / volume;
            U0 = fmaxf(0.0000001f, (mu / 2.0f) * I1 + (lambda / 2.0f) * (J - a) * (J - a));
        } else {
            comp0 = 1.0f / (mu * volume);
            comp1 = 1.0f / (lambda * volume);
            U0 = I1;
            if (skin) {
                float IM = I1 - 3.0f;
                U0 = fmaxf(0.0001f, C0 * IM + C1 * IM * IM + C2 * IM * IM * IM);
                sc = C0 + 2.0f * C1 * IM + 3.0f * C2 * IM * IM;
            }
            U1 = (J - a) * (J - a);
            s1 = 2.0f * (J - a);
        }
    }
    // the scaled gradients of ring node n
    auto scaled = [&](uint32_t n, float g0[3], float g1[3]) {
        for (uint32_t r = 0; r < 3; r++) {
            const float u = T.g[r * nmax + n], v = T.g[(3 + r) * nmax + n];
            if (!two) {
                g0[r] = (mu / 2.0f) * u + (lambda / 2.0f) * 2.0f * (J - a) * v;
                g1[r] = v;
            } else {
                g0[r] = skin ? u * sc : u;
                g1[r] = v * s1;
            }
        }
    };

    // The constraint sums, each in ring-node order (the sums of
    // Xpbd.h:87-263):
    //   wgg[0] = 1e-22 + sum w g0.g0     wgg[1] = 1e-22 + sum w g1.g0
    //   wgg[2] = 1e-22 + sum w g1.g1     gV[0] = sum +-g0.v, gV[1] = sum +-g1.v
    // with v = X - O (projection) or V (damping pass, where the two-constraint
    // RayleighDamp sums -g.v). A lane per node forms the terms, into the
    // entries, free after phase 2; then every lane adds them. Multiplying by 1 and negating are
    // exact, so each sum rounds as the reference's does; the padding to sixteen
    // terms adds 0 to sums that are never -0.
    const bool with_v = POST || damped_proj;
    const uint32_t n16 = (nn + 15u) & ~15u;
    float g0[3] = {0.0f, 0.0f, 0.0f}, g1[3] = {0.0f, 0.0f, 0.0f};  // of the lane's first node
    if (nt > 0)
        for (uint32_t n = lane; n < n16; n += LANES) {
            float h0[3], h1[3], t[5] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
            if (n < nn) {
                scaled(n, h0, h1);
                if (n == lane)
                    for (int r = 0; r < 3; r++) {
                        g0[r] = h0[r];
                        g1[r] = h1[r];
                    }
                const float w = T.ws[n];
                t[0] = w * dot3(h0, h0);
                t[1] = w * dot3(h1, h0);
                t[2] = w * dot3(h1, h1);
                if (with_v) {
                    const uint32_t id = n == lane ? nd.x : node_of(n).x;
                    float v[3];
                    if (POST) {
                        const double4 vd = V[id];
                        v[0] = (float)vd.x;
                        v[1] = (float)vd.y;
                        v[2] = (float)vd.z;
                    } else {
                        const double4 o = O[id];
                        v[0] = (float)(T.x(0, n) - o.x);
                        v[1] = (float)(T.x(1, n) - o.y);
                        v[2] = (float)(T.x(2, n) - o.z);
                    }
                    t[3] = dot3(h0, v);
                    t[4] = dot3(h1, v);
                    if (POST && two) {
                        t[3] = -1.0f * t[3];
                        t[4] = -1.0f * t[4];
                    }
                }
            }
            for (uint32_t q = 0; q < 3; q++) T.c[q * n16 + n] = t[q];
            if (with_v)
                for (uint32_t q = 3; q < 5; q++) T.c[q * n16 + n] = t[q];
        }
    team_sync<LANES>();
    float wgg[3] = {1.0e-22f, 1.0e-22f, 1.0e-22f}, gV[2] = {0.0f, 0.0f};
    auto add4 = [&](uint32_t q, uint32_t n, float& acc) {
        const float4 t = *reinterpret_cast<const float4*>(T.c + q * n16 + n);
        acc = acc + t.x;
        acc = acc + t.y;
        acc = acc + t.z;
        acc = acc + t.w;
    };
    if (nt > 0) {
        for (uint32_t n = 0; n < n16; n += 16)
#pragma unroll
            for (uint32_t u = 0; u < 16; u += 4)
#pragma unroll
                for (uint32_t q = 0; q < 3; q++) add4(q, n + u, wgg[q]);
        if (with_v)
            for (uint32_t n = 0; n < n16; n += 16)
#pragma unroll
                for (uint32_t u = 0; u < 16; u += 4)
#pragma unroll
                    for (uint32_t q = 0; q < 2; q++) add4(3 + q, n + u, gV[q]);
    }

    // The Lagrange multipliers, in every lane.
    float l0 = 0.0f, l1 = 0.0f;
    if (nt > 0) {
        if (!two && !POST) {
            // EnergyXpbdConstrain (Xpbd.h:87-120)
            float alpha = comp0 / (dt * dt);
            if (damped_proj) {
                float gamma = damp / dt;
                if (rtype == 0u) {
                    float A = wgg[0] * (1.0f + gamma) + (2.0f * U0 * alpha);
                    l0 = (-2.0f * U0 - gamma * gV[0]) / A;
                } else {
                    l0 = (-2.0f * U0) / (wgg[0] + (2.0f * U0 * alpha));
                    float invBeta = comp0 / (dt * damp);
                    float A = wgg[0] + 2.0f * U0 * invBeta;
                    float b = -gV[0] - wgg[0] * l0;
                    b = b * (A / fmaxf(A, 4.0f * wgg[0]));
                    l0 = l0 + b / A;
                }
            } else {
                l0 = (-2.0f * U0) / (wgg[0] + (2.0f * U0 * alpha));
            }
        } else if (!POST) {
            // EnergyXpbdConstrainSimultaneous<2> (Xpbd.h:123-214)
            float U[2] = {U0, U1}, comp[2] = {comp0, comp1};
            float alpha[2] = {comp0 / (dt * dt), comp1 / (dt * dt)};
            float gamma = damp / dt;
            float A[3] = {wgg[0], wgg[1], wgg[2]}, b[2];
            for (int k = 0; k < 2; k++) {
                int d = 2 * k;
                if (damped_proj && rtype == 0u && gamma > 0.0f) {
                    A[d] = A[d] + (2.0f * U[k] * alpha[k]) / (1.0f + gamma);
                    b[k] = (-2.0f * U[k] - gamma * gV[k]) / (1.0f + gamma);
                } else {
                    A[d] = A[d] + 2.0f * U[k] * alpha[k];
                    b[k] = -2.0f * U[k];
                }
            }
            // Cramer's rule (Xpbd.h:173-179)
            float invA00 = 1.0f / A[0];
            float invA11 = 1.0f / A[2];
            float invDet = 1.0f / fmaxf(0.00000001f, 1.0f - (A[1] * invA00) * (A[1] * invA11));
            l0 = invDet * ((b[0] * invA00) - (A[1] * invA00) * (b[1] * invA11));
            l1 = invDet * ((b[1] * invA11) - (b[0] * invA00) * (A[1] * invA11));
            if (damped_proj && rtype == 1u && gamma > 0.0f) {
                float lam[2] = {l0, l1};
                for (int k = 0; k < 2; k++) {
                    int d = 2 * k;
                    float invBeta = comp[k] / (dt * damp);
                    A[d] = wgg[d] + 2.0f * U[k] * invBeta;
                    b[k] = b[k] * (-1.0f - alpha[k] * lam[k]);
                    b[k] = b[k] + -gV[k];
                    b[k] = b[k] * (A[d] / fmaxf(A[d], 8.0f * wgg[d]));
                }
                invA00 = 1.0f / A[0];
                invA11 = 1.0f / A[2];
                invDet = 1.0f / fmaxf(0.00000001f, 1.0f - (A[1] * invA00) * (A[1] * invA11));
                l0 = l0 + invDet * ((b[0] * invA00) - (A[1] * invA00) * (b[1] * invA11));
                l1 = l1 + invDet * ((b[1] * invA11) - (b[0] * invA00) * (A[1] * invA11));
            }
        } else if (!two) {
            // RayleighDamp, one constraint (Xpbd.h:216-230)
            float invBeta = comp0 / (dt * damp);
            l0 = -gV[0] / (2.0f * U0 * invBeta + wgg[0]);
        } else {
            // RayleighDamp, two coupled constraints (Xpbd.h:232-263); gV holds b
            float invBeta0 = comp0 / (dt * damp), invBeta1 = comp1 / (dt * damp);
            float A0 = wgg[0] + 2.0f * U0 * invBeta0;
            float A1 = wgg[1];
            float A2 = wgg[2] + 2.0f * U1 * invBeta1;
            float b0 = gV[0], b1 = gV[1];
            float invA00 = 1.0f / A0;
            float invA11 = 1.0f / A2;
            float invDet = 1.0f / fmaxf(0.00000001f, 1.0f - (A1 * invA00) * (A1 * invA11));
            l0 = invDet * ((b0 * invA00) - (A1 * invA00) * (b1 * invA11));
            l1 = invDet * ((b1 * invA11) - (b0 * invA00) * (A1 * invA11));
        }
    }

    // Phase 4: node updates.
    if (nt > 0) {
        for (uint32_t n = lane; n < nn; n += LANES) {
            const float wn = T.ws[n];
            const uint32_t id = n == lane ? nd.x : node_of(n).x;
            if (n != lane) scaled(n, g0, g1);
            if (!POST) {
                double xr[3];
                for (uint32_t r = 0; r < 3; r++) {
                    if (!two) {
                        float s = wn * l0;
                        xr[r] = T.x(r, n) + (double)(s * g0[r]);
                    } else {
                        float acc = 0.0f + l0 * g0[r];
                        acc = acc + l1 * g1[r];
                        xr[r] = T.x(r, n) + (double)(wn * acc);
                    }
                }
                // x, y, z only: w (the inverse mass) stays as stored
                double* xn = reinterpret_cast<double*>(X + id);
                xn[0] = xr[0];
                xn[1] = xr[1];
                xn[2] = xr[2];
            } else {
                double4 vd = V[id];
                double* vr[3] = {&vd.x, &vd.y, &vd.z};
                for (uint32_t r = 0; r < 3; r++) {
                    if (!two) *vr[r] = *vr[r] + (double)((wn * l0) * g0[r]);
                    else *vr[r] = *vr[r] + (double)(wn * (l0 * g0[r] + l1 * g1[r]));
                }
                V[id] = vd;
            }
        }
    }
}

}  // namespace

// LDS bytes of one ring team (nmax ring nodes, tmax ring tets at most).
extern "C" size_t xf_ring_team_bytes(uint32_t nmax, uint32_t tmax) { return ring_team_bytes(nmax, tmax); }

// One colour of the ring sweep (post = false) or of the ring damping pass
// (post = true), `teams` rings per workgroup and `lanes` (16, 32, 64 or 128)
// lanes per ring. clock: advanced by the first colour of a substep (pass it for that
// launch only); read by the damping pass for the amortized range.
extern "C" hipError_t xf_launch_rings(hipStream_t s, bool post, uint32_t lanes, uint32_t teams, uint32_t slabs,
                                      uint32_t begin, uint32_t count, uint32_t nmax, uint32_t tmax,
                                      const uint4* rmeta, const uint4* rinfo, const uint2* rnode, const float4* rtet,
                                      const uint2* rnode_more, const float4* rtet_more, double4* X, const double4* O,
                                      double4* V, const XfBodyParams* bodies, float dt, float* clock) {
    if (count == 0) return hipSuccess;
    if ((lanes != 16 && lanes != 32 && lanes != 64 && lanes != 128) || teams == 0 || teams * lanes > 256) return hipErrorInvalidValue;
    size_t lds = (size_t)teams * ring_team_bytes(nmax, tmax);
    dim3 grid(xf::colour_grid(count, teams, slabs)), block(teams * lanes);
    auto k = post ? (lanes == 16   ? xf_ring_colour<true, 16>
                     : lanes == 32 ? xf_ring_colour<true, 32>
                     : lanes == 64 ? xf_ring_colour<true, 64>
                                   : xf_ring_colour<true, 128>)
                  : (lanes == 16   ? xf_ring_colour<false, 16>
                     : lanes == 32 ? xf_ring_colour<false, 32>
                     : lanes == 64 ? xf_ring_colour<false, 64>
                                   : xf_ring_colour<false, 128>);
    hipLaunchKernelGGL(k, grid, block, lds, s, begin, count, slabs, nmax, tmax, rmeta, rinfo, rnode, rtet, rnode_more,
                       rtet_more, X, O, V, bodies, dt, clock);
    return hipGetLastError();
}
