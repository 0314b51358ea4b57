// xf_tet.h -- device functions of one tet and one node of the substep, shared
// by the kernels that sweep them: per-colour, sweep-block and persistent
// launches (xf_kernels.hip) and whole step calls of small bodies
// (xf_body.hip). Every expression keeps the reference's operation order; see
// xf_kernels.hip for the rounding. Included once more inside namespace
// xf_contract by xf_blocks_contract.hip.
#ifndef XF_TET_H
#define XF_TET_H

#include <hip/hip_runtime.h>

#include "xf_device.h"
#include "xf_element.h"
#include "xf_sched.h"

namespace {

using xf::adjdet;
using xf::apply_grad;
using xf::constrain2;
using xf::defgrad;
using xf::dot3;
using xf::gather_p;
using xf::neo_prefactored;
using xf::root_grad;
using xf::volume_term;

// I1 term by one-point quadrature (energies 3/5/6, Fem.cpp:461-477).
__device__ __forceinline__ void i1_quad_term(bool yeoh, const float C[3], const float Qi[3][3], const float P[3][3],
                                             float& U0, float g0[4][3]) {
    float F[3][3], G[3][3];
    defgrad(Qi, P, F);
    float I1 = dot3(F[0], F[0]) + dot3(F[1], F[1]) + dot3(F[2], F[2]);
    float s;
    if (!yeoh) {
        U0 = U0 + 1.0f * I1;
        s = 1.0f * 2.0f;
    } else {
        float IM = I1 - 3.0f;
        U0 = U0 + 1.0f * (C[0] * IM + C[1] * IM * IM + C[2] * IM * IM * IM);
        s = (1.0f * (C[0] + 2.0f * C[1] * IM + 3.0f * C[2] * IM * IM)) * 2.0f;
    }
#pragma unroll
    for (int c = 0; c < 3; c++)
#pragma unroll
        for (int r = 0; r < 3; r++) G[c][r] = F[r][c] * s;
    apply_grad(G, Qi, g0);
}

// EnergyXpbdConstrain without damping (Xpbd.h:110-119).
__device__ __forceinline__ void constrain1(double x[4][3], const float w[4], float U, const float g[4][3], float dt,
                                           float comp) {
    float alpha = comp / (dt * dt);
    float wgg = 1.0e-22f;
#pragma unroll
    for (int n = 0; n < 4; n++) wgg = wgg + w[n] * dot3(g[n], g[n]);
    float lp = (-2.0f * U) / (wgg + (2.0f * U * alpha));
#pragma unroll
    for (int n = 0; n < 4; n++) {
        float s = w[n] * lp;
#pragma unroll
        for (int r = 0; r < 3; r++) x[n][r] = x[n][r] + (double)(s * g[n][r]);
    }
}

// EnergyXpbdConstrain with in-projection Rayleigh damping (Xpbd.h:87-120):
// rtype Rayleigh_Paper (0) or Rayleigh_Limit (1) damp along the substep
// displacement x - o; without damping this is constrain1.
__device__ __forceinline__ void constrain1_damped(double x[4][3], const double o[4][3], const float w[4], float U,
                                                  const float g[4][3], float dt, float comp, float damp, uint32_t rtype) {
    if (!(damp > 0.0f && rtype < 2u)) {
        constrain1(x, w, U, g, dt, comp);
        return;
    }
    float alpha = comp / (dt * dt);
    float gamma = damp / dt;
    float wgg = 1.0e-22f, gV = 0.0f;
#pragma unroll
    for (int n = 0; n < 4; n++) {
        float v[3] = {(float)(x[n][0] - o[n][0]), (float)(x[n][1] - o[n][1]), (float)(x[n][2] - o[n][2])};
        wgg = wgg + w[n] * dot3(g[n], g[n]);
        gV = gV + dot3(v, g[n]);
    }
    float lp;
    if (rtype == 0u) {
        float A = wgg * (1.0f + gamma) + (2.0f * U * alpha);
        lp = (-2.0f * U - gamma * gV) / A;
    } else {
        lp = (-2.0f * U) / (wgg + (2.0f * U * alpha));
        float invBeta = comp / (dt * damp);
        float A = wgg + 2.0f * U * invBeta;
        float b = -gV - wgg * lp;
        b = b * (A / fmaxf(A, 4.0f * wgg));
        lp = lp + b / A;
    }
#pragma unroll
    for (int n = 0; n < 4; n++) {
        float s = w[n] * lp;
#pragma unroll
        for (int r = 0; r < 3; r++) x[n][r] = x[n][r] + (double)(s * g[n][r]);
    }
}

// EnergyXpbdConstrainSimultaneous<2> with in-projection Rayleigh damping,
// gamma = damp / dt on both constraints (Xpbd.h:123-214).
__device__ __forceinline__ void constrain2_damped(double x[4][3], const double o[4][3], const float w[4],
                                                  const float U[2], const float g0[4][3], const float g1[4][3],
                                                  float dt, float comp0, float comp1, float damp, uint32_t rtype) {
    if (!(damp > 0.0f && rtype < 2u)) {
        constrain2(x, w, U, g0, g1, dt, comp0, comp1);
        return;
    }
    float comp[2] = {comp0, comp1};
    float alpha[2] = {comp0 / (dt * dt), comp1 / (dt * dt)};
    float gamma = damp / dt;
    float gV[2] = {0.0f, 0.0f};
#pragma unroll
    for (int n = 0; n < 4; n++) {
        float v[3] = {(float)(x[n][0] - o[n][0]), (float)(x[n][1] - o[n][1]), (float)(x[n][2] - o[n][2])};
        gV[0] = gV[0] + dot3(g0[n], v);
        gV[1] = gV[1] + dot3(g1[n], v);
    }
    float wgg[3] = {1.0e-22f, 1.0e-22f, 1.0e-22f};
#pragma unroll
    for (int n = 0; n < 4; n++) wgg[0] = wgg[0] + w[n] * dot3(g0[n], g0[n]);
#pragma unroll
    for (int n = 0; n < 4; n++) wgg[1] = wgg[1] + w[n] * dot3(g1[n], g0[n]);
#pragma unroll
    for (int n = 0; n < 4; n++) wgg[2] = wgg[2] + w[n] * dot3(g1[n], g1[n]);
    float A[3] = {wgg[0], wgg[1], wgg[2]}, b[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        int d = 2 * i;
        if (rtype == 0u && gamma > 0.0f) {
            A[d] = A[d] + (2.0f * U[i] * alpha[i]) / (1.0f + gamma);
            b[i] = (-2.0f * U[i] - gamma * gV[i]) / (1.0f + gamma);
        } else {
            A[d] = A[d] + 2.0f * U[i] * alpha[i];
            b[i] = -2.0f * U[i];
        }
    }
    float invA00 = 1.0f / A[0];
    float invA11 = 1.0f / A[2];
    float invDet = 1.0f / fmaxf(0.00000001f, 1.0f - (A[1] * invA00) * (A[1] * invA11));
    float l0 = invDet * ((b[0] * invA00) - (A[1] * invA00) * (b[1] * invA11));
    float l1 = invDet * ((b[1] * invA11) - (b[0] * invA00) * (A[1] * invA11));
    if (rtype == 1u && gamma > 0.0f) {
        float lam[2] = {l0, l1};
#pragma unroll
        for (int i = 0; i < 2; i++) {
            int d = 2 * i;
            float invBeta = comp[i] / (dt * damp);
            A[d] = wgg[d] + 2.0f * U[i] * invBeta;
            b[i] = b[i] * (-1.0f - alpha[i] * lam[i]);
            b[i] = b[i] + -gV[i];
            b[i] = b[i] * (A[d] / fmaxf(A[d], 8.0f * wgg[d]));
        }
        invA00 = 1.0f / A[0];
        invA11 = 1.0f / A[2];
        invDet = 1.0f / fmaxf(0.00000001f, 1.0f - (A[1] * invA00) * (A[1] * invA11));
        l0 = l0 + invDet * ((b[0] * invA00) - (A[1] * invA00) * (b[1] * invA11));
        l1 = l1 + invDet * ((b[1] * invA11) - (b[0] * invA00) * (A[1] * invA11));
    }
#pragma unroll
    for (int n = 0; n < 4; n++) {
#pragma unroll
        for (int r = 0; r < 3; r++) {
            float acc = 0.0f + l0 * g0[n][r];
            acc = acc + l1 * g1[n][r];
            x[n][r] = x[n][r] + (double)(w[n] * acc);
        }
    }
}

// SolveElementMixed for a linear tet (Fem.cpp:437-564), damping off.
// SolveElementPixar's energy and root-completed gradient for a linear tet
// (Fem.cpp:362-432; one quadrature point of weight 1, so Full and Reduced
// coincide): mu = 2, lambda = 2 / (1 - 2 nu) and a = 1 + mu / lambda come in
// the per-tet material slots. SEL: PixarOptions::Selective (the J term at the
// point plus the prefactored I1 term).
template <bool SEL>
__device__ __forceinline__ void pixar_ug(const float Qi[3][3], const float QQ[3], const float QR[3],
                                         const float P[3][3], float lambda, float a, float& U, float g[4][3]) {
    const float mu = 2.0f, weight = 1.0f;
    float F[3][3], adj[3][3], G[3][3];
    defgrad(Qi, P, F);
    float u = 0.0f;
    if constexpr (!SEL) {
        float I1 = dot3(F[0], F[0]) + dot3(F[1], F[1]) + dot3(F[2], F[2]);
        u = u + weight * (mu / 2.0f) * I1;
    }
    float J = adjdet(F, adj);
    u = u + weight * (lambda / 2.0f) * ((J - a) * (J - a));
    float sJ = weight * (lambda / 2.0f) * 2.0f * (J - a);
    float sI = weight * (mu / 2.0f) * 2.0f;
#pragma unroll
    for (int c = 0; c < 3; c++)
#pragma unroll
        for (int r = 0; r < 3; r++) G[c][r] = SEL ? sJ * adj[c][r] : sI * F[r][c] + sJ * adj[c][r];
#pragma unroll
    for (int n = 0; n < 4; n++)
#pragma unroll
        for (int r = 0; r < 3; r++) g[n][r] = 0.0f;
    apply_grad(G, Qi, g);
    root_grad(g);
    if constexpr (SEL) {
        float UI1, gI1[4][3];
        neo_prefactored(QQ, QR, P, UI1, gI1);
        u = u + (mu / 2.0f) * UI1;
#pragma unroll
        for (int n = 0; n < 4; n++)
#pragma unroll
            for (int r = 0; r < 3; r++) g[n][r] = g[n][r] + (mu / 2.0f) * gI1[n][r];
    }
    U = u;
}

// E: 3 Mixed, 4 MixedSel, 5 YeohSkin, 6 YeohSkinSel, 7 YeohSkinFast,
//    0 = MixedSel or YeohSkinFast chosen per tet by `yeohFast`,
//    20 = Pixar / PixarReduced, 22 = PixarSel (comp0 = compliance / V,
//    comp1 = lambda, a from the Pixar material).
// DAMP: in-projection Rayleigh damping of the body (damp, rtype) along x - o.
template <int E, bool SIM, bool DAMP = false>
__device__ __forceinline__ void solve_tet(bool yeohFast, const float C[3], double x[4][3], const float w[4],
                                          const float Qi[3][3], const float QQ[3], const float QR[3], float comp0,
                                          float comp1, float a, float dt, const double (*o)[3] = nullptr,
                                          float damp = 0.0f, uint32_t rtype = 0u) {
    float P[3][3];
    gather_p(x, P);
    float U[2] = {0.0f, 0.0f};
    float g0[4][3], g1[4][3];
#pragma unroll
    for (int n = 0; n < 4; n++)
#pragma unroll
        for (int r = 0; r < 3; r++) { g0[n][r] = 0.0f; g1[n][r] = 0.0f; }

    if constexpr (E == 20 || E == 22) {
        pixar_ug<E == 22>(Qi, QQ, QR, P, comp1, a, U[0], g0);
        if constexpr (DAMP) constrain1_damped(x, o, w, U[0], g0, dt, comp0, damp, rtype);
        else constrain1(x, w, U[0], g0, dt, comp0);
    } else if constexpr (E == 3 || E == 5 || E == 6) {
        i1_quad_term(E != 3, C, Qi, P, U[0], g0);
        if constexpr (SIM && E != 6) volume_term(Qi, P, a, U[1], g1);
        U[0] = fmaxf(0.0001f, U[0]);
        if constexpr (SIM) {
            if constexpr (E == 6) volume_term(Qi, P, a, U[1], g1);
            root_grad(g0);
            root_grad(g1);
            if constexpr (DAMP) constrain2_damped(x, o, w, U, g0, g1, dt, comp0, comp1, damp, rtype);
            else constrain2(x, w, U, g0, g1, dt, comp0, comp1);
        } else {
            root_grad(g0);
            if constexpr (DAMP) constrain1_damped(x, o, w, U[0], g0, dt, comp0, damp, rtype);
            else constrain1(x, w, U[0], g0, dt, comp0);
            gather_p(x, P);
            volume_term(Qi, P, a, U[1], g1);
            root_grad(g1);
            if constexpr (DAMP) constrain1_damped(x, o, w, U[1], g1, dt, comp1, damp, rtype);
            else constrain1(x, w, U[1], g1, dt, comp1);
        }
    } else {
        neo_prefactored(QQ, QR, P, U[0], g0);
        bool yf = (E == 7) || (E == 0 && yeohFast);
        if (yf) {
            float IM = U[0] - 3.0f;
            U[0] = fmaxf(0.0001f, C[0] * IM + C[1] * IM * IM + C[2] * IM * IM * IM);
            float gScale = C[0] + 2.0f * C[1] * IM + 3.0f * C[2] * IM * IM;
#pragma unroll
            for (int n = 0; n < 4; n++)
#pragma unroll
                for (int r = 0; r < 3; r++) g0[n][r] = g0[n][r] * gScale;
        }
        if constexpr (!SIM) {
            if constexpr (DAMP) constrain1_damped(x, o, w, U[0], g0, dt, comp0, damp, rtype);
            else constrain1(x, w, U[0], g0, dt, comp0);
            gather_p(x, P);
        }
        volume_term(Qi, P, a, U[1], g1);
        root_grad(g1);
        if constexpr (!SIM) {
            if constexpr (DAMP) constrain1_damped(x, o, w, U[1], g1, dt, comp1, damp, rtype);
            else constrain1(x, w, U[1], g1, dt, comp1);
        } else {
            if constexpr (DAMP) constrain2_damped(x, o, w, U, g0, g1, dt, comp0, comp1, damp, rtype);
            else constrain2(x, w, U, g0, g1, dt, comp0, comp1);
        }
    }
}

// SolveVolumeOnly of one tet (Fem.cpp:840-867): the (J - 1)^2 term alone with
// compliance comp = settings.compliance * volume and a scalar XPBD update.
__device__ __forceinline__ void volume_solve(const float4& q0, const float4& q1, const float4& q2, double x[4][3],
                                             const float w[4], float comp, float dt) {
    float Qi[3][3] = {{q0.x, q0.y, q0.z}, {q0.w, q1.x, q1.y}, {q1.z, q1.w, q2.x}};
    float P[3][3];
    gather_p(x, P);
    float U = 0.0f;
    float g[4][3];
#pragma unroll
    for (int n = 0; n < 4; n++)
#pragma unroll
        for (int r = 0; r < 3; r++) g[n][r] = 0.0f;
    volume_term(Qi, P, 1.0f, U, g);
    root_grad(g);
    constrain1(x, w, U, g, dt, comp);
}

// volume_solve of tet i of the sweep order (compliance in taux.w). Bodies
// with fewer than pass + 1 volume passes skip the tet.
__device__ __forceinline__ void volume_one(uint32_t i, uint32_t pass, const uint4* __restrict__ tidx,
                                           const float4* __restrict__ tg0, const float4* __restrict__ tg1,
                                           const float4* __restrict__ tg2, const float4* __restrict__ taux,
                                           double4* __restrict__ X, const XfBodyParams* __restrict__ bodies,
                                           float dt) {
    float4 ax = taux[i];
    if (pass >= bodies[__float_as_uint(ax.z)].volume_passes) return;
    uint4 id = tidx[i];
    float4 q0 = tg0[i], q1 = tg1[i], q2 = tg2[i];
    double4 na = X[id.x], nb = X[id.y], nc = X[id.z], nd = X[id.w];
    double x[4][3] = {{na.x, na.y, na.z}, {nb.x, nb.y, nb.z}, {nc.x, nc.y, nc.z}, {nd.x, nd.y, nd.z}};
    float w[4] = {(float)na.w, (float)nb.w, (float)nc.w, (float)nd.w};
    volume_solve(q0, q1, q2, x, w, ax.w, dt);
    X[id.x] = make_double4(x[0][0], x[0][1], x[0][2], na.w);
    X[id.y] = make_double4(x[1][0], x[1][1], x[1][2], nb.w);
    X[id.z] = make_double4(x[2][0], x[2][1], x[2][2], nc.w);
    X[id.w] = make_double4(x[3][0], x[3][1], x[3][2], nd.w);
}

// U and root-completed gradients of SolveElementMixed in DampingMode::On
// (Fem.cpp:437-564 with the solve forced to Simultaneous), no projection.
template <int E>
__device__ __forceinline__ void element_ug(bool yeohFast, const float C[3], const double x[4][3], const float Qi[3][3],
                                           const float QQ[3], const float QR[3], float lambda, float a, float U[2],
                                           float g0[4][3], float g1[4][3]) {
    float P[3][3];
    gather_p(x, P);
    U[0] = 0.0f;
    U[1] = 0.0f;
#pragma unroll
    for (int n = 0; n < 4; n++)
#pragma unroll
        for (int r = 0; r < 3; r++) { g0[n][r] = 0.0f; g1[n][r] = 0.0f; }
    if constexpr (E == 20 || E == 22) {
        pixar_ug<E == 22>(Qi, QQ, QR, P, lambda, a, U[0], g0);
    } else if constexpr (E == 3 || E == 5 || E == 6) {
        i1_quad_term(E != 3, C, Qi, P, U[0], g0);
        if constexpr (E != 6) volume_term(Qi, P, a, U[1], g1);
        U[0] = fmaxf(0.0001f, U[0]);
        if constexpr (E == 6) volume_term(Qi, P, a, U[1], g1);
        root_grad(g0);
        root_grad(g1);
    } else {
        neo_prefactored(QQ, QR, P, U[0], g0);
        if ((E == 7) || (E == 0 && yeohFast)) {
            float IM = U[0] - 3.0f;
            U[0] = fmaxf(0.0001f, C[0] * IM + C[1] * IM * IM + C[2] * IM * IM * IM);
            float gScale = C[0] + 2.0f * C[1] * IM + 3.0f * C[2] * IM * IM;
#pragma unroll
            for (int n = 0; n < 4; n++)
#pragma unroll
                for (int r = 0; r < 3; r++) g0[n][r] = g0[n][r] * gScale;
        }
        volume_term(Qi, P, a, U[1], g1);
        root_grad(g1);
    }
}

// RayleighDamp, one constraint (Xpbd.h:216-230).
__device__ __forceinline__ void rayleigh1(double v[4][3], const float w[4], float U, const float g[4][3], float dt,
                                          float comp, float damp) {
    float invBeta = comp / (dt * damp);
    float wgg = 1.0e-22f, gV = 0.0f;
#pragma unroll
    for (int n = 0; n < 4; n++) {
        float vf[3] = {(float)v[n][0], (float)v[n][1], (float)v[n][2]};
        wgg = wgg + w[n] * dot3(g[n], g[n]);
        gV = gV + dot3(g[n], vf);
    }
    float lambda = -gV / (2.0f * U * invBeta + wgg);
#pragma unroll
    for (int n = 0; n < 4; n++) {
        float s = w[n] * lambda;
#pragma unroll
        for (int r = 0; r < 3; r++) v[n][r] = v[n][r] + (double)(s * g[n][r]);
    }
}

// RayleighDamp, two coupled constraints (Xpbd.h:232-263).
__device__ __forceinline__ void rayleigh2(double v[4][3], const float w[4], const float U[2], const float g0[4][3],
                                          const float g1[4][3], float dt, float comp0, float comp1, float damp) {
    float invBeta0 = comp0 / (dt * damp), invBeta1 = comp1 / (dt * damp);
    float A0 = 1.0e-22f, A1 = 1.0e-22f, A2 = 1.0e-22f, b0 = 0.0f, b1 = 0.0f;
#pragma unroll
    for (int n = 0; n < 4; n++) {
        A0 = A0 + w[n] * dot3(g0[n], g0[n]);
        A1 = A1 + w[n] * dot3(g0[n], g1[n]);
        A2 = A2 + w[n] * dot3(g1[n], g1[n]);
        float vf[3] = {(float)v[n][0], (float)v[n][1], (float)v[n][2]};
        b0 = b0 - dot3(g0[n], vf);
        b1 = b1 - dot3(g1[n], vf);
    }
    A0 = A0 + 2.0f * U[0] * invBeta0;
    A2 = A2 + 2.0f * U[1] * invBeta1;
    float invA00 = 1.0f / A0;
    float invA11 = 1.0f / A2;
    float invDet = 1.0f / fmaxf(0.00000001f, 1.0f - (A1 * invA00) * (A1 * invA11));
    float l0 = invDet * ((b0 * invA00) - (A1 * invA00) * (b1 * invA11));
    float l1 = invDet * ((b1 * invA11) - (b0 * invA00) * (A1 * invA11));
#pragma unroll
    for (int n = 0; n < 4; n++)
#pragma unroll
        for (int r = 0; r < 3; r++) v[n][r] = v[n][r] + (double)(w[n] * (l0 * g0[n][r] + l1 * g1[n][r]));
}

// cross(x, y) of vectormath.h:364.
__device__ __forceinline__ void cross3(const float x[3], const float y[3], float o[3]) {
    o[0] = x[1] * y[2] - y[1] * x[2];
    o[1] = x[2] * y[0] - y[2] * x[0];
    o[2] = x[0] * y[1] - y[0] * x[1];
}

// PbdDamp<4> for dvec3 (Xpbd.h:306-348): pull the node velocities toward the
// tet's mass-weighted rigid motion by `damping`; inertia inverted as
// inverse(mat3) does (vectormath.cpp:41-60: adjugate in FP64, det and the
// 1/det scale in FP32).
__device__ __forceinline__ void pbd_damp(const double x[4][3], double v[4][3], const float W[4], float damping) {
    float X[4][3], V[4][3], M[4];
    float Xcm[3] = {0.0f, 0.0f, 0.0f}, Vcm[3] = {0.0f, 0.0f, 0.0f};
    float Msum = 0.0f;
    float Wsum = 1.0e-8f;
#pragma unroll
    for (int i = 0; i < 4; i++) Wsum = Wsum + W[i];
    float Waverage = Wsum * (1.0f / 4.0f);
    float Wmin = 0.0001f * Waverage;
#pragma unroll
    for (int i = 0; i < 4; i++) {
#pragma unroll
        for (int r = 0; r < 3; r++) {
            X[i][r] = (float)(x[i][r] - x[3][r]);
            V[i][r] = (float)v[i][r];
        }
        M[i] = Waverage / fmaxf(Wmin, W[i]);
#pragma unroll
        for (int r = 0; r < 3; r++) Xcm[r] = Xcm[r] + X[i][r] * M[i];
#pragma unroll
        for (int r = 0; r < 3; r++) Vcm[r] = Vcm[r] + V[i][r] * M[i];
        Msum = Msum + M[i];
    }
#pragma unroll
    for (int r = 0; r < 3; r++) {
        Xcm[r] = Xcm[r] / Msum;
        Vcm[r] = Vcm[r] / Msum;
    }
    float rv[4][3], L[3] = {0.0f, 0.0f, 0.0f};
    float I[3][3] = {{0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f}};
#pragma unroll
    for (int i = 0; i < 4; i++) {
#pragma unroll
        for (int r = 0; r < 3; r++) rv[i][r] = X[i][r] - Xcm[r];
        float c[3];
        cross3(rv[i], V[i], c);
#pragma unroll
        for (int r = 0; r < 3; r++) L[r] = L[r] + M[i] * c[r];
        const float* q = rv[i];
        float rr[3] = {q[0] * q[0], q[1] * q[1], q[2] * q[2]};
        float rp[3] = {q[0] * q[1], q[1] * q[2], q[2] * q[0]};
        float K[3][3] = {{rr[2] + rr[1], -rp[0], -rp[2]}, {-rp[0], rr[2] + rr[0], -rp[1]}, {-rp[2], -rp[1], rr[1] + rr[0]}};
#pragma unroll
        for (int cc = 0; cc < 3; cc++)
#pragma unroll
            for (int r = 0; r < 3; r++) I[cc][r] = I[cc][r] + K[cc][r] * M[i];
    }
    double m00 = I[0][0], m01 = I[0][1], m02 = I[0][2];
    double m10 = I[1][0], m11 = I[1][1], m12 = I[1][2];
    double m20 = I[2][0], m21 = I[2][1], m22 = I[2][2];
    float adj[3][3];
    adj[0][0] = (float)(+(m11 * m22 - m12 * m21));
    adj[0][1] = (float)(-(m01 * m22 - m02 * m21));
    adj[0][2] = (float)(+(m01 * m12 - m02 * m11));
    adj[1][0] = (float)(-(m10 * m22 - m12 * m20));
    adj[1][1] = (float)(+(m00 * m22 - m02 * m20));
    adj[1][2] = (float)(-(m00 * m12 - m02 * m10));
    adj[2][0] = (float)(+(m10 * m21 - m11 * m20));
    adj[2][1] = (float)(-(m00 * m21 - m01 * m20));
    adj[2][2] = (float)(+(m00 * m11 - m01 * m10));
    float det = I[0][0] * adj[0][0] + I[0][1] * adj[1][0] + I[0][2] * adj[2][0];
    float inv = 1.0f / det;
    float om[3];
#pragma unroll
    for (int r = 0; r < 3; r++) om[r] = (adj[0][r] * inv) * L[0] + (adj[1][r] * inv) * L[1] + (adj[2][r] * inv) * L[2];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        float c[3];
        cross3(om, rv[i], c);
#pragma unroll
        for (int r = 0; r < 3; r++) v[i][r] = v[i][r] + (double)(damping * ((Vcm[r] + c[r]) - V[i][r]));
    }
}

// Amortized damping (Rayleigh_PostAmortized) covers sweep positions
// [T k / 8, T (k + 1) / 8) of the body, k = tickId % 8 (Geo.cpp:794-798).
__device__ __forceinline__ bool in_damp_range(const XfBodyParams& bp, float2 dm, uint32_t tick) {
    if (bp.rtype != 3u) return true;
    uint32_t k = tick % 8u;
    uint32_t pos = __float_as_uint(dm.y);
    return pos >= bp.n_tets * k / 8u && pos < bp.n_tets * (k + 1u) / 8u;
}

// Whether the Rayleigh post pass / the PBD pass of this substep covers a tet
// (dm: its surface area and position in the body's sweep order).
__device__ __forceinline__ bool damps_post(const XfBodyParams& bp, float2 dm, uint32_t tick) {
    return bp.rtype >= 2u && bp.damping > 0.0f && in_damp_range(bp, dm, tick);
}
__device__ __forceinline__ bool damps_pbd(const XfBodyParams& bp, float2 dm, uint32_t tick) {
    return bp.pbd > 0.0f && in_damp_range(bp, dm, tick);
}

// Rayleigh post damping of one tet (DampElement, Fem.cpp:910-929) on the
// velocities v of its nodes.
template <int E>
__device__ __forceinline__ void damp_solve(const XfBodyParams& bp, const float4& q0, const float4& q1,
                                           const float4& q2, const float4& q3, float comp1, float a,
                                           const double x[4][3], double v[4][3], const float w[4], float dt) {
    float damp = bp.rtype == 3u ? bp.damping * 8.0f : bp.damping;
    float C[3] = {bp.yeoh[0], bp.yeoh[1], bp.yeoh[2]};
    float Qi[3][3] = {{q0.x, q0.y, q0.z}, {q0.w, q1.x, q1.y}, {q1.z, q1.w, q2.x}};
    float QQ[3] = {q2.y, q2.z, q2.w};
    float QR[3] = {q3.x, q3.y, q3.z};
    float U[2], g0[4][3], g1[4][3];
    element_ug<E>(bp.energy == 7u, C, x, Qi, QQ, QR, comp1, a, U, g0, g1);
    if constexpr (E == 20 || E == 22) {
        rayleigh1(v, w, U[0], g0, dt, q3.w, damp);  // SolveElementPixar in DampingMode::On
    } else if (bp.simultaneous) {
        rayleigh2(v, w, U, g0, g1, dt, q3.w, comp1, damp);
    } else {
        rayleigh1(v, w, U[0], g0, dt, q3.w, damp);
        rayleigh1(v, w, U[1], g1, dt, comp1, damp);
    }
}

// damp_solve of tet i of the sweep order.
template <int E, bool AUX>
__device__ __forceinline__ void damp_one(uint32_t i, const uint4* __restrict__ tidx, const float4* __restrict__ tg0,
                                         const float4* __restrict__ tg1, const float4* __restrict__ tg2,
                                         const float4* __restrict__ tg3, const float4* __restrict__ taux,
                                         const float2* __restrict__ tdmp, const double4* __restrict__ X,
                                         double4* __restrict__ V, const XfBodyParams* __restrict__ bodies,
                                         float comp1_u, float a_u, float dt, uint32_t tick) {
    float comp1 = comp1_u, a = a_u;
    uint32_t body = 0;
    if constexpr (AUX) {
        float4 ax = taux[i];
        comp1 = ax.x;
        a = ax.y;
        body = __float_as_uint(ax.z);
    }
    const XfBodyParams& bp = bodies[body];
    if (!damps_post(bp, tdmp[i], tick)) return;
    uint4 id = tidx[i];
    float4 q0 = tg0[i], q1 = tg1[i], q2 = tg2[i], q3 = tg3[i];
    double4 na = X[id.x], nb = X[id.y], nc = X[id.z], nd = X[id.w];
    double4 va = V[id.x], vb = V[id.y], vc = V[id.z], vd = V[id.w];
    double x[4][3] = {{na.x, na.y, na.z}, {nb.x, nb.y, nb.z}, {nc.x, nc.y, nc.z}, {nd.x, nd.y, nd.z}};
    double v[4][3] = {{va.x, va.y, va.z}, {vb.x, vb.y, vb.z}, {vc.x, vc.y, vc.z}, {vd.x, vd.y, vd.z}};
    float w[4] = {(float)na.w, (float)nb.w, (float)nc.w, (float)nd.w};
    damp_solve<E>(bp, q0, q1, q2, q3, comp1, a, x, v, w, dt);
    V[id.x] = make_double4(v[0][0], v[0][1], v[0][2], 0.0);
    V[id.y] = make_double4(v[1][0], v[1][1], v[1][2], 0.0);
    V[id.z] = make_double4(v[2][0], v[2][1], v[2][2], 0.0);
    V[id.w] = make_double4(v[3][0], v[3][1], v[3][2], 0.0);
}

// PBD damping of one tet (Geo.cpp:806-809), factor min(1, pbd / surfaceArea).
__device__ __forceinline__ void pbd_solve(const XfBodyParams& bp, float area, const double x[4][3], double v[4][3],
                                          const float w[4]) {
    float f = (bp.rtype == 3u ? bp.pbd_amortized : bp.pbd) / area;
    f = f < 1.0f ? f : 1.0f;
    pbd_damp(x, v, w, f);
}

// pbd_solve of tet i of the sweep order.
template <bool AUX>
__device__ __forceinline__ void pbd_one(uint32_t i, const uint4* __restrict__ tidx, const float4* __restrict__ taux,
                                        const float2* __restrict__ tdmp, const double4* __restrict__ X,
                                        double4* __restrict__ V, const XfBodyParams* __restrict__ bodies,
                                        uint32_t tick) {
    uint32_t body = 0;
    if constexpr (AUX) body = __float_as_uint(taux[i].z);
    const XfBodyParams& bp = bodies[body];
    float2 dm = tdmp[i];
    if (!damps_pbd(bp, dm, tick)) return;
    uint4 id = tidx[i];
    double4 na = X[id.x], nb = X[id.y], nc = X[id.z], nd = X[id.w];
    double4 va = V[id.x], vb = V[id.y], vc = V[id.z], vd = V[id.w];
    double x[4][3] = {{na.x, na.y, na.z}, {nb.x, nb.y, nb.z}, {nc.x, nc.y, nc.z}, {nd.x, nd.y, nd.z}};
    double v[4][3] = {{va.x, va.y, va.z}, {vb.x, vb.y, vb.z}, {vc.x, vc.y, vc.z}, {vd.x, vd.y, vd.z}};
    float w[4] = {(float)na.w, (float)nb.w, (float)nc.w, (float)nd.w};
    pbd_solve(bp, dm.x, x, v, w);
    V[id.x] = make_double4(v[0][0], v[0][1], v[0][2], 0.0);
    V[id.y] = make_double4(v[1][0], v[1][1], v[1][2], 0.0);
    V[id.z] = make_double4(v[2][0], v[2][1], v[2][2], 0.0);
    V[id.w] = make_double4(v[3][0], v[3][1], v[3][2], 0.0);
}

// The projection of one tet from its loaded element data (q0..q3: Qi, QQ,
// QR, comp0; ax: comp1, a, body when AUX) on positions x, inverse masses w.
// DAMP: bodies may damp inside the projection (Rayleigh_Paper / _Limit);
// reads O of the 4 nodes (global ids id).
template <int E, bool SIM, bool AUX, bool DAMP>
__device__ __forceinline__ void project_loaded(const float4& q0, const float4& q1, const float4& q2, const float4& q3,
                                               const float4& ax, const uint4& id, double x[4][3], const float w[4],
                                               const double4* __restrict__ O, const XfBodyParams* __restrict__ bodies,
                                               float comp1_u, float a_u, float dt) {
    float comp1 = comp1_u, a = a_u;
    uint32_t body = 0;
    if constexpr (AUX) {
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
    if constexpr (DAMP) {
        double4 oa = O[id.x], ob = O[id.y], oc = O[id.z], od = O[id.w];
        double o[4][3] = {{oa.x, oa.y, oa.z}, {ob.x, ob.y, ob.z}, {oc.x, oc.y, oc.z}, {od.x, od.y, od.z}};
        solve_tet<E, SIM, true>(yeohFast, C, x, w, Qi, QQ, QR, q3.w, comp1, a, dt, o, bp.damping, bp.rtype);
    } else {
        solve_tet<E, SIM>(yeohFast, C, x, w, Qi, QQ, QR, q3.w, comp1, a, dt);
    }
}

// Element data of one tet of the schedule and its four block-local nodes
// (loc: 16 bits each, x: corners 0 | 1 << 16, y: corners 2 | 3 << 16).
struct BlockTet {
    float4 q0, q1, q2, q3, ax;
    uint2 loc;
};

template <bool AUX>
__device__ __forceinline__ BlockTet load_block_tet(uint32_t i, const uint2* __restrict__ tloc,
                                                   const float4* __restrict__ tg0, const float4* __restrict__ tg1,
                                                   const float4* __restrict__ tg2, const float4* __restrict__ tg3,
                                                   const float4* __restrict__ taux) {
    BlockTet t;
    t.q0 = tg0[i];
    t.q1 = tg1[i];
    t.q2 = tg2[i];
    t.q3 = tg3[i];
    t.ax = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if constexpr (AUX) t.ax = taux[i];
    t.loc = tloc[i];
    return t;
}

// Material and body of a tet: per tet (AUX), else uniform and body 0.
struct TetMaterial {
    float comp1, a;
    uint32_t body;
};
template <bool AUX>
__device__ __forceinline__ TetMaterial tet_material(const float4& ax, float comp1_u, float a_u) {
    if constexpr (AUX) return {ax.x, ax.y, __float_as_uint(ax.z)};
    return {comp1_u, a_u, 0u};
}

// A slot's nodes in LDS, node k at byte k * NS: (x, y) in its first 16
// bytes, (z, w) in the next. NS = 32 packs them; NS = 48 spreads their
// 16-byte halves over every bank group of a 128-byte LDS row (with 32 only
// every other group is reached), so the four-node gathers of a phase meet
// fewer bank conflicts, for half as much LDS again.
template <uint32_t NS>
struct NodeLds {
    static_assert(NS == 32u || NS == 48u, "32 or 48 bytes per node");
    double2* base;  // 16-byte units
    __device__ __forceinline__ double2* at(uint32_t k) const { return base + k * (NS / 16u); }
    __device__ __forceinline__ double4 get(uint32_t k) const {
        const double2* p = at(k);
        const double2 a = p[0], b = p[1];
        return make_double4(a.x, a.y, b.x, b.y);
    }
    __device__ __forceinline__ void put(uint32_t k, double4 v) const {
        double2* p = at(k);
        p[0] = make_double2(v.x, v.y);
        p[1] = make_double2(v.z, v.w);
    }
    // component c of node k (x, y, z, w)
    __device__ __forceinline__ double* comp(uint32_t k, uint32_t c) const {
        return reinterpret_cast<double*>(at(k)) + c;
    }
    // position only (w, the inverse mass, is not changed by a projection)
    __device__ __forceinline__ void put_xyz(uint32_t k, double x, double y, double z) const {
        double2* p = at(k);
        p[0] = make_double2(x, y);
        p[1].x = z;
    }
};

// A slot's nodes into LDS (stage_nodes) and back (write_nodes), kStage list
// entries per lane at a time: the batch's id loads are issued together,
// then its node loads (at clamped in-range positions, so that no branch
// separates them), so a batch costs two memory round trips whatever its
// size, where one entry per iteration waits for each id before its node.
constexpr uint32_t kStage = 4;

template <uint32_t NS>
__device__ __forceinline__ void stage_nodes(uint32_t tid, uint32_t bs, uint32_t n, const uint32_t* __restrict__ bn,
                                            const double4* __restrict__ X, NodeLds<NS> xs) {
    for (uint32_t k0 = tid; k0 < n; k0 += kStage * bs) {
        uint32_t g[kStage];
#pragma unroll
        for (uint32_t u = 0; u < kStage; u++) g[u] = bn[min(k0 + u * bs, n - 1u)];
        double4 v[kStage];
#pragma unroll
        for (uint32_t u = 0; u < kStage; u++) v[u] = X[g[u] != xf::kNoNode ? g[u] : 0u];
#pragma unroll
        for (uint32_t u = 0; u < kStage; u++) {
            const uint32_t k = k0 + u * bs;
            if (k < n && g[u] != xf::kNoNode) xs.put(k, v[u]);
        }
    }
}

// One tet of a phase in LDS, one lane: nodes from LDS, projected, written back.
// yf, C: the energy term and coefficients of its body.
template <int E, bool SIM, uint32_t NS>
__device__ __forceinline__ void lds_tet(const BlockTet& t, NodeLds<NS> xs, bool yf, const float C[3], float comp1,
                                        float a, float dt) {
    const uint32_t id[4] = {t.loc.x & 0xFFFFu, t.loc.x >> 16, t.loc.y & 0xFFFFu, t.loc.y >> 16};
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
    const float Qi[3][3] = {{t.q0.x, t.q0.y, t.q0.z}, {t.q0.w, t.q1.x, t.q1.y}, {t.q1.z, t.q1.w, t.q2.x}};
    const float QQ[3] = {t.q2.y, t.q2.z, t.q2.w};
    const float QR[3] = {t.q3.x, t.q3.y, t.q3.z};
    solve_tet<E, SIM>(yf, C, x, w, Qi, QQ, QR, t.q3.w, comp1, a, dt);
#pragma unroll
    for (int k = 0; k < 4; k++) xs.put_xyz(id[k], x[k][0], x[k][1], x[k][2]);
}

// The same with damping inside the projection (reads O of the tet's nodes,
// global ids gid, and the body's damping).
template <int E, bool SIM, bool AUX, uint32_t NS>
__device__ __forceinline__ void lds_tet_damped(const BlockTet& t, const uint4& gid, NodeLds<NS> xs,
                                               const double4* __restrict__ O, const XfBodyParams* __restrict__ bodies,
                                               float comp1_u, float a_u, float dt) {
    uint32_t ia = t.loc.x & 0xFFFFu, ib = t.loc.x >> 16, ic = t.loc.y & 0xFFFFu, id = t.loc.y >> 16;
    double4 na = xs.get(ia), nb = xs.get(ib), nc = xs.get(ic), nd = xs.get(id);
    double x[4][3] = {{na.x, na.y, na.z}, {nb.x, nb.y, nb.z}, {nc.x, nc.y, nc.z}, {nd.x, nd.y, nd.z}};
    float w[4] = {(float)na.w, (float)nb.w, (float)nc.w, (float)nd.w};
    project_loaded<E, SIM, AUX, true>(t.q0, t.q1, t.q2, t.q3, t.ax, gid, x, w, O, bodies, comp1_u, a_u, dt);
    xs.put_xyz(ia, x[0][0], x[0][1], x[0][2]);
    xs.put_xyz(ib, x[1][0], x[1][1], x[1][2]);
    xs.put_xyz(ic, x[2][0], x[2][1], x[2][2]);
    xs.put_xyz(id, x[3][0], x[3][1], x[3][2]);
}

// v of another lane of this lane's quad (lanes 4k .. 4k + 3), by DPP
// quad_perm: lane i reads lane Pi. Bounds control on with full masks lets the
// compiler fold the move into the instruction that uses it.
template <int P0, int P1, int P2, int P3>
__device__ __forceinline__ float quad_perm(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), P0 | (P1 << 2) | (P2 << 4) | (P3 << 6), 0xF,
                                                      0xF, true));
}
template <int P0, int P1, int P2, int P3>
__device__ __forceinline__ double quad_perm(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xFFFFFFFFll), P0 | (P1 << 2) | (P2 << 4) | (P3 << 6), 0xF,
                                               0xF, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), P0 | (P1 << 2) | (P2 << 4) | (P3 << 6), 0xF, 0xF, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
template <int L, class R>
__device__ __forceinline__ R quad_lane(R v) {
    return quad_perm<L, L, L, L>(v);
}
// a . b of two vectors held one component per lane, valid in lanes 0 and 1:
// (x + y) + z, where x + y and y + x round alike.
template <class R>
__device__ __forceinline__ R quad_dot(R a, R b) {
    const R m = a * b;
    return (m + quad_perm<1, 0, 2, 3>(m)) + quad_lane<2>(m);
}

// Element constants of a tet in the element precision R.
template <class R>
struct QuadTet {
    R Qi[3][3], QQ[3], QR[3], comp0;
};
template <class R>
__device__ __forceinline__ QuadTet<R> quad_tet(const BlockTet& t) {
    return {{{(R)t.q0.x, (R)t.q0.y, (R)t.q0.z}, {(R)t.q0.w, (R)t.q1.x, (R)t.q1.y}, {(R)t.q1.z, (R)t.q1.w, (R)t.q2.x}},
            {(R)t.q2.y, (R)t.q2.z, (R)t.q2.w},
            {(R)t.q3.x, (R)t.q3.y, (R)t.q3.z},
            (R)t.q3.w};
}

// The projection of one tet on the four lanes of a quad, split by component:
// lanes 0, 1, 2 hold x, y, z of every vector of the tet (positions,
// gradients, rows of F); x: this lane's component of the four positions (any
// value in lane 3), w: the inverse masses, in every lane; xn: the component
// after the projection. SolveElementMixed with the simultaneous
// solve (MixedSel / YeohSkinFast), damping off, in
// exactly the operations and order of solve_tet and solve_mixed_sim:
//  - P, the gradients, F, the updates: each lane its own component;
//  - column a of the adjugate is the cross product of rows a + 1 and a + 2 of
//    F, which the lane reads from its neighbours (cofactors that solve_tet
//    negates come out as the reversed difference, the same value);
//  - dot products by quad_dot, so scalars are valid in lanes 0 and 1;
//  - the 2x2 system: lane 0 holds the I1 row, lane 1 the volume row, so one
//    reciprocal serves both and the Cramer solve is one expression.
// Results equal those of one lane bit for bit. The chain is about half as long
// as one lane's (293 against 520 VALU instructions for MixedSel), which
// counts where a phase has fewer waves than the chip has SIMDs.
// yf: the body's energy is YeohSkinFast, with coefficients C.
template <class R>
__device__ __forceinline__ void quad_solve(const QuadTet<R>& t, uint32_t q, const double x[4], const float w[4],
                                           bool yf, const R C[3], R comp1, R a, R dt, double xn[4]) {
    R P[3];
#pragma unroll
    for (int i = 0; i < 3; i++) P[i] = (R)(x[i] - x[3]);

    // prefactored I1 (neo_prefactored)
    R u = R(0.0), g0[4], g1[4];
#pragma unroll
    for (int i = 0; i < 3; i++) {
        u = u + t.QQ[i] * quad_dot(P[i], P[i]);
        g0[i] = (R(2.0) * t.QQ[i]) * P[i];
    }
    {
        int k = 0;
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int j = i + 1; j < 3; j++) {
                u = u + t.QR[k] * quad_dot(P[i], P[j]);
                g0[i] = g0[i] + t.QR[k] * P[j];
                g0[j] = g0[j] + t.QR[k] * P[i];
                ++k;
            }
    }
    g0[3] = ((R(0.0) - g0[0]) - g0[1]) - g0[2];
    R U0 = u;
    if (yf) {
        const R IM = U0 - R(3.0);
        U0 = fmax(R(0.0001), C[0] * IM + C[1] * IM * IM + C[2] * IM * IM * IM);
        const R gScale = quad_lane<0>(C[0] + R(2.0) * C[1] * IM + R(3.0) * C[2] * IM * IM);
#pragma unroll
        for (int n = 0; n < 4; n++) g0[n] = g0[n] * gScale;
    }

    // (J - a)^2 volume term (volume_term)
    R F[3], A[3], B[3], adj[3];
#pragma unroll
    for (int r = 0; r < 3; r++) F[r] = t.Qi[0][r] * P[0] + t.Qi[1][r] * P[1] + t.Qi[2][r] * P[2];
#pragma unroll
    for (int r = 0; r < 3; r++) {
        A[r] = quad_perm<1, 2, 0, 3>(F[r]);
        B[r] = quad_perm<2, 0, 1, 3>(F[r]);
    }
    adj[0] = A[1] * B[2] - A[2] * B[1];
    adj[1] = A[2] * B[0] - A[0] * B[2];
    adj[2] = A[0] * B[1] - A[1] * B[0];
    const R J = quad_lane<0>(F[0] * adj[0] + F[1] * adj[1] + F[2] * adj[2]);
    const R U1 = (J - a) * (J - a);
    const R sJ = R(2.0) * (J - a);
#pragma unroll
    for (int c = 0; c < 3; c++) adj[c] = adj[c] * sJ;
#pragma unroll
    for (int j = 0; j < 3; j++) g1[j] = R(0.0) + (adj[0] * t.Qi[j][0] + adj[1] * t.Qi[j][1] + adj[2] * t.Qi[j][2]);
    g1[3] = ((R(0.0) - g1[0]) - g1[1]) - g1[2];

    // EnergyXpbdConstrainSimultaneous<2>, Cramer branch (constrain2)
    R A0 = R(1.0e-22), A1 = R(1.0e-22), A2 = R(1.0e-22);
#pragma unroll
    for (int n = 0; n < 4; n++) {
        A0 = A0 + w[n] * quad_dot(g0[n], g0[n]);
        A1 = A1 + w[n] * quad_dot(g1[n], g0[n]);
        A2 = A2 + w[n] * quad_dot(g1[n], g1[n]);
    }
    const bool row1 = (q & 1u) != 0u;
    const R U = row1 ? U1 : U0;
    const R alpha = row1 ? comp1 / (dt * dt) : t.comp0 / (dt * dt);
    const R Ad = (row1 ? A2 : A0) + R(2.0) * U * alpha;
    const R invA = R(1.0) / Ad;
    const R be = (R(-2.0) * U) * invA;  // b0 invA00 | b1 invA11
    const R pq = A1 * invA;             // A1 invA00 | A1 invA11
    const R invDet = R(1.0) / fmax(R(0.00000001), R(1.0) - pq * quad_perm<1, 0, 2, 3>(pq));
    const R l = invDet * (be - pq * quad_perm<1, 0, 2, 3>(be));
    const R l0 = quad_lane<0>(l), l1 = quad_lane<1>(l);
#pragma unroll
    for (int n = 0; n < 4; n++) {
        R acc = R(0.0) + l0 * g0[n];
        acc = acc + l1 * g1[n];
        xn[n] = x[n] + (double)(w[n] * acc);
    }
}

// The components of a tet's four nodes in LDS that lane q of its quad holds.
template <uint32_t NS>
struct QuadNodes {
    double* n[4];
    __device__ __forceinline__ QuadNodes(NodeLds<NS> s, const uint2& loc, uint32_t q)
        : n{s.comp(loc.x & 0xFFFFu, q), s.comp(loc.x >> 16, q), s.comp(loc.y & 0xFFFFu, q), s.comp(loc.y >> 16, q)} {}
    // the components, and the inverse masses (the fourth component) in every lane
    __device__ __forceinline__ void get(double x[4], float w[4]) const {
#pragma unroll
        for (int k = 0; k < 4; k++) x[k] = *n[k];
#pragma unroll
        for (int k = 0; k < 4; k++) w[k] = quad_lane<3>((float)x[k]);
    }
    // positions only
    __device__ __forceinline__ void put(uint32_t q, const double x[4]) const {
        if (q != 3u)
#pragma unroll
            for (int k = 0; k < 4; k++) *n[k] = x[k];
    }
};

// One tet of a block phase on the four lanes of a quad (quad_solve).
template <uint32_t NS>
__device__ __forceinline__ void block_tet_quad(const BlockTet& t, uint32_t q, NodeLds<NS> xs, bool yf,
                                               const float C[3], float comp1, float a, float dt) {
    const QuadNodes<NS> nodes(xs, t.loc, q);
    double x[4], xn[4];
    float w[4];
    nodes.get(x, w);
    quad_solve<float>(quad_tet<float>(t), q, x, w, yf, C, comp1, a, dt, xn);
    nodes.put(q, xn);
}

// Collision projection of one unpinned node (no reference counterpart).
// Ground plane y >= ground_y and a kinematic sphere; Coulomb friction on the
// tangential displacement of the substep (static if |d_t| <= mu * depth).
// Corrections are computed in FP32 and added to the FP64 position.
__device__ __forceinline__ void collide_node(const XfBodyParams& p, float t_end, const double o[3], double x[3]) {
    float mu = p.friction;
    if (p.collide & 1u) {
        float gy = p.ground_y;
        float xy = (float)x[1];
        if (xy < gy) {
            float depth = gy - xy;
            x[1] = (double)gy;
            float dx = (float)(x[0] - o[0]);
            float dz = (float)(x[2] - o[2]);
            float t2 = dx * dx + dz * dz;
            float lim = mu * depth;
            if (t2 <= lim * lim) {
                x[0] = o[0];
                x[2] = o[2];
            } else {
                float s = lim / sqrtf(t2);
                x[0] = x[0] - (double)(dx * s);
                x[2] = x[2] - (double)(dz * s);
            }
        }
    }
    if (p.collide & 2u) {
        float c[3], d[3];
#pragma unroll
        for (int r = 0; r < 3; r++) c[r] = p.sc0[r] + p.sv[r] * t_end;
#pragma unroll
        for (int r = 0; r < 3; r++) d[r] = (float)x[r] - c[r];
        float d2 = dot3(d, d);
        float rad = p.sr;
        if (d2 < rad * rad && d2 > 0.0f) {
            float dist = sqrtf(d2);
            float inv = 1.0f / dist;
            float n[3] = {d[0] * inv, d[1] * inv, d[2] * inv};
            float depth = rad - dist;
#pragma unroll
            for (int r = 0; r < 3; r++) x[r] = x[r] + (double)(n[r] * depth);
            float rel[3], rt[3];
#pragma unroll
            for (int r = 0; r < 3; r++) rel[r] = (float)(x[r] - o[r]) - p.sv[r] * p.dt;
            float rn = dot3(rel, n);
#pragma unroll
            for (int r = 0; r < 3; r++) rt[r] = rel[r] - n[r] * rn;
            float t2 = dot3(rt, rt);
            float lim = mu * depth;
            float s = 1.0f;
            if (t2 > lim * lim) s = lim / sqrtf(t2);
#pragma unroll
            for (int r = 0; r < 3; r++) x[r] = x[r] - (double)(rt[r] * s);
        }
    }
}

// Prediction (Geo.cpp:307-312), FP64 state with FP32 settings products.
__device__ __forceinline__ void predict(const XfBodyParams& p, double v[3], const double x[3], double4* Xo,
                                        double4* Oo, double w, double oflags) {
    v[0] = v[0] + (double)p.gdx;
    v[1] = v[1] + (double)p.gdy;
    v[2] = v[2] + (double)0.0f;
    double dragf = (double)p.dragf;
#pragma unroll
    for (int r = 0; r < 3; r++) v[r] = v[r] * dragf;
    double dt = (double)p.dt;
    *Oo = make_double4(x[0], x[1], x[2], oflags);
    *Xo = make_double4(x[0] + v[0] * dt, x[1] + v[1] * dt, x[2] + v[2] * dt, w);
}

// The lock of Geo3d::Substep (Geo.cpp:318-322) and the contact pass for one
// node: a pinned node of a body whose pins are locked this step returns to
// O and its inverse mass becomes 0 (from then on; it may be finite until its
// first locked substep); other nodes with mass take contact. Returns the
// node's inverse mass after the lock.
__device__ __forceinline__ double lock_contact(const XfBodyParams& p, uint32_t flags, float t_end, double w,
                                               const double o[3], double x[3]) {
    if ((flags & 1u) && !p.unlock) {
        x[0] = o[0];
        x[1] = o[1];
        x[2] = o[2];
        return 0.0;
    }
    if (p.collide && w != 0.0) collide_node(p, t_end, o, x);
    return w;
}

__device__ __forceinline__ void finish_predict(double4 xi, double4 oi, uint32_t i, double4* __restrict__ X,
                                               double4* __restrict__ O, const XfBodyParams& p, float t_end) {
    uint32_t flags = (uint32_t)oi.w;
    double x[3] = {xi.x, xi.y, xi.z};
    double o[3] = {oi.x, oi.y, oi.z};
    const double w = lock_contact(p, flags, t_end, xi.w, o, x);
    double v[3];
    double invdt = (double)p.invdt;
#pragma unroll
    for (int r = 0; r < 3; r++) v[r] = (x[r] - o[r]) * invdt;
    predict(p, v, x, &X[i], &O[i], w, oi.w);
}

}  // namespace

#endif  // XF_TET_H
