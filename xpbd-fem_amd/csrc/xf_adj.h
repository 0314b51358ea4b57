// xf_adj.h -- device functions of the adjoint of one tet and one node, and of
// the FP64 element model's node steps, shared by the launches per colour
// (xf_adjoint.hip) and by whole checkpoint windows of small bodies
// (xf_body_adjoint.hip). Precision and scope: see xf_adjoint.hip.
#pragma once

#include <hip/hip_runtime.h>

#include "xf_device.h"
#include "xf_element.h"
#include "xf_tet.h"

namespace {

// Adjoint of one simultaneous projection (forward: xf::solve_mixed_sim, as
// xf_kernels.hip solve_tet for E = 4 / 7) in element precision R. x:
// positions before it; xbar: in, adjoint of the positions after it; out,
// adjoint of the positions before it. Returns d(loss)/d(log comp0) of this
// projection.
template <class R>
__device__ __forceinline__ R adjoint_tet(bool yeoh, const R C[3], const double x[4][3], const float w[4],
                                         const R Qi[3][3], const R QQ[3], const R QR[3], R comp0, R comp1, R a, R dt,
                                         double xbar[4][3]) {
    R P[3][3];
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int r = 0; r < 3; r++) P[i][r] = (R)(x[i][r] - x[3][r]);
    R g0n[4][3], U0n;
    neo_prefactored(QQ, QR, P, U0n, g0n);
    R U0 = U0n, IM = R(0.0), cpoly = R(0.0), s = R(1.0), g0[4][3];
#pragma unroll
    for (int n = 0; n < 4; n++)
#pragma unroll
        for (int r = 0; r < 3; r++) g0[n][r] = g0n[n][r];
    if (yeoh) {
        IM = U0n - R(3.0);
        cpoly = C[0] * IM + C[1] * IM * IM + C[2] * IM * IM * IM;
        U0 = fmax(R(0.0001), cpoly);
        s = C[0] + R(2.0) * C[1] * IM + R(3.0) * C[2] * IM * IM;
#pragma unroll
        for (int n = 0; n < 4; n++)
#pragma unroll
            for (int r = 0; r < 3; r++) g0[n][r] = g0n[n][r] * s;
    }
    R F[3][3], adj[3][3], G[3][3], g1[4][3];
    defgrad(Qi, P, F);
    R J = adjdet(F, adj);
    R d = J - a;
    R U1 = R(0.0) + R(1.0) * (d * d);
    R sv = R(2.0) * d;
#pragma unroll
    for (int c = 0; c < 3; c++)
#pragma unroll
        for (int r = 0; r < 3; r++) G[c][r] = adj[c][r] * sv;
#pragma unroll
    for (int n = 0; n < 4; n++)
#pragma unroll
        for (int r = 0; r < 3; r++) g1[n][r] = R(0.0);
    apply_grad(G, Qi, g1);
    root_grad(g1);
    R alpha0 = comp0 / (dt * dt), alpha1 = comp1 / (dt * dt);
    R A0 = R(1.0e-22), A1 = R(1.0e-22), A2 = R(1.0e-22);
#pragma unroll
    for (int n = 0; n < 4; n++) A0 = A0 + w[n] * dot3(g0[n], g0[n]);
    A0 = A0 + R(2.0) * U0 * alpha0;
    R b0 = -R(2.0) * U0;
#pragma unroll
    for (int n = 0; n < 4; n++) A1 = A1 + w[n] * dot3(g1[n], g0[n]);
#pragma unroll
    for (int n = 0; n < 4; n++) A2 = A2 + w[n] * dot3(g1[n], g1[n]);
    A2 = A2 + R(2.0) * U1 * alpha1;
    R b1 = -R(2.0) * U1;
    R u = R(1.0) / A0, v = R(1.0) / A2;
    R p = A1 * u, q = A1 * v, be0 = b0 * u, be1 = b1 * v;
    R Dr = R(1.0) - p * q;
    R invDet = R(1.0) / fmax(R(0.00000001), Dr);
    R r0 = be0 - p * be1, r1 = be1 - be0 * q;
    R l0 = invDet * r0, l1 = invDet * r1;

    R g0b[4][3], g1b[4][3];
    R l0b = R(0.0), l1b = R(0.0);
#pragma unroll
    for (int n = 0; n < 4; n++)
#pragma unroll
        for (int r = 0; r < 3; r++) {
            R accb = w[n] * (R)xbar[n][r];
            l0b = l0b + g0[n][r] * accb;
            l1b = l1b + g1[n][r] * accb;
            g0b[n][r] = l0 * accb;
            g1b[n][r] = l1 * accb;
        }
    R invDetb = l0b * r0 + l1b * r1;
    R r0b = l0b * invDet, r1b = l1b * invDet;
    R be0b = r0b - r1b * q, be1b = r1b - r0b * p;
    R pb = R(0.0) - r0b * be1, qb = R(0.0) - r1b * be0;
    R Drb = Dr > R(0.00000001) ? (R(0.0) - invDetb * invDet * invDet) : R(0.0);
    pb = pb - Drb * q;
    qb = qb - Drb * p;
    R A1b = pb * u + qb * v;
    R ub = pb * A1 + be0b * b0, vb = qb * A1 + be1b * b1;
    R b0b = be0b * u, b1b = be1b * v;
    R A0b = R(0.0) - ub * u * u, A2b = R(0.0) - vb * v * v;
    R U0b = -R(2.0) * b0b + R(2.0) * alpha0 * A0b;
    R U1b = -R(2.0) * b1b + R(2.0) * alpha1 * A2b;
    R alpha0b = R(2.0) * U0 * A0b;
#pragma unroll
    for (int n = 0; n < 4; n++)
#pragma unroll
        for (int r = 0; r < 3; r++) {
            g0b[n][r] = g0b[n][r] + R(2.0) * A0b * w[n] * g0[n][r] + A1b * w[n] * g1[n][r];
            g1b[n][r] = g1b[n][r] + A1b * w[n] * g0[n][r] + R(2.0) * A2b * w[n] * g1[n][r];
        }
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int r = 0; r < 3; r++) g1b[i][r] = g1b[i][r] - g1b[3][r];
    R adjb[3][3], Fb[3][3], Pb[3][3];
    R svb = R(0.0);
#pragma unroll
    for (int m = 0; m < 3; m++)
#pragma unroll
        for (int r = 0; r < 3; r++) {
            R Gb = g1b[0][r] * Qi[0][m] + g1b[1][r] * Qi[1][m] + g1b[2][r] * Qi[2][m];
            adjb[m][r] = Gb * sv;
            svb = svb + Gb * adj[m][r];
        }
    R db = R(2.0) * svb + R(2.0) * d * U1b;
#pragma unroll
    for (int c = 0; c < 3; c++)
#pragma unroll
        for (int r = 0; r < 3; r++) Fb[c][r] = db * adj[r][c];
    {
        R m00 = F[0][0], m01 = F[0][1], m02 = F[0][2];
        R m10 = F[1][0], m11 = F[1][1], m12 = F[1][2];
        R m20 = F[2][0], m21 = F[2][1], m22 = F[2][2];
        R t;
        t = adjb[0][0]; Fb[1][1] += t * m22; Fb[2][2] += t * m11; Fb[1][2] -= t * m21; Fb[2][1] -= t * m12;
        t = adjb[0][1]; Fb[0][1] -= t * m22; Fb[2][2] -= t * m01; Fb[0][2] += t * m21; Fb[2][1] += t * m02;
        t = adjb[0][2]; Fb[0][1] += t * m12; Fb[1][2] += t * m01; Fb[0][2] -= t * m11; Fb[1][1] -= t * m02;
        t = adjb[1][0]; Fb[1][0] -= t * m22; Fb[2][2] -= t * m10; Fb[1][2] += t * m20; Fb[2][0] += t * m12;
        t = adjb[1][1]; Fb[0][0] += t * m22; Fb[2][2] += t * m00; Fb[0][2] -= t * m20; Fb[2][0] -= t * m02;
        t = adjb[1][2]; Fb[0][0] -= t * m12; Fb[1][2] -= t * m00; Fb[0][2] += t * m10; Fb[1][0] += t * m02;
        t = adjb[2][0]; Fb[1][0] += t * m21; Fb[2][1] += t * m10; Fb[1][1] -= t * m20; Fb[2][0] -= t * m11;
        t = adjb[2][1]; Fb[0][0] -= t * m21; Fb[2][1] -= t * m00; Fb[0][1] += t * m20; Fb[2][0] += t * m01;
        t = adjb[2][2]; Fb[0][0] += t * m11; Fb[1][1] += t * m00; Fb[0][1] -= t * m10; Fb[1][0] -= t * m01;
    }
#pragma unroll
    for (int m = 0; m < 3; m++)
#pragma unroll
        for (int j = 0; j < 3; j++) Pb[m][j] = Qi[m][0] * Fb[j][0] + Qi[m][1] * Fb[j][1] + Qi[m][2] * Fb[j][2];
    R g0nb[4][3], U0nb;
    if (yeoh) {
        R polyb = cpoly > R(0.0001) ? U0b : R(0.0);
        R sb = R(0.0);
#pragma unroll
        for (int n = 0; n < 4; n++)
#pragma unroll
            for (int r = 0; r < 3; r++) {
                sb = sb + g0b[n][r] * g0n[n][r];
                g0nb[n][r] = g0b[n][r] * s;
            }
        U0nb = polyb * s + sb * (R(2.0) * C[1] + R(6.0) * C[2] * IM);
    } else {
#pragma unroll
        for (int n = 0; n < 4; n++)
#pragma unroll
            for (int r = 0; r < 3; r++) g0nb[n][r] = g0b[n][r];
        U0nb = U0b;
    }
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int r = 0; r < 3; r++) g0nb[i][r] = g0nb[i][r] - g0nb[3][r];
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int r = 0; r < 3; r++) Pb[i][r] = Pb[i][r] + U0nb * g0n[i][r] + R(2.0) * QQ[i] * g0nb[i][r];
    {
        int k = 0;
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int j = i + 1; j < 3; j++) {
#pragma unroll
                for (int r = 0; r < 3; r++) {
                    Pb[j][r] = Pb[j][r] + QR[k] * g0nb[i][r];
                    Pb[i][r] = Pb[i][r] + QR[k] * g0nb[j][r];
                }
                ++k;
            }
    }
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int r = 0; r < 3; r++) {
            xbar[i][r] = xbar[i][r] + (double)Pb[i][r];
            xbar[3][r] = xbar[3][r] - (double)Pb[i][r];
        }
    return alpha0b * alpha0;
}

// adjoint_tet on the four lanes of a quad, split by component as quad_solve
// (the same operations in the same order; results equal it bit for bit). x:
// this lane's component of the four positions before the projection, xbar:
// of their adjoints, in and out. Returns d(loss)/d(log comp0), valid in
// lane 0. Sums over nodes and components run in adjoint_tet's order, one
// component after another from the lanes that hold them (quad_sum3). The
// adjoint of the adjugate adds its four terms to each entry of F's adjoint in
// an order that differs in lane 1 by a swap within each pair, and there with
// the opposite signs: the lanes read their two neighbours in that order
// (first / second below) and lane 1 negates what it reads.
template <class R>
__device__ __forceinline__ R quad_sum3(R acc, R m) {  // ((acc + m.x) + m.y) + m.z, in every lane
    acc = acc + quad_lane<0>(m);
    acc = acc + quad_lane<1>(m);
    return acc + quad_lane<2>(m);
}
template <class R>
__device__ __forceinline__ R adjoint_quad(const QuadTet<R>& t, uint32_t q, bool yeoh, const R C[3], const double x[4],
                                          const float w[4], R comp1, R a, R dt, double xbar[4]) {
    R P[3];
#pragma unroll
    for (int i = 0; i < 3; i++) P[i] = (R)(x[i] - x[3]);
    R U0n = R(0.0), g0n[4];
#pragma unroll
    for (int i = 0; i < 3; i++) {
        U0n = U0n + t.QQ[i] * quad_dot(P[i], P[i]);
        g0n[i] = (R(2.0) * t.QQ[i]) * P[i];
    }
    {
        int k = 0;
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int j = i + 1; j < 3; j++) {
                U0n = U0n + t.QR[k] * quad_dot(P[i], P[j]);
                g0n[i] = g0n[i] + t.QR[k] * P[j];
                g0n[j] = g0n[j] + t.QR[k] * P[i];
                ++k;
            }
    }
    g0n[3] = ((R(0.0) - g0n[0]) - g0n[1]) - g0n[2];
    R U0 = U0n, IM = R(0.0), cpoly = R(0.0), s = R(1.0), g0[4];
#pragma unroll
    for (int n = 0; n < 4; n++) g0[n] = g0n[n];
    if (yeoh) {
        IM = U0n - R(3.0);
        cpoly = C[0] * IM + C[1] * IM * IM + C[2] * IM * IM * IM;
        U0 = fmax(R(0.0001), cpoly);
        s = quad_lane<0>(C[0] + R(2.0) * C[1] * IM + R(3.0) * C[2] * IM * IM);
#pragma unroll
        for (int n = 0; n < 4; n++) g0[n] = g0n[n] * s;
    }
    R F[3], adj[3], g1[4];
#pragma unroll
    for (int r = 0; r < 3; r++) F[r] = t.Qi[0][r] * P[0] + t.Qi[1][r] * P[1] + t.Qi[2][r] * P[2];
    {
        R A[3], B[3];
#pragma unroll
        for (int r = 0; r < 3; r++) {
            A[r] = quad_perm<1, 2, 0, 3>(F[r]);
            B[r] = quad_perm<2, 0, 1, 3>(F[r]);
        }
        adj[0] = A[1] * B[2] - A[2] * B[1];
        adj[1] = A[2] * B[0] - A[0] * B[2];
        adj[2] = A[0] * B[1] - A[1] * B[0];
    }
    const R J = quad_lane<0>(F[0] * adj[0] + F[1] * adj[1] + F[2] * adj[2]);
    const R d = J - a;
    const R U1 = R(0.0) + R(1.0) * (d * d);
    const R sv = R(2.0) * d;
    {
        R G[3];
#pragma unroll
        for (int c = 0; c < 3; c++) G[c] = adj[c] * sv;
#pragma unroll
        for (int j = 0; j < 3; j++) g1[j] = R(0.0) + (G[0] * t.Qi[j][0] + G[1] * t.Qi[j][1] + G[2] * t.Qi[j][2]);
    }
    g1[3] = ((R(0.0) - g1[0]) - g1[1]) - g1[2];

    // the 2x2 system: lane 0 the I1 row, lane 1 the volume row
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
    const R b = -R(2.0) * U;
    const R inv = R(1.0) / Ad;                       // u | v
    const R pq = A1 * inv, be = b * inv;             // p | q, be0 | be1
    const R pq_o = quad_perm<1, 0, 2, 3>(pq), be_o = quad_perm<1, 0, 2, 3>(be);
    const R Dr = R(1.0) - pq * pq_o;
    const R invDet = R(1.0) / fmax(R(0.00000001), Dr);
    const R rr = be - pq * be_o;                     // r0 | r1
    const R l = invDet * rr;
    const R l0 = quad_lane<0>(l), l1 = quad_lane<1>(l);

    R g0b[4], g1b[4], l0b = R(0.0), l1b = R(0.0);
#pragma unroll
    for (int n = 0; n < 4; n++) {
        const R accb = w[n] * (R)xbar[n];
        l0b = quad_sum3(l0b, g0[n] * accb);
        l1b = quad_sum3(l1b, g1[n] * accb);
        g0b[n] = l0 * accb;
        g1b[n] = l1 * accb;
    }
    const R lb = row1 ? l1b : l0b;
    const R mb = lb * rr;
    const R invDetb = mb + quad_perm<1, 0, 2, 3>(mb);
    const R rb = lb * invDet;                                    // r0b | r1b
    const R beb = rb - quad_perm<1, 0, 2, 3>(rb) * pq_o;         // be0b | be1b
    R pqb = R(0.0) - rb * be_o;                                  // pb | qb
    const R Drb = Dr > R(0.00000001) ? (R(0.0) - invDetb * invDet * invDet) : R(0.0);
    pqb = pqb - Drb * pq_o;
    const R ma = pqb * inv;
    const R A1b = quad_lane<0>(ma + quad_perm<1, 0, 2, 3>(ma));
    const R ib = pqb * A1 + beb * b;                             // ub | vb
    const R bb = beb * inv;                                      // b0b | b1b
    const R Ab = R(0.0) - ib * inv * inv;                        // A0b | A2b
    const R Ub = -R(2.0) * bb + R(2.0) * alpha * Ab;             // U0b | U1b
    const R alpha0b = R(2.0) * U * Ab;
    const R A0b = quad_lane<0>(Ab), A2b = quad_lane<1>(Ab);
#pragma unroll
    for (int n = 0; n < 4; n++) {
        g0b[n] = g0b[n] + R(2.0) * A0b * w[n] * g0[n] + A1b * w[n] * g1[n];
        g1b[n] = g1b[n] + A1b * w[n] * g0[n] + R(2.0) * A2b * w[n] * g1[n];
    }
#pragma unroll
    for (int i = 0; i < 3; i++) g1b[i] = g1b[i] - g1b[3];
    R adjb[3], Fb[3], Pb[3], svb = R(0.0);
#pragma unroll
    for (int m = 0; m < 3; m++) {
        const R Gb = g1b[0] * t.Qi[0][m] + g1b[1] * t.Qi[1][m] + g1b[2] * t.Qi[2][m];
        adjb[m] = Gb * sv;
        svb = quad_sum3(svb, Gb * adj[m]);
    }
    const R db = R(2.0) * svb + R(2.0) * d * quad_lane<1>(Ub);
#pragma unroll
    for (int r = 0; r < 3; r++) Fb[r] = db * adj[r];
    {
        const R sign = q == 1u ? R(-1.0) : R(1.0);
        R t1[3], t2[3], f1[3], f2[3];  // first and second neighbour's adjb column and F row
#pragma unroll
        for (int r = 0; r < 3; r++) {
            t1[r] = sign * quad_perm<1, 0, 0, 3>(adjb[r]);
            t2[r] = sign * quad_perm<2, 2, 1, 3>(adjb[r]);
            f1[r] = quad_perm<2, 2, 1, 3>(F[r]);
            f2[r] = quad_perm<1, 0, 0, 3>(F[r]);
        }
        Fb[0] += t1[1] * f1[2]; Fb[0] -= t2[1] * f2[2]; Fb[0] -= t1[2] * f1[1]; Fb[0] += t2[2] * f2[1];
        Fb[1] -= t1[0] * f1[2]; Fb[1] += t2[0] * f2[2]; Fb[1] += t1[2] * f1[0]; Fb[1] -= t2[2] * f2[0];
        Fb[2] += t1[0] * f1[1]; Fb[2] -= t2[0] * f2[1]; Fb[2] -= t1[1] * f1[0]; Fb[2] += t2[1] * f2[0];
    }
#pragma unroll
    for (int m = 0; m < 3; m++) Pb[m] = t.Qi[m][0] * Fb[0] + t.Qi[m][1] * Fb[1] + t.Qi[m][2] * Fb[2];
    R g0nb[4], U0nb;
    if (yeoh) {
        const R polyb = cpoly > R(0.0001) ? Ub : R(0.0);
        R sb = R(0.0);
#pragma unroll
        for (int n = 0; n < 4; n++) {
            sb = quad_sum3(sb, g0b[n] * g0n[n]);
            g0nb[n] = g0b[n] * s;
        }
        U0nb = polyb * s + sb * (R(2.0) * C[1] + R(6.0) * C[2] * IM);
    } else {
#pragma unroll
        for (int n = 0; n < 4; n++) g0nb[n] = g0b[n];
        U0nb = Ub;
    }
    U0nb = quad_lane<0>(U0nb);
#pragma unroll
    for (int i = 0; i < 3; i++) g0nb[i] = g0nb[i] - g0nb[3];
#pragma unroll
    for (int i = 0; i < 3; i++) Pb[i] = Pb[i] + U0nb * g0n[i] + R(2.0) * t.QQ[i] * g0nb[i];
    {
        int k = 0;
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int j = i + 1; j < 3; j++) {
                Pb[j] = Pb[j] + t.QR[k] * g0nb[i];
                Pb[i] = Pb[i] + t.QR[k] * g0nb[j];
                ++k;
            }
    }
#pragma unroll
    for (int i = 0; i < 3; i++) {
        xbar[i] = xbar[i] + (double)Pb[i];
        xbar[3] = xbar[3] - (double)Pb[i];
    }
    return alpha0b * alpha;
}

// FP64 element model, start of a substep for one node (Geo.cpp:307-312): g dt
// and 1 - drag formed in double; x and v in, x predicted and v advanced out.
__device__ __forceinline__ void predict64_one(const XfBodyParams& p, double x[3], double v[3]) {
    const double d = (double)p.dt;
    const double gdx = (double)p.gravity[0] * d, gdy = (double)p.gravity[1] * d;
    const double dragf = 1.0 - (double)p.drag;
    v[0] = v[0] + gdx;
    v[1] = v[1] + gdy;
    v[2] = v[2] + 0.0;
#pragma unroll
    for (int r = 0; r < 3; r++) v[r] = v[r] * dragf;
#pragma unroll
    for (int r = 0; r < 3; r++) x[r] = x[r] + v[r] * d;
}

// FP64 element model, end of a substep for one node: a pinned node returns to
// O; other nodes take the ground contact in double (static friction when the
// tangential displacement is within mu * depth, else it shrinks by mu *
// depth); then V = (X - O) / dt with 1 / dt in double.
__device__ __forceinline__ void finish64_one(const XfBodyParams& p, uint32_t flags, const double o[3], double x[3],
                                             double v[3]) {
    if (flags & 1u) {
        x[0] = o[0];
        x[1] = o[1];
        x[2] = o[2];
    } else if (p.collide & 1u) {
        const double gy = (double)p.ground_y;
        if (x[1] < gy) {
            const double mu = (double)p.friction;
            const double depth = gy - x[1];
            x[1] = gy;
            const double dx = x[0] - o[0], dz = x[2] - o[2];
            const double t2 = dx * dx + dz * dz;
            const double lim = mu * depth;
            if (t2 <= lim * lim) {
                x[0] = o[0];
                x[2] = o[2];
            } else {
                const double sc = lim / sqrt(t2);
                x[0] = x[0] - dx * sc;
                x[2] = x[2] - dz * sc;
            }
        }
    }
    const double invdt = 1.0 / (double)p.dt;
#pragma unroll
    for (int r = 0; r < 3; r++) v[r] = (x[r] - o[r]) * invdt;
}

// Square root of the element precision.
__device__ __forceinline__ float rsqrt_of(float x) { return sqrtf(x); }
__device__ __forceinline__ double rsqrt_of(double x) { return sqrt(x); }

// Reverse of the end of one substep (velocity, pin, ground contact) for one
// node, with the loss injected first when this substep ends a loss frame:
// Xb += lw_i * (x_loss - target). xs / o: the node's position before the
// contact pass and at the substep start (recorded by the forward replay).
// R: element precision of the forward (float: FP32 contact and 1.0f / dt;
// double: the FP64 element model). xbv / vbv: the node's Xb, Vb in, Xb out;
// ob receives Ob.
template <class R>
__device__ __forceinline__ void node_end_one(uint32_t i, uint32_t flags, const XfBodyParams& p,
                                             const double4* __restrict__ xs, const double4* __restrict__ o,
                                             const double4* __restrict__ xloss, const double4* __restrict__ target,
                                             const double* __restrict__ lw, double xbv[3], const double vbv[3],
                                             double ob[3]) {
    if (xloss) {
        double4 xl = xloss[i], tg = target[i];
        double wl = lw[i];
        xbv[0] = xbv[0] + wl * (xl.x - tg.x);
        xbv[1] = xbv[1] + wl * (xl.y - tg.y);
        xbv[2] = xbv[2] + wl * (xl.z - tg.z);
    }
    const double invdt = sizeof(R) == 4 ? (double)p.invdt : 1.0 / (double)p.dt;
    double xcb[3];
#pragma unroll
    for (int r = 0; r < 3; r++) {
        xcb[r] = xbv[r] + vbv[r] * invdt;
        ob[r] = 0.0 - vbv[r] * invdt;
    }
    double out[3] = {xcb[0], xcb[1], xcb[2]};
    if (flags & 1u) {
#pragma unroll
        for (int r = 0; r < 3; r++) {
            ob[r] = ob[r] + xcb[r];
            out[r] = 0.0;
        }
    } else if (p.collide & 1u) {
        double4 s4 = xs[i], o4 = o[i];
        R gy = (R)p.ground_y;
        R xy = (R)s4.y;
        if (xy < gy) {
            R mu = (R)p.friction;
            R depth = gy - xy;
            R dx = (R)(s4.x - o4.x), dz = (R)(s4.z - o4.z);
            R t2 = dx * dx + dz * dz;
            R lim = mu * depth;
            out[1] = 0.0;
            if (t2 <= lim * lim) {
                ob[0] = ob[0] + xcb[0];
                ob[2] = ob[2] + xcb[2];
                out[0] = 0.0;
                out[2] = 0.0;
            } else {
                R L = rsqrt_of(t2);
                R ux = dx / L, uz = dz / L;
                R bx = (R)xcb[0], bz = (R)xcb[2];
                R ubv = ux * bx + uz * bz;
                R kk = lim / L;
                R px = kk * (bx - ux * ubv), pz = kk * (bz - uz * ubv);
                out[0] = xcb[0] - (double)px;
                out[2] = xcb[2] - (double)pz;
                ob[0] = ob[0] + (double)px;
                ob[2] = ob[2] + (double)pz;
                out[1] = (double)(mu * ubv);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < 3; r++) xbv[r] = out[r];
}

// Reverse of the prediction (Geo.cpp:307-312) for one node: Xb <- Xb + Ob,
// Vb <- Xb_pred * dt * (1 - drag) (1 - drag: the FP32 value, or formed in
// double for the FP64 element model).
template <class R>
__device__ __forceinline__ void node_start_one(const XfBodyParams& p, double xb[3], const double ob[3],
                                               double vb[3]) {
    const double dt = (double)p.dt;
    const double dragf = sizeof(R) == 4 ? (double)p.dragf : 1.0 - (double)p.drag;
#pragma unroll
    for (int r = 0; r < 3; r++) {
        const double x0b = xb[r];
        xb[r] = x0b + ob[r];
        vb[r] = (x0b * dt) * dragf;
    }
}

}  // namespace
