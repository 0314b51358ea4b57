// xf_body.h -- arguments of the whole-call launches of small bodies
// (xf_body.hip), filled by xf_scene.cpp.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "xf_device.h"

// LDS slot of the body's node i: the index with its two low bits turned by the
// higher ones. Tets of a structured colour take nodes at strides of 4 and of
// whole rows, whose 32-byte records would lie in one of the four bank groups
// (24 colours of 256 tets: 1.58 us a phase, 2.27 without the turn; 48-byte
// records 1.48 to 1.72, but they leave fewer bodies that fit).
__host__ __device__ inline uint32_t xf_body_slot(uint32_t i) {
    return i ^ (((i >> 2) ^ (i >> 4) ^ (i >> 6) ^ (i >> 8) ^ (i >> 10)) & 3u);
}

// One workgroup per body runs every substep of a step call with the body's
// nodes in LDS.
struct XfBodyArgs {
    uint32_t substeps;
    uint32_t ncol;      // colours per body in rec, padded to an even number with empty ones
    uint32_t ntet;      // tets of the scene
    uint32_t nmax;      // LDS slots of the largest body (its nodes, rounded up to 4)
    uint32_t vpasses;   // volume passes (most of any body)
    uint32_t post;      // damping passes after the velocity update: bit 0 Rayleigh post, bit 1 PBD
    uint32_t tick;      // Settings::tickId of the first substep
    float time;         // simulation time before the first substep
    float dt, comp1, a; // substep length, uniform material (scenes without per-tet slots)
};

// The device arrays of such a launch.
struct XfBodyData {
    const uint32_t* rec;     // per body, ncol (first schedule position, count) pairs
    const uint2* loc;        // per schedule position: four body-local nodes, 16 bits each
    const float4 *tg0, *tg1, *tg2, *tg3, *taux;
    const float2* tdmp;
    double4 *X, *O, *V;
    const XfBodyParams* bodies;
    float* clock;            // left at the end of the call
};

// Checkpoint windows of the adjoint of small bodies (xf_body_adjoint.hip):
// one launch replays one window (workgroups [0, replays)) and reverses
// another (the rest), a workgroup per body. N: nodes of the scene.
struct XfBodyWindowArgs {
    uint32_t nbodies;
    uint32_t replays;   // workgroups that roll a window forward: nbodies or 0
    uint32_t reverses;  // workgroups that reverse one: nbodies or 0
    uint32_t ncol, ntet, nmax, N;
    uint32_t cmax;      // most tets of a body in one colour
    uint32_t roll_len, rev_len;  // substeps of the two windows
    uint32_t rev_end;   // substep count at the end of the reversed window
    uint32_t n_loss;    // loss substeps up to rev_end
    float dt, comp1, a;
};

struct XfBodyWindowData {
    const uint32_t* rec;
    const uint2* loc;
    const float4 *tg0, *tg1, *tg2, *tg3, *taux;
    const XfBodyParams* bodies;
    const double4* O;    // flags (.w)
    // roll: start state, and either its records (tape, xs, oo) or its end state (x1, v1)
    const double4 *x0, *v0;
    double* tape_rec;
    double4 *xs_rec, *oo_rec;
    double4 *x1, *v1;
    // reverse: records of its window, inverse masses, adjoint state, gradients, loss frames
    const double* tape_rev;
    const double4 *xs_rev, *oo_rev, *W;
    double4 *Xb, *Vb;
    void* gacc;          // float, or double in the FP64 element model
    double* glog;
    const double4 *xloss, *target;
    const double* lw;
    const uint32_t* loss_at;
};
