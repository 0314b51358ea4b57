// xf_tile.h -- tile launches: several colours of a sweep in one launch, a
// workgroup per tile of nodes. PlanTiles (xf_tiles.cpp) cuts a scene into
// tiles and a sweep into spans of colours; xf_tile.hip runs them.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <memory>
#include <vector>

#include "xf_device.h"

// A tile owns a set of nodes. A span is a run of consecutive colours. For its
// own nodes' values after the span a tile needs the span's last colour's tets
// that touch them, the tets of the colour before that touch those tets'
// nodes, and so on: it projects all of these, some of them also projected by
// its neighbours, from the node values before the span, and stores its own
// nodes only. The values before the span are left alone (the launches
// alternate between two node arrays), so tiles of a launch are independent.
//
// A tile's colours are projected in order, tets of a colour share no node, and
// a tet that two tiles project reads the same values in both: the results are
// those of a launch per colour, bit for bit.
struct XfTileSpan {
    uint32_t nph = 0;   // colours
    uint32_t nmax = 0;  // most nodes of a tile
    uint32_t pmax = 0;  // most tets of a tile in one colour
    size_t meta = 0, rec = 0;  // first tile in meta; first pair in rec
    uint32_t node0 = 0, n_node = 0, ent0 = 0, n_ent = 0;  // its part of the node list and of the entries
    std::unique_ptr<uint32_t[]> node;  // scene nodes of a tile
    std::unique_ptr<uint32_t[]> pos;   // schedule position of an entry
    std::unique_ptr<uint2[]> loc;      // its four tile-local nodes, 16 bits each
};

struct XfTilePlan {
    uint32_t ntile = 0, own_max = 0;
    double us = 0.0;  // estimated time of a sweep
    uint32_t n_node = 0, n_ent = 0;
    std::vector<XfTileSpan> spans;  // last to first
    std::vector<uint4> meta;        // per span and tile: first node, nodes, own nodes (first in the list), body
    std::vector<uint2> rec;         // per span, tile and colour: first entry, tets
};

struct XfTileMesh {
    uint32_t n_nodes = 0, n_tets = 0, ncol = 0;
    const uint4* tidx = nullptr;             // by schedule position
    const uint32_t* colour_begin = nullptr;  // ncol + 1
    std::vector<uint32_t> body_begin;        // first node of each body, then n_nodes
    std::vector<const float*> xyz;           // per body
    uint32_t n_cu = 0, lds_limit = 0;
};

// Empty (no spans) when a tile of one colour is larger than a workgroup takes,
// or when memory runs out.
XfTilePlan PlanTiles(const XfTileMesh& mesh);

// Limits of a tile launch.
constexpr uint32_t kTileThreads = 512;     // most lanes
constexpr uint32_t kTileQuadTets = 64;     // a phase of up to so many tets runs on quads
constexpr uint32_t kTileNodeBytes = 48;    // LDS per node

// Threads of a launch whose tiles have at most `lanes` tets in a colour and
// own at most as many nodes.
inline uint32_t xf_tile_threads(uint32_t lanes) { return lanes <= 256 ? 256u : kTileThreads; }

struct XfTileArgs {
    uint32_t nph, nent;
    uint32_t end;  // 0: store the nodes; 1: end the substep and predict the next; 2: end it and store velocities
    float dt, comp1, a;
};

struct XfTileData {
    const uint4* meta;
    const uint2* rec;
    const uint32_t* node;
    const uint2* loc;  // by entry, as the element data and material
    const float4 *tg0, *tg1, *tg2, *tg3, *taux;
    const double4* Xin;
    double4 *Xout, *O, *V;
    const XfBodyParams* bodies;
    float* clock;  // advanced where advance is set, read by a launch with end != 0
};
