// xf_tiles.cpp -- cuts a scene into tiles and a sweep into spans of colours
// for the tile launches (xf_tile.hip).
#include <algorithm>
#include <cmath>
#include <new>
#include <numeric>
#include <system_error>
#include <thread>

#include "xf_tile.h"

namespace {

constexpr uint32_t kNone = ~0u;
constexpr uint32_t kMaxSpan = 12;
constexpr uint32_t kMaxPhase = 4 * kTileThreads;

// Estimated times in microseconds (measured): a launch up to its first phase
// and after its last, and a phase of cnt tets (up to 64 on quads; a wave on
// each SIMD; two; further tets in turn). A sweep's sum and what it took:
// 12x7x7 beam, 24 colours 35.5 and 32.2, 24x12x12 41.1 and 34.8, 64x16x16 47.3
// and 43.8, 96x24x24 58.4 and 65.5 (31 greedy colours 76.1 and 86.8), 128x36x36
// 86.1 and 107 (99.6 and 137): a fifth too much to a quarter too little,
// where the launches per colour that it is compared with take twice as long.
double LaunchUs(size_t nodes) { return 4.6 + 0.5 * (double)nodes / 1024.0; }
double PhaseUs(uint32_t cnt) {
    if (cnt == 0) return 0.1;
    if (cnt <= kTileQuadTets) return 0.85;
    if (cnt <= 256) return 1.3;
    return 2.0 + 1.4 * ((cnt - 1) / 512);
}

// Halves ids along the longest side of its box until a part is one tile.
void Bisect(const float* xyz, uint32_t* ids, uint32_t n, uint32_t parts, std::vector<uint32_t>* size) {
    if (parts <= 1) {
        size->push_back(n);
        return;
    }
    auto at = [&](uint32_t i, int r) {
        const float v = xyz[3 * (size_t)i + r];
        return std::isfinite(v) ? v : 0.0f;  // an order for any input
    };
    float lo[3], hi[3];
    for (int r = 0; r < 3; r++) lo[r] = hi[r] = at(ids[0], r);
    for (uint32_t i = 1; i < n; i++)
        for (int r = 0; r < 3; r++) {
            lo[r] = std::min(lo[r], at(ids[i], r));
            hi[r] = std::max(hi[r], at(ids[i], r));
        }
    int ax = 0;
    for (int r = 1; r < 3; r++)
        if (hi[r] - lo[r] > hi[ax] - lo[ax]) ax = r;
    const uint32_t left = parts / 2, cut = (uint32_t)((uint64_t)n * left / parts);
    std::nth_element(ids, ids + cut, ids + n, [&](uint32_t a, uint32_t b) {
        const float va = at(a, ax), vb = at(b, ax);
        return va < vb || (va == vb && a < b);
    });
    Bisect(xyz, ids, cut, left, size);
    Bisect(xyz, ids + cut, n - cut, parts - left, size);
}

// What a tile reads for a span, built from its last colour backwards: the
// nodes in the order they are needed, and per depth (colours from the end)
// the tets.
struct Reach {
    std::vector<uint32_t> nodes;
    std::vector<uint32_t> pos;
    std::vector<uint2> loc;
    std::vector<uint32_t> ent_end, node_end;  // per depth
    std::vector<double> us;                   // of the launch, by the depth
};

// Builds the reach of one tile after another.
class Reacher {
public:
    Reacher(const XfTileMesh& m, const uint32_t* touch, uint32_t node_limit)
        : m_(m), touch_(touch), node_limit_(node_limit) {}

    // The reach of the tile that owns the n nodes own, for spans of up to
    // depths colours that end before colour end. Returns the depths that are
    // of use: within the limits of a workgroup, and not far past the one at
    // which the tile's time per colour is least.
    uint32_t Run(Reach* r, const uint32_t* own, uint32_t n, uint32_t end, uint32_t depths) {
        r->nodes.assign(own, own + n);
        r->pos.clear();
        r->loc.clear();
        r->ent_end.clear();
        r->node_end.clear();
        r->us.clear();
        if (node_seen_.empty()) {
            node_seen_.assign(m_.n_nodes, 0u);
            tet_seen_.assign(m_.n_tets, 0u);
            local_.resize(m_.n_nodes);
        }
        ++stamp_;
        for (uint32_t k = 0; k < n; k++) {
            node_seen_[own[k]] = stamp_;
            local_[own[k]] = (uint16_t)k;
        }
        double us = 0.0, least = 0.0;
        for (uint32_t d = 0; d < depths; d++) {
            const uint32_t c = end - 1 - d, known = (uint32_t)r->nodes.size(), before = (uint32_t)r->pos.size();
            for (uint32_t k = 0; k < known; k++) {
                const uint32_t t = touch_[(size_t)r->nodes[k] * m_.ncol + c];
                if (t == kNone || tet_seen_[t] == stamp_) continue;
                tet_seen_[t] = stamp_;
                const uint4 id = m_.tidx[t];
                uint32_t l[4];
                int i = 0;
                for (uint32_t g : {id.x, id.y, id.z, id.w}) {
                    if (node_seen_[g] != stamp_) {
                        node_seen_[g] = stamp_;
                        local_[g] = (uint16_t)r->nodes.size();
                        r->nodes.push_back(g);
                    }
                    l[i++] = local_[g];
                }
                r->pos.push_back(t);
                r->loc.push_back(make_uint2(l[0] | (l[1] << 16), l[2] | (l[3] << 16)));
            }
            const uint32_t cnt = (uint32_t)r->pos.size() - before;
            if (r->nodes.size() > node_limit_ || cnt > kMaxPhase) return d;
            us += PhaseUs(cnt);
            r->us.push_back(us + LaunchUs(r->nodes.size()));
            r->ent_end.push_back((uint32_t)r->pos.size());
            r->node_end.push_back((uint32_t)r->nodes.size());
            const double per = r->us.back() / (d + 1);
            if (d == 0 || per < least) least = per;
            else if (per > 1.05 * least) return d + 1;
        }
        return depths;
    }

private:
    const XfTileMesh& m_;
    const uint32_t* touch_;
    uint32_t node_limit_, stamp_ = 0;
    std::vector<uint32_t> node_seen_, tet_seen_;  // by stamp
    std::vector<uint16_t> local_;
};

// Workers for a scene of so many tets.
uint32_t Workers(uint32_t n_tets) {
    return std::max(1u, std::min({8u, std::thread::hardware_concurrency(), n_tets / 4096}));
}

// f(k) for k < n on a thread each (on this one where there is one, or no
// thread or memory for one to be had); the least of the results, 0 if one ran
// out of memory.
template <class F>
uint32_t Share(uint32_t n, F f) {
    std::vector<uint32_t> out(n, 0u);
    auto run = [&](uint32_t k) {
        try {
            out[k] = f(k);
        } catch (const std::bad_alloc&) {
            out[k] = 0;
        }
    };
    std::vector<std::thread> threads;
    threads.reserve(n);
    uint32_t started = 1;
    try {
        for (; started < n; started++) threads.emplace_back(run, started);
    } catch (const std::system_error&) {
    } catch (const std::bad_alloc&) {  // the threads that run are still joined
    }
    run(0);
    for (uint32_t k = started; k < n; k++) run(k);
    for (std::thread& t : threads) t.join();
    return *std::min_element(out.begin(), out.end());
}

XfTilePlan Plan(const XfTileMesh& m) {
    XfTilePlan plan;
    const uint32_t B = (uint32_t)m.xyz.size();
    // tiles per body: one to a compute unit, each next one to the body whose
    // tiles are largest, down to 16 nodes
    std::vector<uint32_t> tiles(B, 1u);
    auto nodes_of = [&](uint32_t b) { return m.body_begin[b + 1] - m.body_begin[b]; };
    auto smaller = [&](uint32_t a, uint32_t b) {
        return (uint64_t)nodes_of(a) * tiles[b] < (uint64_t)nodes_of(b) * tiles[a];
    };
    std::vector<uint32_t> heap(B);
    std::iota(heap.begin(), heap.end(), 0u);
    std::make_heap(heap.begin(), heap.end(), smaller);
    for (uint32_t total = B; total < m.n_cu && nodes_of(heap[0]) > 16 * tiles[heap[0]]; total++) {
        std::pop_heap(heap.begin(), heap.end(), smaller);
        tiles[heap.back()]++;
        std::push_heap(heap.begin(), heap.end(), smaller);
    }
    std::vector<uint32_t> order(m.n_nodes), size, body;
    for (uint32_t b = 0; b < B; b++) {
        const uint32_t first = m.body_begin[b], n = nodes_of(b);
        std::vector<uint32_t> ids(n);
        std::iota(ids.begin(), ids.end(), 0u);
        Bisect(m.xyz[b], ids.data(), n, tiles[b], &size);
        for (uint32_t i = 0; i < n; i++) order[first + i] = first + ids[i];
        body.resize(size.size(), b);
    }
    const uint32_t S = (uint32_t)size.size();
    plan.ntile = S;
    plan.own_max = *std::max_element(size.begin(), size.end());
    const uint32_t node_limit = std::min(65535u, m.lds_limit / kTileNodeBytes);
    if (S > m.n_cu || plan.own_max > node_limit) return XfTilePlan();

    // the tet of a node in a colour
    std::unique_ptr<uint32_t[]> touch(new uint32_t[(size_t)m.n_nodes * m.ncol]);
    const uint32_t fillers = Workers(m.n_tets);
    Share(fillers, [&](uint32_t k) {
        const size_t all = (size_t)m.n_nodes * m.ncol;
        std::fill(&touch[all * k / fillers], &touch[0] + all * (k + 1) / fillers, kNone);
        return 1u;
    });
    Share(fillers, [&](uint32_t k) {
        for (uint32_t c = k; c < m.ncol; c += fillers)
            for (uint32_t i = m.colour_begin[c]; i < m.colour_begin[c + 1]; i++) {
                const uint4 t = m.tidx[i];
                for (uint32_t g : {t.x, t.y, t.z, t.w}) touch[(size_t)g * m.ncol + c] = i;
            }
        return 1u;
    });

    std::vector<uint32_t> own(S);  // a tile's first node in order
    for (uint32_t s = 1; s < S; s++) own[s] = own[s - 1] + size[s - 1];
    std::vector<Reach> reach(S);
    std::vector<Reacher> workers;
    for (uint32_t w = 0; w < Workers(m.n_tets); w++) workers.emplace_back(m, touch.get(), node_limit);
    const uint32_t W = (uint32_t)workers.size();
    uint32_t depth_limit = kMaxSpan;
    for (uint32_t end = m.ncol; end > 0;) {
        const uint32_t depths = Share(W, [&](uint32_t k) {
            uint32_t most = std::min(end, depth_limit);
            for (uint32_t s = k; s < S && most > 0; s += W)
                most = workers[k].Run(&reach[s], order.data() + own[s], size[s], end, most);
            return most;
        });
        if (depths == 0) return XfTilePlan();
        // the span length of the least time per colour
        uint32_t best = 0;
        double best_us = 0.0;
        for (uint32_t d = 1; d <= depths; d++) {
            double us = 0.0;
            for (const Reach& r : reach) us = std::max(us, r.us[d - 1]);
            if (best == 0 || us * best < best_us * d) {
                best = d;
                best_us = us;
            }
        }
        plan.us += best_us;
        depth_limit = std::min(kMaxSpan, best + 2);
        XfTileSpan span;
        span.nph = best;
        span.meta = plan.meta.size();
        span.rec = plan.rec.size();
        span.node0 = plan.n_node;
        span.ent0 = plan.n_ent;
        for (uint32_t s = 0; s < S; s++) {
            const Reach& r = reach[s];
            const uint32_t n = r.node_end[best - 1];
            span.nmax = std::max(span.nmax, n);
            plan.meta.push_back(make_uint4(plan.n_node, n, size[s], body[s]));
            plan.n_node += n;
            for (uint32_t d = best; d-- > 0;) {
                const uint32_t cnt = r.ent_end[d] - (d ? r.ent_end[d - 1] : 0u);
                span.pmax = std::max(span.pmax, cnt);
                plan.rec.push_back(make_uint2(plan.n_ent, cnt));
                plan.n_ent += cnt;
            }
        }
        span.n_node = plan.n_node - span.node0;
        span.n_ent = plan.n_ent - span.ent0;
        span.node.reset(new uint32_t[span.n_node]);
        span.pos.reset(new uint32_t[span.n_ent]);
        span.loc.reset(new uint2[span.n_ent]);
        Share(W, [&](uint32_t k) {
            for (uint32_t s = k; s < S; s += W) {
                const Reach& r = reach[s];
                const uint4 t = plan.meta[span.meta + s];
                std::copy_n(r.nodes.begin(), t.y, &span.node[t.x - span.node0]);
                for (uint32_t j = 0; j < best; j++) {
                    const uint2 e = plan.rec[span.rec + (size_t)s * best + j];
                    const uint32_t d = best - 1 - j, lo = d ? r.ent_end[d - 1] : 0u;
                    std::copy_n(r.pos.begin() + lo, e.y, &span.pos[e.x - span.ent0]);
                    std::copy_n(r.loc.begin() + lo, e.y, &span.loc[e.x - span.ent0]);
                }
            }
            return 1u;
        });
        plan.spans.push_back(std::move(span));
        end -= best;
    }
    return plan;
}

}  // namespace

XfTilePlan PlanTiles(const XfTileMesh& m) {
    try {
        return Plan(m);
    } catch (const std::bad_alloc&) {
        return XfTilePlan();
    }
}
