// tile_plan_test.cpp -- the plan of the tile launches on the CPU: prints the
// spans of a block's plan, or runs PlanTiles with memory that runs out at the
// k-th allocation for k = 0, step, 2 step, ... (once, or from then on): it must
// return, with a whole plan or none.
//   tile_plan_test plan W H D colours       colours: 24 (structured) or greedy
//   tile_plan_test memory W H D colours step
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>

#include "../../xpbd-fem_amd/csrc/xf_tiles.cpp"

static std::atomic<long> g_left{-1};  // allocations until one fails; < 0: none does
static std::atomic<bool> g_stay{false};
static std::atomic<long> g_count{0};

void* operator new(size_t n) {
    g_count++;
    if (g_left.load() >= 0) {
        const long k = g_left.fetch_sub(1);
        if (k <= 0) {
            if (g_stay.load()) g_left.store(0);
            else g_left.store(-1);
            throw std::bad_alloc();
        }
    }
    if (void* p = malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void* operator new[](size_t n) { return operator new(n); }
void operator delete(void* p) noexcept { free(p); }
void operator delete[](void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }
void operator delete[](void* p, size_t) noexcept { free(p); }

int main(int argc, char** argv) {
    if (argc < 6) return 2;
    const uint32_t W = atoi(argv[2]), H = atoi(argv[3]), D = atoi(argv[4]);
    const bool greedy = strcmp(argv[5], "greedy") == 0;
    const uint32_t N = (W + 1) * (H + 1) * (D + 1), T = 6 * W * H * D;
    std::vector<float> xyz;
    for (uint32_t z = 0; z <= D; z++)
        for (uint32_t y = 0; y <= H; y++)
            for (uint32_t x = 0; x <= W; x++) xyz.insert(xyz.end(), {(float)x, (float)y, (float)z});
    // the six tets of a cell: paths of unit steps from corner to corner
    static const int kPath[6][3] = {{0, 1, 2}, {1, 2, 0}, {2, 0, 1}, {1, 0, 2}, {0, 2, 1}, {2, 1, 0}};
    const uint32_t stride[3] = {1, W + 1, (W + 1) * (H + 1)};
    std::vector<uint4> tets;
    std::vector<uint32_t> colour;
    std::vector<uint64_t> used(N, 0);
    for (uint32_t z = 0; z < D; z++)
        for (uint32_t y = 0; y < H; y++)
            for (uint32_t x = 0; x < W; x++)
                for (uint32_t s = 0; s < 6; s++) {
                    uint32_t n[4];
                    n[0] = x + (W + 1) * (y + (H + 1) * z);
                    for (int k = 0; k < 3; k++) n[k + 1] = n[k] + stride[kPath[s][k]];
                    uint32_t c = 6 * ((x + y + z) % 4) + s;
                    if (greedy) {
                        const uint64_t m = used[n[0]] | used[n[1]] | used[n[2]] | used[n[3]];
                        c = (uint32_t)__builtin_ctzll(~m);
                        for (uint32_t g : n) used[g] |= 1ull << c;
                    }
                    tets.push_back(make_uint4(n[0], n[1], n[2], n[3]));
                    colour.push_back(c);
                }
    const uint32_t ncol = *std::max_element(colour.begin(), colour.end()) + 1;
    std::vector<uint4> tidx;
    std::vector<uint32_t> begin;
    for (uint32_t c = 0; c < ncol; c++) {
        begin.push_back((uint32_t)tidx.size());
        for (uint32_t t = 0; t < T; t++)
            if (colour[t] == c) tidx.push_back(tets[t]);
    }
    begin.push_back(T);
    XfTileMesh m;
    m.n_nodes = N;
    m.n_tets = T;
    m.ncol = ncol;
    m.tidx = tidx.data();
    m.colour_begin = begin.data();
    m.body_begin = {0u, N};
    m.xyz = {xyz.data()};
    m.n_cu = 256;
    m.lds_limit = 160 * 1024;

    auto colours_of = [](const XfTilePlan& p) {
        uint32_t n = 0;
        for (const XfTileSpan& sp : p.spans) n += sp.nph;
        return n;
    };
    if (strcmp(argv[1], "plan") == 0) {
        const XfTilePlan p = PlanTiles(m);
        printf("%ux%ux%u, %u colours: %u tiles, %u own nodes, %zu spans, %.1f us, %.2f entries a tet\n", W, H, D, ncol,
               p.ntile, p.own_max, p.spans.size(), p.us, (double)p.n_ent / T);
        for (size_t k = p.spans.size(); k-- > 0;)
            printf("  %u colours, %u nodes, %u tets a phase\n", p.spans[k].nph, p.spans[k].nmax, p.spans[k].pmax);
        return colours_of(p) == ncol ? 0 : 1;
    }
    const long step = argc > 6 ? atol(argv[6]) : 1;
    g_count = 0;
    if (colours_of(PlanTiles(m)) != ncol) return 1;
    const long all = g_count.load();
    uint32_t none = 0, whole = 0;
    for (int stay = 0; stay < 2; stay++)
        for (long k = 0; k < all; k += step) {
            g_stay = stay != 0;
            g_left = k;
            const XfTilePlan p = PlanTiles(m);
            g_left = -1;
            const uint32_t n = colours_of(p);
            if (n == 0) none++;
            else if (n == ncol) whole++;
            else return printf("allocation %ld: a plan of %u of %u colours\n", k, n, ncol), 1;
        }
    printf("%ld allocations: %u plans, %u without\n", all, whole, none);
    return 0;
}
