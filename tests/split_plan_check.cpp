// Host-only check of the panel planner (no device calls): the descriptors of
// large split batches fit the server's first slot size, every tile stands in the
// work list once per modulus, the reconstruction items cover every result,
// products with an empty K keep their tiles, and planes of 4 GiB and more run in
// tiles that reach all of them.
// Block addresses are stand-in integers (the planner only compares them).
#include <algorithm>
#include <cstdio>
#include <map>
#include <tuple>
#include <vector>
#include "internal.h"
using namespace sipgpu;

static int fails = 0;
#define CHECK(c) do { if (!(c)) { std::printf("FAIL %s:%d %s\n", __FILE__, __LINE__, #c); ++fails; } } while (0)

// n contractions D(a,b,i,j) = V(a,b,c,d) T(c,d,i,j) of seg^4 blocks over
// `shared` left and right blocks (0: each its own)
static rt::PanelPlan plan_of(int n, int seg, int shared, int nmod) {
    int dr = 4, lr = 4, rr = 4, ptrn[8], ierr = 0;
    int aces[12] = {1, 2, 3, 4, 1, 2, 5, 6, 5, 6, 3, 4};
    get_contraction_ptrn_(&dr, &lr, &rr, aces, ptrn, &ierr);
    CHECK(ierr == 0);
    auto ptr = [&](int id) { return (double *)(((uintptr_t)id + 1) << 32); };
    std::vector<sipgpu_contraction> list;
    for (int i = 0; i < n; ++i) {
        sipgpu_contraction e{};
        e.l = ptr(shared ? i % shared : i);
        e.r = ptr(10000 + (shared ? i / shared : i));
        e.d = ptr(20000 + i);
        e.lrank = e.rrank = e.drank = 4;
        for (int k = 0; k < 4; ++k) e.ldims[k] = e.rdims[k] = e.ddims[k] = seg;
        for (int k = 0; k < 8; ++k) e.ptrn[k] = ptrn[k];
        e.accumulate = 1;
        list.push_back(e);
    }
    rt::PanelPlan p;
    CHECK(rt::build_panel_plan(list.data(), n, nmod, p) == 0);
    return p;
}

static void check_lists(const rt::PanelPlan &p) {
    const OzTask *tasks = (const OzTask *)(p.host.data() + p.o_tasks);
    const OzUnit *units = (const OzUnit *)(p.host.data() + p.o_tiles);
    const int edge = oz_tile_size(p.tile);
    std::map<std::tuple<int, int, int>, int> seen; // (task, tile, modulus)
    for (int i = 0; i < p.ntiles; ++i)
        if (units[i].task >= 0)
            seen[{units[i].task, (int)(units[i].tile >> 4), (int)(units[i].tile & 15)}]++;
    size_t want = 0;
    for (int t = 0; t < p.ngroups; ++t) {
        const int tiles = ((tasks[t].M + edge - 1) / edge) * ((tasks[t].N + edge - 1) / edge);
        want += (size_t)tiles * p.nmod;
        for (int q = 0; q < tiles; ++q)
            for (int m = 0; m < p.nmod; ++m) CHECK((seen[{t, q, m}]) == 1);
    }
    CHECK(seen.size() == want);
    const OzRecItem *rec = (const OzRecItem *)(p.host.data() + p.o_rec);
    std::vector<long long> next(p.ngroups, 0);
    for (int i = 0; i < p.nrec; ++i) {
        CHECK(rec[i].e0 == next[rec[i].task]);
        next[rec[i].task] += kOzRecPer * kOzRecChunk;
    }
    for (int t = 0; t < p.ngroups; ++t) CHECK(next[t] >= (long long)tasks[t].M * tasks[t].N);
}

// Batches of n products D(m,n) = L(k,m) R(k,n), every third with an empty K.
static void check_empty(int n, int nmod) {
    auto ptr = [&](int id) { return (double *)(((uintptr_t)id + 1) << 24); };
    std::vector<sipgpu_contraction> list;
    for (int i = 0; i < n; ++i) {
        sipgpu_contraction e{};
        const int K = i % 3 == 2 ? 0 : 40, ptrn[4] = {-1, 1, -1, 2};
        e.l = ptr(3 * i), e.r = ptr(3 * i + 1), e.d = ptr(3 * i + 2);
        e.lrank = e.rrank = e.drank = 2;
        e.ldims[0] = e.rdims[0] = K;
        e.ldims[1] = e.ddims[0] = 150, e.rdims[1] = e.ddims[1] = 130;
        for (int k = 0; k < 4; ++k) e.ptrn[k] = ptrn[k];
        list.push_back(e);
    }
    rt::PanelPlan p;
    CHECK(rt::build_panel_plan(list.data(), n, nmod, p) == 0);
    const OzTask *tasks = (const OzTask *)(p.host.data() + p.o_tasks);
    if (nmod) {
        check_lists(p);
        for (int t = 0; t < p.ngroups; ++t) CHECK(tasks[t].nchunks > 0 && tasks[t].nchunks % 16 == 0);
        return;
    }
    // packed: every tile once in the units or, in one or more parts, in the fixups
    const OzTile *units = (const OzTile *)(p.host.data() + p.o_tiles);
    std::map<std::tuple<int, int, int>, int> stages;
    for (int i = 0; i < p.ntiles; ++i)
        if (units[i].task >= 0)
            stages[{units[i].task, units[i].mt, units[i].nt}] += units[i].s1 - units[i].s0;
    size_t want = 0;
    for (int t = 0; t < p.ngroups; ++t)
        for (int m = 0; m < (tasks[t].M + p.tile - 1) / p.tile; ++m)
            for (int q = 0; q < (tasks[t].N + p.tile - 1) / p.tile; ++q, ++want) {
                CHECK(stages.count({t, m, q}) == 1);
                CHECK((stages[{t, m, q}]) == tasks[t].nchunks);
            }
    CHECK(stages.size() == want);
}

int main() {
    const size_t slot = 32u << 20;
    const int batches[3][3] = {{256, 50, 0}, {256, 60, 16}, {120, 64, 0}};
    for (const auto &b : batches) {
        const rt::PanelPlan p = plan_of(b[0], b[1], b[2], 14);
        std::printf("%d of %d^4: %.1f MiB\n", b[0], b[1], p.host.size() / 1048576.0);
        CHECK(p.host.size() <= slot);
    }
    check_lists(plan_of(3, 7, 0, 6));
    check_lists(plan_of(5, 17, 2, 14));
    check_lists(plan_of(40, 23, 0, 13));
    {
        const rt::PanelPlan below = plan_of(100, 64, 0, 6), above = plan_of(140, 64, 0, 6);
        CHECK(below.plane_bytes < 1LL << 32 && below.tile == kOzWideTile);
        CHECK(above.plane_bytes > 1LL << 32 && above.tile == kOzBM);
        check_lists(above);
        // every chunk's rows lie inside the plane, at offsets past 32 bits too
        const OzTask *tasks = (const OzTask *)(above.host.data() + above.o_tasks);
        const OzChunkRef *chunks = (const OzChunkRef *)(above.host.data() + above.o_chunks);
        long long last = 0;
        for (int t = 0; t < above.ngroups; ++t)
            for (int c = 0; c < tasks[t].nchunks; ++c) {
                const OzChunkRef &r = chunks[tasks[t].chunk0 + c];
                last = std::max({last, oz_row(r.a, tasks[t].M - 1, r.stride),
                                 oz_row(r.b, tasks[t].N - 1, r.stride)});
            }
        CHECK(last > 1LL << 32 && last + kOzChunk <= above.plane_bytes);
    }
    for (int n : {1, 3, 20, 900})
        for (int nmod : {0, 6, 14}) check_empty(n, nmod);
    std::printf(fails ? "FAILED %d\n" : "all ok\n", fails);
    return fails != 0;
}
