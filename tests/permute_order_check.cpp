// Host-only check of the permutes' tile order (no device calls): over a batch's
// workgroups every tile of every entry is visited once, workgroup numbers decoded
// as the kernel decodes them; entries of fewer than 8 tiles have no empty
// workgroup; blocks beyond the cache stream whole lines (a permute on its own: half
// lines) and whole rows only.
#include <cstdio>
#include <vector>
#include "kernels.h"
#include "plan.h"
using namespace sipgpu;

static int fails = 0;
#define CHECK(c) do { if (!(c)) { std::printf("FAIL %s:%d %s\n", __FILE__, __LINE__, #c); ++fails; } } while (0)

struct Shape {
    std::vector<int> dims, perm;
};

static std::vector<PermArgs> args_of(const std::vector<Shape> &shapes, std::vector<int> &first,
                                     uintptr_t base = 1 << 20) {
    const int n = (int)shapes.size();
    std::vector<PermutePlan> plans(n);
    std::vector<const double *> in(n);
    std::vector<double *> out(n);
    for (int e = 0; e < n; ++e) {
        std::vector<int> t{1};
        t.insert(t.end(), shapes[e].perm.begin(), shapes[e].perm.end());
        CHECK(plan_permute((int)shapes[e].dims.size(), shapes[e].dims.data(), t.data(), plans[e]) == 0);
        in[e] = (const double *)(base + ((uintptr_t)e << 36));
        out[e] = (double *)(base + ((uintptr_t)e << 36) + ((uintptr_t)1 << 35));
    }
    std::vector<PermArgs> a(n);
    first.assign(n + 1, 0);
    int cap = 0, tv = 0;
    const int64_t total = permute_batch_args(plans.data(), in.data(), out.data(), n, a.data(),
                                             first.data(), &cap, &tv);
    CHECK(total == first[n]);
    return a;
}

static void check(const std::vector<Shape> &shapes) {
    std::vector<int> first;
    const auto args = args_of(shapes, first);
    for (size_t e = 0; e < args.size(); ++e) {
        const PermArgs &a = args[e];
        const int tiles = a.tilesU * a.tilesV, groups = first[e + 1] - first[e];
        std::vector<int> seen(tiles, 0);
        for (int blk = 0; blk < groups; ++blk) {
            const int r = (int)fastdiv(blk, a.round), q = blk - r * (int)a.round.d;
            const int at = r * 8 + ((q - a.turn) & 7), in_patch = q >> 3;
            const int pv = (int)fastdiv(at, a.patchesU), pu = at - pv * (int)a.patchesU.d;
            const int iv = (int)fastdiv(in_patch, a.patchU), iu = in_patch - iv * (int)a.patchU.d;
            const int bu = pu * (int)a.patchU.d + iu;
            const int bv = pv * (int)fastdiv(a.patch.d, a.patchU) + iv;
            if (bu >= a.tilesU || bv >= a.tilesV) continue;
            seen[bv * a.tilesU + bu]++;
        }
        for (int s : seen) CHECK(s == 1);
        if (tiles < 8) CHECK(groups == tiles);
    }
}

int main() {
    const std::vector<Shape> small = {
        {{2, 3}, {2, 1}}, {{32, 64}, {2, 1}}, {{33, 65}, {2, 1}}, {{10, 10, 10, 10}, {3, 4, 1, 2}},
        {{4, 5, 6}, {3, 1, 2}}, {{21, 10, 12, 9}, {2, 1, 4, 3}}, {{13, 11, 17}, {1, 2, 3}}};
    const std::vector<Shape> mid = {
        {{512, 1024}, {2, 1}}, {{511, 1025}, {2, 1}}, {{31, 7, 29, 21}, {3, 4, 1, 2}},
        {{40, 39, 38, 37}, {4, 3, 2, 1}}, {{41, 30, 29, 7}, {1, 3, 2, 4}}, {{16, 32, 48, 16}, {3, 4, 1, 2}}};
    for (const Shape &s : small) check({s});
    check(small);
    std::vector<Shape> all = mid;
    for (int c = 0; c < 3; ++c)
        for (size_t i = 0; i < small.size(); ++i) {
            all.push_back(small[(i + c) % small.size()]);
            all.push_back(mid[(i * 5 + c) % mid.size()]);
        }
    check(all);
    // stores of a batch beyond the cache: whole lines written (reads ragged or
    // not), whole rows, identity; ragged runs, and a block off its line
    std::vector<int> first;
    auto streams = [&](const Shape &s, uintptr_t base) {
        return args_of({s, {{7001, 5003}, {2, 1}}}, first, base)[0].stream;
    };
    CHECK(streams({{512, 1024}, {2, 1}}, 1 << 20) == 1);
    CHECK(streams({{511, 1024}, {2, 1}}, 1 << 20) == 1);
    CHECK(streams({{512, 1041}, {2, 1}}, 1 << 20) == 0);
    CHECK(streams({{36, 14, 18, 18, 20, 15}, {6, 2, 4, 3, 5, 1}}, 1 << 20) == 0);
    CHECK(streams({{36, 14, 18, 18, 20, 16}, {6, 2, 4, 3, 5, 1}}, 1 << 20) == 1);
    CHECK(streams({{512, 1024}, {2, 1}}, (1 << 20) + 8) == 0);
    // runs of several dims: 18 x 22, 26, 12 follow each other, 24.75 lines each
    CHECK(streams({{23, 15, 26, 18, 22, 12}, {5, 6, 3, 1, 2, 4}}, 1 << 20) == 1);
    CHECK(streams({{23, 15, 26, 18, 22, 11}, {5, 6, 3, 1, 2, 4}}, 1 << 20) == 0);
    CHECK(args_of({{{25, 44, 50, 31, 36}, {5, 3, 1, 4, 2}}}, first)[0].TV % 16 == 0);
    CHECK(streams({{42, 39, 28, 42, 22}, {3, 5, 1, 2, 4}}, 1 << 20) == 0);
    CHECK(streams({{41, 30, 29, 7}, {1, 3, 2, 4}}, 1 << 20) == 1);
    CHECK(streams({{13, 11, 17}, {1, 2, 3}}, 1 << 20) == 1);
    // a permute on its own also streams whole halves of lines: 28 x 42 = 73.5 lines,
    // blocks at half a line; not quarters, nor tiles of 66 v
    auto alone = [&](const Shape &s, uintptr_t base) {
        std::vector<int> t{1};
        t.insert(t.end(), s.perm.begin(), s.perm.end());
        PermutePlan plan;
        CHECK(plan_permute((int)s.dims.size(), s.dims.data(), t.data(), plan) == 0);
        PermArgs a;
        CHECK(permute_args(plan, (const double *)base, (double *)(base + ((uintptr_t)1 << 35)), a) > 0);
        return a.stream;
    };
    CHECK(alone({{42, 39, 28, 42, 22}, {3, 5, 1, 2, 4}}, 1 << 20) == 1);
    CHECK(alone({{42, 39, 28, 42, 22}, {3, 5, 1, 2, 4}}, (1 << 20) + 64) == 1);
    CHECK(alone({{42, 39, 28, 42, 22}, {3, 5, 1, 2, 4}}, (1 << 20) + 32) == 0);
    CHECK(alone({{5934, 6104}, {2, 1}}, 1 << 20) == 1);
    CHECK(alone({{33, 35, 30, 34, 31}, {3, 5, 1, 2, 4}}, 1 << 20) == 0);
    CHECK(alone({{93, 72, 110, 73}, {2, 1, 3, 4}}, 1 << 20) == 0);
    std::printf(fails ? "FAILED %d\n" : "all ok\n", fails);
    return fails != 0;
}
