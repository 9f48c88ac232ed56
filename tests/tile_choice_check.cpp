// Host-only check of the planner's choice of tiles and path (no device calls): few
// small blocks run in 32 x 32 tiles with K split, batches whose 64 x 64 tiles
// fill the chip in those, large blocks in 64 x 64 tiles beside few small ones;
// batches of 1e9 to 5e9 flop on packed panels where their tables' chains are long.
#include <cstdio>
#include <vector>
#include "internal.h"
using namespace sipgpu;

static int fails = 0;
#define CHECK(c) do { if (!(c)) { std::printf("FAIL %s:%d %s\n", __FILE__, __LINE__, #c); ++fails; } } while (0)

// n blocks D(m,n) of `pairs` products of K each; form 0: both operands read
// along k, 1: one of them, 2: neither
static void add(std::vector<sipgpu_contraction> &list, int n, int M, int N, int K, int pairs, int form) {
    static const int ptrn[3][4] = {{-1, 1, -1, 2}, {1, -1, -2, 2}, {1, -2, 2, -2}};
    auto ptr = [&](size_t id) { return (double *)((id + 1) << 26); };
    for (int i = 0; i < n; ++i) {
        const size_t d = 3 * list.size();
        for (int p = 0; p < pairs; ++p) {
            sipgpu_contraction e{};
            e.l = ptr(3 * list.size() + 1), e.r = ptr(3 * list.size() + 2), e.d = ptr(d);
            e.lrank = e.rrank = e.drank = 2;
            e.ldims[form != 0] = e.rdims[form == 2] = K;
            e.ldims[form == 0] = e.ddims[0] = M, e.rdims[form != 2] = e.ddims[1] = N;
            for (int k = 0; k < 4; ++k) e.ptrn[k] = ptrn[form][k];
            e.accumulate = 1;
            list.push_back(e);
        }
    }
}

static std::vector<int> configs(const std::vector<sipgpu_contraction> &list) {
    rt::BatchImage img;
    CHECK(rt::build_batch_image(list.data(), (int)list.size(), img) == 0);
    std::vector<int> c;
    for (int i = 0; i < img.nlaunches; ++i) c.push_back(img.launch[i].cfg);
    return c;
}

static std::vector<int> batch(int n, int M, int N, int K, int pairs, int form) {
    std::vector<sipgpu_contraction> list;
    add(list, n, M, N, K, pairs, form);
    return configs(list);
}

// the same with one pair of operands for all
static std::vector<int> shared(int n, int M, int N, int K, int pairs, int form) {
    std::vector<sipgpu_contraction> list;
    add(list, n, M, N, K, pairs, form);
    for (auto &e : list) e.l = list[0].l, e.r = list[0].r;
    return configs(list);
}

static bool packed(int n, int M, int N, int K, int pairs, int form) {
    std::vector<sipgpu_contraction> list;
    add(list, n, M, N, K, pairs, form);
    rt::BatchImage img;
    CHECK(rt::build_batch_image(list.data(), (int)list.size(), img) == 0);
    return img.prefer_packed;
}

int main() {
    const std::vector<int> split{kGemmSplitK}, big{kGemm64x64};
    for (int form = 0; form < 3; ++form) {
        CHECK(batch(1, 100, 100, 100, 1, form) == split);
        CHECK(batch(16, 100, 100, 100, 16, form) == split); // a ladder of 16 blocks
        CHECK(batch(1000, 320, 320, 200, 1, form) == big);
        CHECK(batch(1000, 100, 100, 100, 1, form) == big);
        CHECK(batch(976, 516, 7, 8, 1, form) == big);
        CHECK(batch(2, 2000, 1100, 6, 1, form) == big);
        std::vector<sipgpu_contraction> mixed; // one large block, a few small ones
        add(mixed, 1, 2000, 1100, 6, 1, form);
        add(mixed, 3, 40, 50, 70, 1, form);
        CHECK((configs(mixed) == std::vector<int>{kGemmSplitK, kGemm64x64}));
    }
    // operands along k beyond the cache: the tiles that read them less often (split-K
    // 2617 us, 64 x 64 1879); within it, or read across k, as above
    CHECK(batch(2663, 29, 135, 391, 4, 0) == big);
    CHECK(batch(318, 14, 162, 648, 16, 0) == big);
    CHECK(shared(2663, 29, 135, 391, 4, 0) == split);
    CHECK(batch(2663, 29, 135, 391, 4, 2) == split);
    CHECK(batch(100, 29, 135, 391, 4, 0) == split);
    // measured, us in tables and packed: 1540 and 450, 990 and 290, 320 and 131
    CHECK(packed(5, 45, 84, 1949, 36, 0));
    CHECK(packed(1, 68, 118, 1760, 36, 1));
    CHECK(packed(8, 80, 78, 1326, 16, 1));
    // 39 and 72, 71 and 151, 191 and 499
    CHECK(!packed(4, 224, 268, 249, 9, 1));
    CHECK(!packed(4, 83, 1164, 320, 9, 2));
    CHECK(!packed(61, 31, 1095, 57, 16, 1));
    // below 1e9 flop, below 5e7 a block; from 5e9 on
    CHECK(!packed(1, 68, 118, 1600, 36, 1));
    CHECK(!packed(200, 100, 100, 100, 10, 0));
    CHECK(packed(64, 450, 450, 450, 1, 2));
    std::printf(fails ? "FAILED %d\n" : "all ok\n", fails);
    return fails != 0;
}
