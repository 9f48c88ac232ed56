// Host-only check of a single contraction's tiles and K segments (no device
// calls).  With an argument, the configuration that SIPGPU_GEMM_CONFIG pins: every
// plan keeps it.
#include <cstdio>
#include <cstdlib>
#include "internal.h"
using namespace sipgpu;

static int fails = 0;
#define CHECK(c) do { if (!(c)) { std::printf("FAIL %s:%d %s\n", __FILE__, __LINE__, #c); ++fails; } } while (0)

static rt::SegmentPlan plan(int M, int N, int K, int kfast, int beta = 0) {
    GemmTask t{};
    GemmPair p{};
    t.M = M, t.N = N, t.npairs = 1, t.beta = beta;
    p.K = K, p.flags = kfast;
    const rt::SegmentPlan s = rt::plan_single(t, p, (int64_t)M * N);
    CHECK(s.nseg >= 1 && (int64_t)s.nseg * s.kseg >= K && (int64_t)(s.nseg - 1) * s.kseg < K);
    CHECK((int64_t)(s.nseg - 1) * M * N <= 2 << 20); // the no-allocation workspace
    return s;
}

int main(int argc, char **argv) {
    if (argc > 1) {
        for (int M : {33, 320, 850})
            for (int K : {100, 1024, 4096})
                for (int kfast : {0, 1, 3}) CHECK(plan(M, 296, K, kfast).cfg == std::atoi(argv[1]));
    } else {
        CHECK(plan(100, 100, 100, 3).cfg == kGemmSplitK && plan(100, 100, 100, 3).nseg == 1);
        CHECK(plan(450, 450, 450, 0).cfg == kGemmSplitK);
        CHECK(plan(850, 296, 2048, 3).cfg == kGemm64x64 && plan(850, 296, 2048, 3).nseg > 1);
        CHECK(plan(1200, 1200, 1200, 0).cfg == kGemmSplitK);
        CHECK(plan(2304, 2304, 1600, 0).cfg == kGemm64x64);
        // more 64 x 64 tiles than CUs: by K
        CHECK(plan(945, 2065, 9, 1).cfg == kGemm64x64);
        CHECK(plan(1453, 1358, 51, 1).cfg == kGemm64x64);
        CHECK(plan(675, 2184, 54, 1, 1).cfg == kGemmSplitK);
        CHECK(plan(1600, 900, 1600, 1).cfg == kGemmSplitK);
    }
    std::printf(fails ? "FAILED %d\n" : "all ok\n", fails);
    return fails != 0;
}
