// Host-only check of a tuple's boxes (sipgpu::rt::triples_tuple_boxes): their
// count and ranges, and the refusal of tuples whose boxes 32-bit work items
// cannot number.
#include <cstdio>
#include <vector>
#include "internal.h"

static int fails = 0;
#define CHECK(c) do { if (!(c)) { std::printf("FAIL %s:%d %s\n", __FILE__, __LINE__, #c); ++fails; } } while (0)

int main() {
    auto boxes = [](const std::vector<int> &v, const std::vector<int> &o, std::vector<int> tuple,
                    sipgpu::TriplesArgs &a, long long &n) {
        n = 0;
        a = sipgpu::TriplesArgs{};
        return sipgpu::rt::triples_tuple_boxes(v, o, tuple.data(), a, n);
    };
    sipgpu::TriplesArgs a{};
    long long n = 0;
    // segments 17, 18 | 13, 14: the second ones start inside a 5-block
    CHECK(boxes({17, 18}, {13, 14}, {0, 1, 0, 1, 0, 0}, a, n) == 0);
    CHECK(n == 4LL * 4 * 4 * 4 * 3 * 3 && a.end[0] == (unsigned)n);
    CHECK(a.lo[1] == 17 && a.first[1] == 3 && a.count[1] == 4 && a.wdims[1] == 18);
    CHECK(a.lo[3] == 13 && a.first[3] == 2 && a.count[3] == 4 && a.wdims[3] == 14);
    CHECK(boxes({17, 18}, {13, 14}, {0, 2, 0, 1, 0, 0}, a, n) == SIPGPU_EARG);
    CHECK(boxes({17, 18}, {13, 14}, {0, 1, 0, -1, 0, 0}, a, n) == SIPGPU_EARG);
    // one segment each: 35, 36 and 41 5-blocks in every index
    CHECK(boxes({175}, {175}, {0, 0, 0, 0, 0, 0}, a, n) == 0 && n == 1838265625LL);
    CHECK(a.end[0] == (unsigned)n);
    CHECK(boxes({180}, {180}, {0, 0, 0, 0, 0, 0}, a, n) == SIPGPU_ESIZE); // 36^6 > 2^31
    CHECK(boxes({205}, {205}, {0, 0, 0, 0, 0, 0}, a, n) == SIPGPU_ESIZE); // 41^6 > 2^32
    CHECK(boxes({2000000}, {2000000}, {0, 0, 0, 0, 0, 0}, a, n) == SIPGPU_ESIZE);
    std::printf(fails ? "FAILED %d\n" : "all ok\n", fails);
    return fails != 0;
}
