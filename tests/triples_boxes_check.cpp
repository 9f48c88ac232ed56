// Host-only check of the boxes of (T) sums: of a tuple (triples_tuple_boxes: their
// count and ranges, and the refusal of tuples whose boxes 32-bit work items
// cannot number) and of short ranges of slots (triples_short_range: a slot has at
// most one box, a range the boxes of its slots, all slots all boxes).
#include <algorithm>
#include <cstdio>
#include <set>
#include <vector>
#include "internal.h"

static int fails = 0;
#define CHECK(c) do { if (!(c)) { std::printf("FAIL %s:%d %s\n", __FILE__, __LINE__, #c); ++fails; } } while (0)

static void check_ranges(int nvb, int nob) {
    using namespace sipgpu;
    rt::TriplesBoxes b;
    rt::triples_boxes(nvb, nob, b);
    const long long n = ((nvb + 1) / 2) * ((nob + 1) / 2), slots = 64 * n * n * n;
    std::set<unsigned> items(b.items.begin(), b.items.end()), seen;
    CHECK(items.size() == b.items.size());
    // boxes that differ by a permutation of their (virtual, occupied) pairs
    const long long pairs = (long long)nvb * nob;
    CHECK((long long)items.size() == pairs * (pairs + 1) * (pairs + 2) / 6);
    std::vector<std::vector<unsigned>> of(slots);
    unsigned list[kTriplesGroups];
    long long boxes = 0;
    for (long long s = 0; s < slots; ++s) {
        const int k = rt::triples_short_range(b, s, 1, list);
        CHECK(k <= 1);
        boxes += k;
        of[s].assign(list, list + k);
        seen.insert(list, list + k);
        for (int i = 0; i < k; ++i) CHECK(items.count(list[i]));
    }
    CHECK(boxes == pairs * pairs * pairs);
    CHECK(seen == items);
    for (long long s = 0; s < slots; s += 29)
        for (long long m : {2LL, 37LL, 64LL, 300LL, 1000LL}) {
            if (s + m > slots) continue;
            std::set<unsigned> want;
            for (long long t = s; t < s + m; ++t) want.insert(of[t].begin(), of[t].end());
            const int k = rt::triples_short_range(b, s, m, list);
            if (want.size() > kTriplesGroups)
                CHECK(k == 0);
            else
                CHECK(k == (int)want.size() && std::set<unsigned>(list, list + k) == want);
        }
}

int main() {
    check_ranges(1, 1);
    check_ranges(3, 2);
    check_ranges(4, 3);
    check_ranges(5, 4);
    auto boxes = [](const std::vector<int> &v, const std::vector<int> &o, std::vector<int> tuple,
                    sipgpu::TriplesArgs &a, long long &n, bool cut = false) {
        n = 0;
        a = sipgpu::TriplesArgs{};
        return sipgpu::rt::triples_tuple_boxes(v, o, tuple.data(), cut, a, n);
    };
    sipgpu::TriplesArgs a{};
    long long n = 0;
    // segments 17, 18 | 13, 14: the second ones start inside a 5-block
    CHECK(boxes({17, 18}, {13, 14}, {0, 1, 0, 1, 0, 0}, a, n) == 0);
    CHECK(n == 4LL * 4 * 4 * 4 * 3 * 3 && a.end[0] == (unsigned)n);
    CHECK(a.lo[1] == 17 && a.first[1] == 3 && a.count[1] == 4 && a.wdims[1] == 18);
    CHECK(a.lo[3] == 13 && a.first[3] == 2 && a.count[3] == 4 && a.wdims[3] == 14);
    // cut from the tuple's own start: the boxes its extents need, its sets one
    // array after the other
    CHECK(boxes({17, 18}, {13, 14}, {0, 1, 0, 1, 0, 0}, a, n, true) == 0);
    CHECK(n == 4LL * 4 * 4 * 3 * 3 * 3 && a.end[0] == (unsigned)n);
    CHECK(a.lo[1] == 17 && a.org[1] == 17 && a.first[1] == 0 && a.count[1] == 4);
    CHECK(a.lo[3] == 13 && a.org[3] == 13 && a.first[3] == 0 && a.count[3] == 3);
    for (int g = 0; g < 6; ++g) {
        CHECK(a.base_b[g] == a.base_a[g] + 4 * 3 * 3 && a.na1[g] == 3 && a.na2[g] == 3);
        CHECK(a.nb1[g] == 4 && a.nb2[g] == 3 && (g == 0 || a.base_a[g] == a.base_b[g - 1] + 4 * 4 * 3));
    }
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
