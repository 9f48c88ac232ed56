// triples.cpp -- host side of the on-chip-W (T) energy (triples.hip).
//
// A plan holds the classes of super-boxes that differ by a permutation of
// the pairs (a,i), (b,j), (c,k), the two packed operand panel arrays (PA over
// row sets (x, y1, y2), PB over column sets (x2, x3, y3)), and one energy
// partial per box slot.  sipgpu_triples_pack fills the panels from the T, V1 and V2
// blocks; sipgpu_triples_run computes the partials of a range of box
// slots (one workgroup per CU, each over many boxes); sipgpu_triples_energy sums
// all partials in slot order into the energy (deterministic).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <exception>
#include <memory>
#include <numeric>
#include <vector>

#include "../../include/sipgpu.h"
#include "internal.h"
#include "kernels.h"

using sipgpu::TriplesOrbit;
using sipgpu::rt::fail;
using sipgpu::rt::hip_fail;

struct sipgpu_triples_s {
    int nv = 0, no = 0;
    std::vector<int> vseg, oseg;
    sipgpu::rt::TriplesBoxes boxes;
    int nvb = 0, nob = 0;             // 5-blocks of the virtual / occupied range
    int kd = 0, kl = 0, nkp = 0;
    // device memory
    void *tables = nullptr; // orbits, ints, pointer tables
    const TriplesOrbit *d_orbits = nullptr;
    const unsigned *d_items = nullptr;
    const int *d_vext = nullptr, *d_oext = nullptr, *d_vseg_of = nullptr, *d_oseg_of = nullptr;
    const int *d_vseg_start = nullptr, *d_oseg_start = nullptr;
    const double *const *d_T = nullptr, *const *d_V1 = nullptr, *const *d_V2 = nullptr;
    const double *e_occ = nullptr, *e_vir = nullptr;
    double *PA = nullptr, *PB = nullptr;
    long long pa_doubles = 0, pb_doubles = 0;
    double *partial = nullptr, *sums = nullptr, *tuple_partial = nullptr;
    // panels cut for one tuple at a time (sipgpu_triples_tuple), allocated by the
    // first tuple that needs them, for the largest
    double *cut = nullptr;
    bool no_cut = false; // there is no room for them
    long long slots = 0;   // box slots of the super-box order
    bool packed = false;

    ~sipgpu_triples_s() {
        for (void *p : {tables, (void *)PA, (void *)PB, (void *)partial, (void *)sums,
                        (void *)tuple_partial, (void *)cut})
            if (p) (void)hipFree(p);
    }
};

namespace {

constexpr int kPerm[6][3] = {{0, 1, 2}, {0, 2, 1}, {1, 0, 2}, {1, 2, 0}, {2, 0, 1}, {2, 1, 0}};

// The 5-blocks of pair m at position q of a super-box (bit 0 virtual, bit 1 occupied).
int sub_of(unsigned q, int m) { return (int)((q >> m) & 1) | (int)((q >> (3 + m)) & 1) << 1; }

// Class that holds a slot's super-box.
long long class_of(const sipgpu::rt::TriplesBoxes &b, long long slot) {
    return std::upper_bound(b.orbits.begin(), b.orbits.end(), slot / 64,
                            [](long long s, const TriplesOrbit &o) { return s < o.first; }) -
           b.orbits.begin() - 1;
}

// True if an arrangement of the pairs of the box at position q of class o lies
// among slots [box0, box0 + nbox) (the kernel's image_slot).
bool has_image(const TriplesOrbit &o, unsigned q, long long box0, long long nbox) {
    const bool eq01 = o.p[0] == o.p[1], eq12 = o.p[1] == o.p[2];
    for (int g = 0; g < 6; ++g) {
        const int *t = kPerm[g];
        int rank = g;
        if (eq01 && eq12)
            rank = 0;
        else if (eq01)
            rank = t[0] == 2 ? 0 : t[1] == 2 ? 1 : 2;
        else if (eq12)
            rank = t[0] == 0 ? 0 : t[1] == 0 ? 1 : 2;
        unsigned at = 0;
        for (int m = 0; m < 3; ++m) {
            const int s = sub_of(q, t[m]);
            at |= (unsigned)(s & 1) << m | (unsigned)(s >> 1) << (3 + m);
        }
        const long long slot = (o.first + rank) * 64 + at;
        if (slot >= box0 && slot < box0 + nbox) return true;
    }
    return false;
}

// the 5-blocks that a segment at global index g touches
void seg_blocks(int g, int ext, int &first, int &count) {
    first = g / sipgpu::kTriplesBox;
    count = (g + ext - 1) / sipgpu::kTriplesBox - first + 1;
}

// most 5-blocks that one segment touches
int max_seg_blocks(const std::vector<int> &seg) {
    int most = 0, g = 0;
    for (int x : seg) {
        int first, count;
        seg_blocks(g, x, first, count);
        most = std::max(most, count);
        g += x;
    }
    return most;
}

} // namespace

void sipgpu::rt::triples_boxes(int nvb, int nob, TriplesBoxes &b) {
    b = TriplesBoxes{};
    b.super_v = (nvb + 1) / 2;
    // the classes and, per class, its first super-box: the 6, 3 or 1 distinct
    // arrangements of a class are consecutive
    const int n = b.super_v * ((nob + 1) / 2);
    long long first = 0;
    for (int p = 0; p < n; ++p)
        for (int q = p; q < n; ++q)
            for (int r = q; r < n; ++r) {
                b.orbits.push_back(TriplesOrbit{{p, q, r}, 0, first});
                first += p == q && q == r ? 1 : p == q || q == r ? 3 : 6;
            }
    // The boxes to compute: positions whose 5-blocks exist and whose pairs are
    // ascending (another order of equal super pairs is an image), the classes
    // dealt to the XCDs in turn.  Bit q of a mask stands for position q.
    uint64_t zero[6] = {}, asc01 = 0, asc12 = 0; // zero[d]: positions with bit d clear
    for (unsigned q = 0; q < 64; ++q) {
        const uint64_t bit = 1ull << q;
        int sub[3];
        for (int m = 0; m < 3; ++m) sub[m] = sub_of(q, m);
        for (int d = 0; d < 6; ++d)
            if (!((q >> d) & 1)) zero[d] |= bit;
        if (sub[0] <= sub[1]) asc01 |= bit;
        if (sub[1] <= sub[2]) asc12 |= bit;
    }
    for (int x = 0; x < 8; ++x) {
        b.xcd_first[x] = b.items.size();
        for (size_t c = x; c < b.orbits.size(); c += 8) {
            const int *p = b.orbits[c].p;
            uint64_t boxes = ~0ull;
            for (int m = 0; m < 3; ++m) {
                if (2 * (p[m] % b.super_v) + 1 >= nvb) boxes &= zero[m];
                if (2 * (p[m] / b.super_v) + 1 >= nob) boxes &= zero[3 + m];
            }
            if (p[0] == p[1]) boxes &= asc01;
            if (p[1] == p[2]) boxes &= asc12;
            for (; boxes; boxes &= boxes - 1)
                b.items.push_back((unsigned)(c * 64) | (unsigned)__builtin_ctzll(boxes));
        }
    }
    b.xcd_first[8] = b.items.size();
}

int sipgpu::rt::triples_short_range(const TriplesBoxes &b, long long box0, long long nbox,
                                    unsigned (&list)[kTriplesGroups]) {
    if (nbox <= 0) return 0;
    const long long c0 = class_of(b, box0), c1 = class_of(b, box0 + nbox - 1);
    if (c1 - c0 >= kTriplesGroups) return 0;
    unsigned n = 0;
    for (long long c = c0; c <= c1; ++c) {
        const auto f = b.items.begin() + b.xcd_first[c % 8],
                   l = b.items.begin() + b.xcd_first[c % 8 + 1];
        for (auto i = std::lower_bound(f, l, (unsigned)c * 64); i != l && *i / 64 == c; ++i) {
            if (!has_image(b.orbits[c], *i % 64, box0, nbox)) continue;
            if (n == kTriplesGroups) return 0;
            list[n++] = *i;
        }
    }
    return (int)n;
}

int sipgpu::rt::triples_tuple_boxes(const std::vector<int> &vseg, const std::vector<int> &oseg,
                                    const int *tuple, bool cut, TriplesArgs &a, long long &boxes) {
    // (the kernel counts work items in 32 bits and adds a stride to them)
    constexpr long long kMost = 1LL << 31;
    boxes = 1;
    for (int d = 0; d < 6; ++d) {
        const std::vector<int> &seg = d < 3 ? vseg : oseg;
        if (tuple[d] < 0 || tuple[d] >= (int)seg.size())
            return fail(SIPGPU_EARG, "triples: tuple outside the segments");
        a.lo[d] = std::accumulate(seg.begin(), seg.begin() + tuple[d], 0);
        a.wdims[d] = seg[tuple[d]];
        a.org[d] = cut ? a.lo[d] : 0;
        seg_blocks(a.lo[d] - a.org[d], a.wdims[d], a.first[d], a.count[d]);
        boxes *= a.count[d];
        if (boxes >= kMost)
            return fail(SIPGPU_ESIZE, "triples: the tuple has 2^31 boxes or more");
    }
    a.end[0] = (unsigned)boxes;
    // where the sets of the permutations are: in the whole ranges' panels, or
    // one array of sets after the other
    long long sets = 0;
    for (int g = 0; g < 6; ++g) {
        const int *p = kPerm[g];
        a.na1[g] = cut ? a.count[3 + p[0]] : a.nob;
        a.na2[g] = cut ? a.count[3 + p[1]] : a.nob;
        a.nb1[g] = cut ? a.count[p[2]] : a.nvb;
        a.nb2[g] = cut ? a.count[3 + p[2]] : a.nob;
        a.base_a[g] = (int)sets;
        if (cut) sets += (long long)a.count[p[0]] * a.na1[g] * a.na2[g];
        a.base_b[g] = (int)sets;
        if (cut) sets += (long long)a.count[p[1]] * a.nb1[g] * a.nb2[g];
        if (sets >= kMost) return fail(SIPGPU_ESIZE, "triples: too many sets in a tuple");
    }
    return 0;
}

namespace {

// Room for the panels of any tuple cut from its own start: true if there is (not
// where it would take more than the whole ranges' panels, and a capture does not
// allocate).
bool cut_room(sipgpu_triples_s &P, hipStream_t s) {
    if (P.cut) return true;
    if (P.no_cut || sipgpu::rt::thread_captures() || sipgpu::rt::capturing(s)) return false;
    auto blocks = [](const std::vector<int> &seg) {
        return (long long)(*std::max_element(seg.begin(), seg.end()) + sipgpu::kTriplesBox - 1) /
               sipgpu::kTriplesBox;
    };
    const long long v = blocks(P.vseg), o = blocks(P.oseg);
    const long long doubles = 6 * (v * o * o + v * v * o) * 8LL * P.nkp * 128;
    P.no_cut = doubles > P.pa_doubles + P.pb_doubles ||
               hipMalloc(&P.cut, (size_t)doubles * sizeof(double)) != hipSuccess;
    if (P.no_cut) {
        P.cut = nullptr;
        (void)hipGetLastError();
    }
    return !P.no_cut;
}

// sipgpu_triples_create after its checks.  Host memory that runs out throws.
int create(int nv, const int *v_seg, int no, const int *o_seg, const double *const *T,
           const double *const *V1, const double *const *V2, const double *e_occ,
           const double *e_vir, sipgpu_triples_t *plan) {
    auto P = std::make_unique<sipgpu_triples_s>();
    P->nv = nv;
    P->no = no;
    P->vseg.assign(v_seg, v_seg + nv);
    P->oseg.assign(o_seg, o_seg + no);
    for (int x : P->vseg)
        if (x < 1) return fail(SIPGPU_EARG, "triples: segment extents must be positive");
    for (int x : P->oseg)
        if (x < 1) return fail(SIPGPU_EARG, "triples: segment extents must be positive");
    for (int x : P->vseg) P->kd += x;
    for (int x : P->oseg) P->kl += x;
    // K in k-pairs of 8, at least four (the kernel's loads run two ahead and
    // cross one permutation boundary at a time)
    P->nkp = std::max(4, (P->kd + P->kl + 7) / 8);
    P->nvb = (P->kd + sipgpu::kTriplesBox - 1) / sipgpu::kTriplesBox;
    P->nob = (P->kl + sipgpu::kTriplesBox - 1) / sipgpu::kTriplesBox;
    const long long nvb = P->nvb, nob = P->nob;
    const long long per_set = 8LL * P->nkp * 128;
    P->pa_doubles = nvb * nob * nob * per_set;
    P->pb_doubles = nvb * nvb * nob * per_set;
    const long long pairs = ((nvb + 1) / 2) * ((nob + 1) / 2);
    P->slots = 64 * pairs * pairs * pairs;
    const long long vmax = max_seg_blocks(P->vseg), omax = max_seg_blocks(P->oseg);
    const long long max_tuple_boxes = vmax * vmax * vmax * omax * omax * omax;

    const size_t nT = (size_t)nv * nv * no * no, nV1 = (size_t)nv * nv * nv * no,
                 nV2 = (size_t)no * nv * no * no;
    for (size_t i = 0; i < nT; ++i)
        if (!T[i]) return fail(SIPGPU_EARG, "triples: null T block");
    for (size_t i = 0; i < nV1; ++i)
        if (!V1[i]) return fail(SIPGPU_EARG, "triples: null V1 block");
    for (size_t i = 0; i < nV2; ++i)
        if (!V2[i]) return fail(SIPGPU_EARG, "triples: null V2 block");

    auto no_memory = [&]() {
        (void)hipGetLastError();
        return fail(SIPGPU_ENOMEM, "triples: device memory for the packed operands");
    };
    hipError_t e = hipMalloc(&P->PA, (size_t)P->pa_doubles * sizeof(double));
    if (e == hipSuccess) e = hipMalloc(&P->PB, (size_t)P->pb_doubles * sizeof(double));
    if (e == hipSuccess) e = hipMalloc(&P->partial, (size_t)P->slots * sizeof(double));
    if (e == hipSuccess) e = hipMalloc(&P->sums, (size_t)sipgpu::kTriplesSums * sizeof(double));
    if (e == hipSuccess)
        e = hipMalloc(&P->tuple_partial, (size_t)max_tuple_boxes * sizeof(double));
    if (e != hipSuccess) return no_memory();
    // built once the device holds a partial per slot: a class (24 bytes) and its
    // items (4 bytes a box, 64 at most) take up to an eleventh of its slots'
    // partials (6 arrangements of 64)
    if (pairs * (pairs + 1) * (pairs + 2) / 6 >= 1LL << 26) // items hold class * 64
        return fail(SIPGPU_ESIZE, "triples: too many super-box classes");
    sipgpu::rt::triples_boxes(P->nvb, P->nob, P->boxes);

    // tables: super-box classes, then int arrays, then pointer tables (16-byte aligned)
    std::vector<int> vseg_of(P->kd), oseg_of(P->kl), vstart(nv), ostart(no);
    for (int s = 0, g = 0; s < nv; g += P->vseg[s], ++s) {
        vstart[s] = g;
        for (int q = 0; q < P->vseg[s]; ++q) vseg_of[g + q] = s;
    }
    for (int s = 0, g = 0; s < no; g += P->oseg[s], ++s) {
        ostart[s] = g;
        for (int q = 0; q < P->oseg[s]; ++q) oseg_of[g + q] = s;
    }
    // (the two long lists are uploaded from where they are)
    auto up16 = [](size_t v) { return (v + 15) & ~(size_t)15; };
    const size_t orbit_bytes = P->boxes.orbits.size() * sizeof(TriplesOrbit),
                 item_bytes = P->boxes.items.size() * sizeof(unsigned);
    const size_t o_orbits = 0, o_items = up16(orbit_bytes), o_img = up16(o_items + item_bytes);
    std::vector<unsigned char> img;
    auto put = [&](const void *p, size_t bytes) {
        const size_t at = up16(img.size());
        img.resize(at + bytes);
        std::memcpy(img.data() + at, p, bytes);
        return o_img + at;
    };
    const size_t o_vext = put(P->vseg.data(), nv * sizeof(int));
    const size_t o_oext = put(P->oseg.data(), no * sizeof(int));
    const size_t o_vso = put(vseg_of.data(), vseg_of.size() * sizeof(int));
    const size_t o_oso = put(oseg_of.data(), oseg_of.size() * sizeof(int));
    const size_t o_vst = put(vstart.data(), nv * sizeof(int));
    const size_t o_ost = put(ostart.data(), no * sizeof(int));
    const size_t o_T = put(T, nT * sizeof(double *));
    const size_t o_V1 = put(V1, nV1 * sizeof(double *));
    const size_t o_V2 = put(V2, nV2 * sizeof(double *));
    e = hipMalloc(&P->tables, o_img + img.size());
    auto upload = [&](size_t at, const void *p, size_t bytes) {
        if (e == hipSuccess)
            e = hipMemcpy(static_cast<unsigned char *>(P->tables) + at, p, bytes,
                          hipMemcpyHostToDevice);
    };
    upload(o_orbits, P->boxes.orbits.data(), orbit_bytes);
    upload(o_items, P->boxes.items.data(), item_bytes);
    upload(o_img, img.data(), img.size());
    if (e != hipSuccess) return no_memory();
    const unsigned char *base = static_cast<const unsigned char *>(P->tables);
    P->d_orbits = reinterpret_cast<const TriplesOrbit *>(base + o_orbits);
    P->d_items = reinterpret_cast<const unsigned *>(base + o_items);
    P->d_vext = reinterpret_cast<const int *>(base + o_vext);
    P->d_oext = reinterpret_cast<const int *>(base + o_oext);
    P->d_vseg_of = reinterpret_cast<const int *>(base + o_vso);
    P->d_oseg_of = reinterpret_cast<const int *>(base + o_oso);
    P->d_vseg_start = reinterpret_cast<const int *>(base + o_vst);
    P->d_oseg_start = reinterpret_cast<const int *>(base + o_ost);
    P->d_T = reinterpret_cast<const double *const *>(base + o_T);
    P->d_V1 = reinterpret_cast<const double *const *>(base + o_V1);
    P->d_V2 = reinterpret_cast<const double *const *>(base + o_V2);
    P->e_occ = e_occ;
    P->e_vir = e_vir;
    *plan = P.release();
    return 0;
}

} // namespace

extern "C" {

int sipgpu_triples_create(int nv, const int *v_seg, int no, const int *o_seg,
                          const double *const *T, const double *const *V1,
                          const double *const *V2, const double *e_occ, const double *e_vir,
                          sipgpu_triples_t *plan) {
    if (int rc = sipgpu::rt::refuse_in_capture("planning the triples")) return rc;
    if (nv < 1 || no < 1 || !v_seg || !o_seg || !T || !V1 || !V2 || !e_occ || !e_vir || !plan)
        return fail(SIPGPU_EARG, "triples: bad arguments");
    if (int rc = sipgpu::rt::ensure_ready()) return rc;
    try {
        return create(nv, v_seg, no, o_seg, T, V1, V2, e_occ, e_vir, plan);
    } catch (const std::exception &) { // std::bad_alloc, std::length_error
        return fail(SIPGPU_ENOMEM, "triples: host memory for the plan");
    }
}

int sipgpu_triples_destroy(sipgpu_triples_t P) {
    if (int rc = sipgpu::rt::refuse_in_capture("freeing the triples")) return rc;
    if (!P) return fail(SIPGPU_EARG, "null triples plan");
    SIPGPU_HIP_TRY(hipDeviceSynchronize());
    delete P;
    return 0;
}

int sipgpu_triples_info(sipgpu_triples_t P, long long *slots, double *flops_per_box,
                        size_t *panel_bytes) {
    if (!P) return fail(SIPGPU_EARG, "null triples plan");
    if (slots) *slots = P->slots;
    // the MFMA work a box issues: six 128 x 128 tiles over the padded K
    if (flops_per_box) *flops_per_box = 6.0 * 2.0 * 128.0 * 128.0 * (8.0 * P->nkp);
    if (panel_bytes) *panel_bytes = (size_t)(P->pa_doubles + P->pb_doubles) * sizeof(double);
    return 0;
}

int sipgpu_triples_pack(sipgpu_triples_t P, sipgpu_stream_t s) {
    if (!P) return fail(SIPGPU_EARG, "null triples plan");
    const hipStream_t hs = sipgpu::rt::stream_of(s);
    for (int side = 0; side < 2; ++side) {
        sipgpu::TriplesPackArgs a{};
        a.out = side == 0 ? P->PA : P->PB;
        a.total = side == 0 ? P->pa_doubles : P->pb_doubles;
        a.side = side;
        a.nkp = P->nkp;
        a.kd = P->kd;
        a.kl = P->kl;
        a.n1 = side == 0 ? P->nob : P->nvb;
        a.n2 = P->nob;
        a.nv = P->nv;
        a.no = P->no;
        a.vext = P->d_vext;
        a.oext = P->d_oext;
        a.vseg_of = P->d_vseg_of;
        a.oseg_of = P->d_oseg_of;
        a.vseg_start = P->d_vseg_start;
        a.oseg_start = P->d_oseg_start;
        a.T = P->d_T;
        a.V1 = P->d_V1;
        a.V2 = P->d_V2;
        SIPGPU_HIP_TRY(sipgpu::launch_triples_pack(a, hs));
    }
    // partials of slots no run has computed count as zero
    SIPGPU_HIP_TRY(sipgpu::launch_block_op(sipgpu::kOpFill, P->partial, nullptr, P->slots, 0.0, hs));
    P->packed = true;
    return 0;
}

namespace {

sipgpu::TriplesArgs box_args(const sipgpu_triples_s &P) {
    sipgpu::TriplesArgs a{};
    a.PA = P.PA;
    a.PB = P.PB;
    a.nkp = P.nkp;
    a.nvb = P.nvb;
    a.nob = P.nob;
    a.kd = P.kd;
    a.kl = P.kl;
    a.super_v = P.boxes.super_v;
    a.orbits = P.d_orbits;
    a.items = P.d_items;
    for (int d = 0; d < 6; ++d) a.wdims[d] = d < 3 ? P.kd : P.kl;
    a.e_vir = P.e_vir;
    a.e_occ = P.e_occ;
    return a;
}

} // namespace

int sipgpu_triples_run(sipgpu_triples_t P, long long box0, long long nbox, sipgpu_stream_t s) {
    if (!P) return fail(SIPGPU_EARG, "null triples plan");
    if (!P->packed) return fail(SIPGPU_EARG, "triples: pack the operands first");
    if (box0 < 0 || nbox < 0 || box0 > P->slots || nbox > P->slots - box0)
        return fail(SIPGPU_EARG, "triples: box slots outside the plan");
    if (nbox == 0) return 0;
    sipgpu::TriplesArgs a = box_args(*P);
    a.partial = P->partial;
    const hipStream_t hs = sipgpu::rt::stream_of(s);
    // one launch per SIPGPU_TRIPLES_LAUNCH_BOXES slots (about 0.3 s of the
    // whole sum at o = 30, v = 240).  A class that a cut divides is computed
    // by both launches.
    for (long long b = box0; b < box0 + nbox; b += SIPGPU_TRIPLES_LAUNCH_BOXES) {
        a.box0 = b;
        a.nbox = std::min<long long>(SIPGPU_TRIPLES_LAUNCH_BOXES, box0 + nbox - b);
        const sipgpu::rt::TriplesBoxes &B = P->boxes;
        a.nlist = sipgpu::rt::triples_short_range(B, b, a.nbox, a.list);
        const unsigned i0 = (unsigned)class_of(B, b) * 64,
                       i1 = ((unsigned)class_of(B, b + a.nbox - 1) + 1) * 64;
        for (int x = 0; x < 8; ++x) {
            const auto f = B.items.begin() + B.xcd_first[x],
                       l = B.items.begin() + B.xcd_first[x + 1];
            a.begin[x] = (unsigned)(std::lower_bound(f, l, i0) - B.items.begin());
            a.end[x] = (unsigned)(std::lower_bound(f, l, i1) - B.items.begin());
        }
        SIPGPU_HIP_TRY(sipgpu::launch_triples_boxes(a, hs));
    }
    return 0;
}

int sipgpu_triples_energy(sipgpu_triples_t P, double factor, double *out, sipgpu_stream_t s) {
    if (!P || !out) return fail(SIPGPU_EARG, "triples: bad arguments");
    SIPGPU_HIP_TRY(sipgpu::launch_triples_reduce(P->partial, P->slots, P->sums, factor, out,
                                                 sipgpu::rt::stream_of(s)));
    return 0;
}

int sipgpu_triples_tuple(sipgpu_triples_t P, const int *tuple, double factor, double *w_out,
                         double *out, sipgpu_stream_t s) {
    if (!P || !tuple || !out) return fail(SIPGPU_EARG, "triples: bad arguments");
    if (!P->packed) return fail(SIPGPU_EARG, "triples: pack the operands first");
    sipgpu::TriplesArgs a = box_args(*P);
    a.tuple_mode = 1;
    a.partial = P->tuple_partial;
    a.wout = w_out;
    long long boxes = 0;
    if (int rc = sipgpu::rt::triples_tuple_boxes(P->vseg, P->oseg, tuple, false, a, boxes)) return rc;
    const hipStream_t hs = sipgpu::rt::stream_of(s);
    // Segments that begin inside 5-blocks touch one more each: panels cut from the
    // tuple's own start save those boxes for a pass over its sets (segments of 17,
    // 18, 17, 14 | 13, 14, tuple (1,1,1,1,1,1): 4096 boxes, or 1728).
    sipgpu::TriplesArgs own = a;
    long long own_boxes = 0;
    if (sipgpu::rt::triples_tuple_boxes(P->vseg, P->oseg, tuple, true, own, own_boxes) == 0 &&
        own_boxes < boxes && cut_room(*P, hs)) {
        a = own;
        boxes = own_boxes;
        a.PA = a.PB = P->cut;
        SIPGPU_HIP_TRY(sipgpu::launch_triples_cut(a, P->PA, P->PB, P->cut, hs));
    }
    SIPGPU_HIP_TRY(sipgpu::launch_triples_boxes(a, hs));
    SIPGPU_HIP_TRY(sipgpu::launch_triples_reduce(P->tuple_partial, boxes, P->sums, factor, out, hs));
    return 0;
}

} // extern "C"
