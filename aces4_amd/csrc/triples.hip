// triples.hip -- the (T) triples energy with W kept on chip.
//
// W(a,b,c,i,j,k) = sum over the 6 permutations P of the pairs (a,i), (b,j),
// (c,k) -- written (x1,y1), (x2,y2), (x3,y3) after permuting -- of
//     sum_d V1(x2,x3,d,y3) T(x1,d,y1,y2)  +  sum_l T(x3,x2,y3,l) V2(l,x1,y2,y1)
// (V2 holds -V), and E += factor * sum (W / D) * W with
// D = e_i + e_j + e_k - e_a - e_b - e_c summed in that order
// (rccsdpt_aaa.sialx:2164-2174, energy_denominator_rhf.F:399-444).
//
// For every P both terms split W's six indices into the same row set
// {x1, y1, y2} and column set {x2, x3, y3}, so a P is one GEMM with
// K = v + o (d, then l).  A workgroup owns a box of W of extent 5 in every
// index (15625 doubles, held in LDS): it runs the six GEMMs of the box
// (125 x 125 tiles, padded to 128) on FP64 MFMA, adds each product into
// the box in P order (the first assigns), then divides, squares and sums
// the box into one partial energy.  W is never written to HBM.
//
// The operands come from two packed panel arrays built once from T, V1 and
// V2: PA over row sets (x, y1, y2) of 5-blocks, PB over column sets
// (x2, x3, y3).  Within a set, rows are x + 5 (y1 + 5 y2) (padded to 128,
// zero rows), and each 16-row block holds its K in MFMA operand order:
// element (row 16 rb + l % 16, k = 8 kp + 4 h + l / 16) sits at
// ((set * 8 + rb) * NKP + kp) * 128 + 2 l + h, so a wave reads the operands
// of two MFMA k-steps with one 16-byte load per lane, 1 KiB contiguous per
// wave.  Every P reads the same two arrays: P only changes which box
// coordinates select the row and column sets.
#include <type_traits>

#include "kernels.h"

namespace sipgpu {

namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef double f64x2 __attribute__((ext_vector_type(2)));

constexpr int kBoxE = kTriplesBox;                 // box extent per index
constexpr int kBoxRows = kBoxE * kBoxE * kBoxE;     // 125 rows / columns per P
constexpr int kBoxElems = kBoxRows * kBoxRows;      // 15625
constexpr int kThreads = 512;
constexpr int kOutside = 1 << 20; // byte offset of a padded row or column: past any box
constexpr int kFinalThreads = 1024;
static_assert(kTriplesSums % kFinalThreads == 0, "the final sum's split");

// the permutations P of (0, 1, 2), in the order W sums them
__constant__ int kPerm[6][3] = {{0, 1, 2}, {0, 2, 1}, {1, 0, 2}, {1, 2, 0}, {2, 0, 1}, {2, 1, 0}};
constexpr int kPermHost[6][3] = {{0, 1, 2}, {0, 2, 1}, {1, 0, 2}, {1, 2, 0}, {2, 0, 1}, {2, 1, 0}};

// box digit strides in LDS: a fastest, then b, c, i, j, k
__device__ __forceinline__ int box_stride(int d) {
    return d == 0 ? 1 : d == 1 ? 5 : d == 2 ? 25 : d == 3 ? 125 : d == 4 ? 625 : 3125;
}

// ---------------------------------------------------------------- pack --

// One thread per panel double; rows and K positions outside the blocks'
// extents are zeros.  Reads gather from the blocks (a one-time pass).
__global__ __launch_bounds__(256) void triples_pack_kernel(TriplesPackArgs a) {
    const long long stride = (long long)gridDim.x * blockDim.x;
    const long long per_set = (long long)8 * a.nkp * 128;
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < a.total;
         e += stride) {
        const long long set = e / per_set;
        const int rem = (int)(e - set * per_set);
        const int rb = rem / (a.nkp * 128);
        const int r2 = rem - rb * (a.nkp * 128);
        const int kp = r2 >> 7;
        const int lh = r2 & 127;
        const int lane = lh >> 1, h = lh & 1;
        const int row = rb * 16 + (lane & 15);
        const int k = kp * 8 + h * 4 + (lane >> 4);
        double v = 0.0;
        if (row < kBoxRows && k < a.kd + a.kl) {
            const int r0 = row % 5, r1 = (row / 5) % 5, r2d = row / 25;
            // set = (s0 * n1 + s1) * n2 + s2 over the set's three 5-block lists
            const int s2 = (int)(set % a.n2);
            const int s1 = (int)((set / a.n2) % a.n1);
            const int s0 = (int)(set / ((long long)a.n2 * a.n1));
            // global indices of the row; the first is virtual, the last
            // occupied, the middle one occupied in PA and virtual in PB
            const int g0 = s0 * kBoxE + r0, g1 = s1 * kBoxE + r1, g2 = s2 * kBoxE + r2d;
            if (g0 < a.kd && g1 < (a.side == 0 ? a.kl : a.kd) && g2 < a.kl) {
                // segment and offset within it
                const int g0s = a.vseg_of[g0], g0o = g0 - a.vseg_start[g0s];
                const int g1s = a.side == 0 ? a.oseg_of[g1] : a.vseg_of[g1];
                const int g1o = g1 - (a.side == 0 ? a.oseg_start[g1s] : a.vseg_start[g1s]);
                const int g2s = a.oseg_of[g2], g2o = g2 - a.oseg_start[g2s];
                if (a.side == 0) {
                    // PA row (x, y1, y2)
                    if (k < a.kd) { // T(x, d, y1, y2)
                        const int ds = a.vseg_of[k], doff = k - a.vseg_start[ds];
                        const double *blk = a.T[((g0s * a.nv + ds) * a.no + g1s) * a.no + g2s];
                        const int e0 = a.vext[g0s], e1 = a.vext[ds], e2 = a.oext[g1s];
                        v = blk[g0o + e0 * (doff + e1 * (g1o + e2 * g2o))];
                    } else { // V2(l, x, y2, y1)
                        const int l = k - a.kd;
                        const int ls = a.oseg_of[l], loff = l - a.oseg_start[ls];
                        const double *blk = a.V2[((ls * a.nv + g0s) * a.no + g2s) * a.no + g1s];
                        const int e0 = a.oext[ls], e1 = a.vext[g0s], e2 = a.oext[g2s];
                        v = blk[loff + e0 * (g0o + e1 * (g2o + e2 * g1o))];
                    }
                } else {
                    // PB column (x2, x3, y3)
                    if (k < a.kd) { // V1(x2, x3, d, y3)
                        const int ds = a.vseg_of[k], doff = k - a.vseg_start[ds];
                        const double *blk = a.V1[((g0s * a.nv + g1s) * a.nv + ds) * a.no + g2s];
                        const int e0 = a.vext[g0s], e1 = a.vext[g1s], e2 = a.vext[ds];
                        v = blk[g0o + e0 * (g1o + e1 * (doff + e2 * g2o))];
                    } else { // T(x3, x2, y3, l)
                        const int l = k - a.kd;
                        const int ls = a.oseg_of[l], loff = l - a.oseg_start[ls];
                        const double *blk = a.T[((g1s * a.nv + g0s) * a.no + g2s) * a.no + ls];
                        const int e0 = a.vext[g1s], e1 = a.vext[g0s], e2 = a.oext[g2s];
                        v = blk[g1o + e0 * (g0o + e1 * (g2o + e2 * loff))];
                    }
                }
            }
        }
        a.out[e] = v;
    }
}

// The sets of a tuple cut from its own start (TriplesArgs::org = lo): blockIdx.y
// = 2 g + side.  One thread per 16 bytes, a row's elements k and k + 4, which
// stand together in the whole ranges' panels as well.
__global__ __launch_bounds__(256) void triples_cut_kernel(TriplesArgs t, const double *PA,
                                                          const double *PB, double *out) {
    const int g = blockIdx.y >> 1, side = blockIdx.y & 1;
    const int p0 = kPerm[g][0], p1 = kPerm[g][1], p2 = kPerm[g][2];
    // the set's three indices: (x1, y1, y2) or (x2, x3, y3)
    const int d0 = side ? p1 : p0, d1 = side ? p2 : 3 + p0, d2 = 3 + (side ? p2 : p1);
    const int n1 = side ? t.nb1[g] : t.na1[g], n2 = side ? t.nb2[g] : t.na2[g];
    const long long total = (long long)t.count[d0] * n1 * n2 * 8 * t.nkp * 64;
    const f64x2 *from = reinterpret_cast<const f64x2 *>(side ? PB : PA);
    f64x2 *to = reinterpret_cast<f64x2 *>(out) +
                (long long)(side ? t.base_b[g] : t.base_a[g]) * 8 * t.nkp * 64;
    for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < total;
         e += (long long)gridDim.x * 256) {
        const int lane = (int)(e & 63);
        const long long u = e >> 6; // (set, row block, k-pair)
        const int kp = (int)(u % t.nkp);
        const long long sr = u / t.nkp;
        const int row = (int)(sr & 7) * 16 + (lane & 15), set = (int)(sr >> 3);
        const int l0 = set / (n1 * n2) * kBoxE + row % kBoxE,
                  l1 = set / n2 % n1 * kBoxE + row / kBoxE % kBoxE,
                  l2 = set % n2 * kBoxE + row / (kBoxE * kBoxE);
        f64x2 v = {0.0, 0.0};
        if (row < kBoxRows && l0 < t.wdims[d0] && l1 < t.wdims[d1] && l2 < t.wdims[d2]) {
            const int g0 = t.lo[d0] + l0, g1 = t.lo[d1] + l1, g2 = t.lo[d2] + l2;
            const long long s = ((long long)(g0 / kBoxE) * (side ? t.nvb : t.nob) + g1 / kBoxE) * t.nob +
                                g2 / kBoxE;
            const int r = g0 % kBoxE + kBoxE * (g1 % kBoxE + kBoxE * (g2 % kBoxE));
            v = from[((s * 8 + (r >> 4)) * t.nkp + kp) * 64 + (r & 15) + (lane & 48)];
        }
        to[e] = v;
    }
}

// ---------------------------------------------------------------- boxes --

// W is unchanged when the pairs (a,i), (b,j), (c,k) are permuted together
// with their indices (its six terms only change places), and so is D: the up
// to six boxes that differ by such a permutation have one energy.  The kernel
// computes it once, on the box whose pairs are in ascending order, and stores
// it for every image: a whole sum runs a sixth of its boxes (o = 30, v = 60,
// segments of 20 and 10: 373,248 slots, 64,824 boxes; this step alone took 133
// -> 25.8 ms).  A slot's value does not depend on which range of slots a call
// covers.
//
// Global mode: item 64 c + q is position q (one bit per index) of class c's
// ascending super-box; the plan lists the items that are boxes (inside the
// index ranges, their pairs ascending) XCD by XCD, the classes dealt to the
// XCDs in turn.  Slots number the 64 boxes of every super-box, the
// arrangements of a class next to each other, so that any range of slots
// holds most images of the boxes it computes.  A range of few boxes comes as a
// list instead, only boxes with an image in it, one to a workgroup over all
// XCDs (one slot 93 us; 177 with its whole class on one XCD).
struct BoxId {
    int p[3];        // the class's super pairs
    long long first; // its first super-box
    int sub[3];      // bit 0: which virtual 5-block of the super-box, bit 1: occupied
};

// the p-th of three values (an array indexed at run time would leave the
// registers)
__device__ __forceinline__ int pick(int x0, int x1, int x2, int p) {
    return p == 0 ? x0 : p == 1 ? x1 : x2;
}

// Slot of the arrangement g of the box's pairs (position t holds pair kPerm[g][t]).
__device__ __forceinline__ long long image_slot(const BoxId &b, int g) {
    const int t0 = kPerm[g][0], t1 = kPerm[g][1], t2 = kPerm[g][2];
    const bool eq01 = b.p[0] == b.p[1], eq12 = b.p[1] == b.p[2];
    // distinct arrangements of the class: by g, by the place of the pair that
    // differs from the other two, or just one
    int rank = g;
    if (eq01 && eq12)
        rank = 0;
    else if (eq01)
        rank = t0 == 2 ? 0 : t1 == 2 ? 1 : 2;
    else if (eq12)
        rank = t0 == 0 ? 0 : t1 == 0 ? 1 : 2;
    const int s0 = pick(b.sub[0], b.sub[1], b.sub[2], t0), s1 = pick(b.sub[0], b.sub[1], b.sub[2], t1), s2 = pick(b.sub[0], b.sub[1], b.sub[2], t2);
    const int q = (s0 & 1) | (s1 & 1) << 1 | (s2 & 1) << 2 | (s0 >> 1) << 3 | (s1 >> 1) << 4 |
                  (s2 >> 1) << 5;
    return (b.first + rank) * 64 + q;
}

// Box coordinates (5-block indices of a, b, c, i, j, k) of work item t.
// Tuple mode: the boxes of one tuple, first index fastest.
template <bool TUPLE>
__device__ __forceinline__ void box_of(const TriplesArgs &a, unsigned t, int (&bc)[6], BoxId &id) {
    if (TUPLE) {
        unsigned q = t;
#pragma unroll
        for (int d = 0; d < 6; ++d) {
            bc[d] = a.first[d] + (int)(q % a.count[d]);
            q /= a.count[d];
        }
        return;
    }
    const unsigned item = a.nlist ? a.list[t] : a.items[t];
    const TriplesOrbit o = a.orbits[item >> 6];
    id.first = o.first;
#pragma unroll
    for (int m = 0; m < 3; ++m) {
        id.p[m] = o.p[m];
        id.sub[m] = ((item >> m) & 1) | ((item >> (3 + m)) & 1) << 1;
        bc[m] = 2 * (o.p[m] % a.super_v) + (id.sub[m] & 1);
        bc[3 + m] = 2 * (o.p[m] / a.super_v) + (id.sub[m] >> 1);
    }
}

// *w += x in LDS, no value returned: the wave does not wait for the sum
// before it goes on with the next product (read, add, write: 21.7 ms a sum of
// o = 30, v = 60, so 20.9 at that time).  Each element is added to once between two
// barriers, so the order of the sums is fixed.
__device__ __forceinline__ void lds_add(double *w, double x) {
    __builtin_amdgcn_ds_atomic_fadd_f64((__attribute__((address_space(3))) double *)w, x);
}

// A barrier that the waves of a workgroup may reach at different places of
// the program, the same number of times each.
__device__ __forceinline__ void group_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// A workgroup runs boxes one after another, each with all six GEMMs and the
// energy partial.  Eight waves in 2 x 4, each a 64 x 32 tile (4 x 2 MFMA
// blocks): two waves per SIMD, so one issues MFMAs while the other waits for
// its operands.  The box fills the LDS, so a CU holds one workgroup and
// nothing else covers its start and end: one workgroup per CU stays and
// fetches its next box's first operands and energies during the present one.
// Adding a product into the box is 16384 LDS operations without a branch: with
// the bounds tested per element, the waits between them and both waves of a
// SIMD adding at once, the sum of o = 30, v = 60 took 24.9 ms; 20.4 now, its
// matrix cores 78% busy by the counters.
template <int REST, bool TUPLE>
__global__ __launch_bounds__(kThreads) void triples_box_kernel(TriplesArgs a) {
    __shared__ double W[kBoxElems + 64]; // 64: where the padded rows and columns go
    __shared__ double eps[6][kBoxE];
    __shared__ int lo[6], hi[6]; // the box's elements that count, per index
    __shared__ double red[kThreads / 64];
    __shared__ double occ[kBoxRows];
    // byte offsets in the box of the product's rows and columns under
    // permutation g: rows by (wave row, lane / 16, block, register), columns
    // by x; past the 125th far outside the box
    __shared__ int rofs[6][2][4][16], cofs[6][128];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave & 1, wn = wave >> 1;
    // this workgroup's work items: item, item + stride, ... < end
    unsigned item, end, stride;
    if (TUPLE || a.nlist) {
        item = blockIdx.x;
        end = TUPLE ? a.end[0] : (unsigned)a.nlist;
        stride = gridDim.x;
    } else {
        const int x = blockIdx.x & 7;
        item = a.begin[x] + (blockIdx.x >> 3);
        end = a.end[x];
        stride = gridDim.x >> 3;
    }
    if (item >= end) return;
    int bc[6]; // the box being loaded
    BoxId id;
    box_of<TUPLE>(a, item, bc, id);

    for (int t = tid; t < 6 * 128; t += kThreads) {
        const int g = t >> 7, x = t & 127;
        const int p0 = kPerm[g][0], p1 = kPerm[g][1], p2 = kPerm[g][2];
        const int d0 = x % kBoxE, d1 = (x / kBoxE) % kBoxE, d2 = x / (kBoxE * kBoxE);
        // row (x1, y1, y2), column (x2, x3, y3)
        const int r = d0 * box_stride(p0) + d1 * box_stride(3 + p0) + d2 * box_stride(3 + p1);
        const int c = d0 * box_stride(p1) + d1 * box_stride(p2) + d2 * box_stride(3 + p2);
        // row x = 64 wm + 16 i + 4 r + lane / 16
        rofs[g][x >> 6][x & 3][(x >> 2) & 15] = x < kBoxRows ? 8 * r : kOutside;
        cofs[g][x] = x < kBoxRows ? 8 * c : kOutside;
    }

    const int nkp = a.nkp;
    // operand pointers of permutation g of the box being loaded: its row set
    // (x1, y1, y2) in PA and column set (x2, x3, y3) in PB, at this wave's
    // first 16-row block
    auto panels = [&](int g, const f64x2 *&pa, const f64x2 *&pb) {
        const int p0 = kPerm[g][0], p1 = kPerm[g][1], p2 = kPerm[g][2];
        const int x1 = pick(bc[0], bc[1], bc[2], p0), y1 = pick(bc[3], bc[4], bc[5], p0);
        const int x2 = pick(bc[0], bc[1], bc[2], p1), y2 = pick(bc[3], bc[4], bc[5], p1);
        const int x3 = pick(bc[0], bc[1], bc[2], p2), y3 = pick(bc[3], bc[4], bc[5], p2);
        const long long rowset = TUPLE ? a.base_a[g] + ((long long)x1 * a.na1[g] + y1) * a.na2[g] + y2
                                       : ((long long)x1 * a.nob + y1) * a.nob + y2;
        const long long colset = TUPLE ? a.base_b[g] + ((long long)x2 * a.nb1[g] + x3) * a.nb2[g] + y3
                                       : ((long long)x2 * a.nvb + x3) * a.nob + y3;
        pa = reinterpret_cast<const f64x2 *>(a.PA) + ((rowset * 8 + wm * 4) * nkp) * 64 + lane;
        pb = reinterpret_cast<const f64x2 *>(a.PB) + ((colset * 8 + wn * 2) * nkp) * 64 + lane;
    };
    // The k-pairs of the six permutations of all boxes form one stream;
    // loads run two k-pairs ahead of the MFMAs through three register sets,
    // across the permutation and box boundaries (nkp >= 4).  Load cursor:
    // k-pair lkp of (lpa, lpb), then the next permutation's (npa, npb).
    f64x2 fa[3][4], fb[3][2];
    const f64x2 *lpa, *lpb, *npa, *npb;
    panels(0, lpa, lpb);
    npa = lpa;
    npb = lpb;
    int lkp = 0;
    auto load_next = [&](int st) {
#pragma unroll
        for (int i = 0; i < 4; ++i) fa[st][i] = lpa[((long long)i * nkp + lkp) * 64];
#pragma unroll
        for (int j = 0; j < 2; ++j) fb[st][j] = lpb[((long long)j * nkp + lkp) * 64];
        if (++lkp == nkp) {
            lkp = 0;
            lpa = npa;
            lpb = npb;
        }
    };
    f64x4 acc[4][2];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = f64x4{0.0, 0.0, 0.0, 0.0};
    auto mma = [&](int st) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[st][i][h], fb[st][j][h],
                                                                     acc[i][j], 0, 0, 0);
    };
    // this thread's share of the box's tables, stored once the previous box's
    // energy is done: an orbital energy (tid < 30), an index's range (tid < 6)
    double my_eps = 0.0;
    int my_lo = 0, my_hi = 0;
    auto fetch_tables = [&]() {
        if (tid < 30) {
            const int d = tid / kBoxE;
            int at = bc[0] * kBoxE + (TUPLE ? a.org[0] : 0);
#pragma unroll
            for (int e = 1; e < 6; ++e)
                at = d == e ? bc[e] * kBoxE + (TUPLE ? a.org[e] : 0) : at;
            const int g = at + tid % kBoxE, total = d < 3 ? a.kd : a.kl;
            my_eps = g < total ? (d < 3 ? a.e_vir : a.e_occ)[g] : 0.0;
        }
        if (tid < 6) {
            // the first element that counts, from the box's own first
            auto from = [&](int e) { return a.lo[e] - (TUPLE ? a.org[e] : 0) - bc[e] * kBoxE; };
            int first = from(0), ext = a.wdims[0];
#pragma unroll
            for (int e = 1; e < 6; ++e) {
                first = tid == e ? from(e) : first;
                ext = tid == e ? a.wdims[e] : ext;
            }
            my_lo = max(0, first);
            my_hi = min(kBoxE, first + ext);
        }
    };
    // add permutation g's product into the box: row (x1, y1, y2), column
    // (x2, x3, y3); the first permutation assigns.  The previous P's adds into
    // the box (the previous box's energy) are complete.
    auto scatter = [&](int g) {
        if (g == 0) {
            if (tid < 30) eps[tid / kBoxE][tid % kBoxE] = my_eps;
            if (tid < 6) {
                lo[tid] = my_lo;
                hi[tid] = my_hi;
            }
        } else if (g == 1 && tid < kBoxRows) {
            // the occupied sums of the box (see the energy below)
            const int i = tid % kBoxE, j = (tid / kBoxE) % kBoxE, k = tid / (kBoxE * kBoxE);
            const bool in = i >= lo[3] && i < hi[3] && j >= lo[4] && j < hi[4] && k >= lo[5] &&
                            k < hi[5];
            occ[tid] = in ? eps[3][i] + eps[4][j] + eps[5][k] : __builtin_nan("");
        }
        int roff[16], coff[2];
#pragma unroll
        for (int q = 0; q < 16; ++q) roff[q] = rofs[g][wm][lane >> 4][q];
#pragma unroll
        for (int j = 0; j < 2; ++j) coff[j] = cofs[g][(wn * 2 + j) * 16 + (lane & 15)];
        // no branch per element: what lies outside goes to 64 spare doubles
        const unsigned outside = 8 * (kBoxElems + lane);
        auto at = [&](int i, int r, int j) {
            const unsigned o = min((unsigned)(roff[4 * i + r] + coff[j]), outside);
            return reinterpret_cast<double *>(reinterpret_cast<char *>(W) + o);
        };
        if (g == 0) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int j = 0; j < 2; ++j) *at(i, r, j) = acc[i][j][r];
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int j = 0; j < 2; ++j) lds_add(at(i, r, j), acc[i][j][r]);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[i][j] = f64x4{0.0, 0.0, 0.0, 0.0};
    };
    // The two waves of a SIMD (w and w + 4) run half a product apart: one adds
    // its product into the box while the other multiplies (together: 21.6 ms,
    // apart: 20.9, before tuples were compiled apart).  Each passes one
    // barrier a product, the first four waves at its end, the others at its
    // middle: behind it every wave has added the product before.
    // (a scalar: the barriers stand under scalar branches)
    const bool late = __builtin_amdgcn_readfirstlane(wave) >= 4;
    const int middle = nkp / 2 / 3 * 3;
    // Permutation g, its first k-pair in register set S: nkp = 3 n + REST
    // k-pairs, so that the sets of three permutations are known here.
    auto product = [&](int g, auto first_set) {
        constexpr int S = decltype(first_set)::value;
        // what is loaded after this permutation: the next one, then the next
        // box (after the last box its own operands, which nothing reads)
        if (g == 5 && item + stride < end) box_of<TUPLE>(a, item + stride, bc, id);
        panels(g == 5 ? 0 : g + 1, npa, npb);
        for (int kp = 0; kp + 3 <= nkp; kp += 3) {
            if (late && kp == middle) group_barrier();
            load_next((S + 2) % 3);
            mma(S);
            load_next(S);
            mma((S + 1) % 3);
            load_next((S + 1) % 3);
            mma((S + 2) % 3);
        }
        if (REST >= 1) {
            load_next((S + 2) % 3);
            mma(S);
        }
        if (REST == 2) {
            load_next(S);
            mma((S + 1) % 3);
        }
        if (!late) group_barrier();
        scatter(g);
    };
    load_next(0);
    load_next(1);
    while (true) {
        fetch_tables();
        for (int g = 0; g < 6; g += 3) {
            product(g, std::integral_constant<int, 0>{});
            product(g + 1, std::integral_constant<int, REST>{});
            product(g + 2, std::integral_constant<int, 2 * REST % 3>{});
        }
        // energy of the box: sum over its elements inside the blocks' extents.
        // Element e = abc + 125 ijk (abc = a + 5 b + 25 c, ijk = i + 5 j + 25 k).
        // D = ((((e_i + e_j) + e_k) - e_a) - e_b) - e_c: the occupied sums of the
        // box's 125 (i, j, k) are formed once (NaN marks an (i, j, k) outside the
        // extents); a thread keeps one abc, its virtual energies in registers,
        // and runs over ijk.
        double sum = 0.0;
        __syncthreads(); // the box is complete
        if (!TUPLE || !a.wout) {
            const int abc = tid & 127;
            const int ea_i = abc % kBoxE, eb_i = (abc / kBoxE) % kBoxE, ec_i = abc / (kBoxE * kBoxE);
            if (abc < kBoxRows && ea_i >= lo[0] && ea_i < hi[0] && eb_i >= lo[1] && eb_i < hi[1] &&
                ec_i >= lo[2] && ec_i < hi[2]) {
                const double ea = eps[0][ea_i], eb = eps[1][eb_i], ec = eps[2][ec_i];
                for (int ijk = tid >> 7; ijk < kBoxRows; ijk += kThreads / 128) {
                    const double o = occ[ijk];
                    if (o != o) continue; // (i, j, k) outside the extents
                    const double w = W[abc + kBoxRows * ijk];
                    const double D = ((o - ea) - eb) - ec;
                    sum += (w / D) * w;
                }
            }
        }
        // tuple mode with W written out: every element's global position
        if (TUPLE && a.wout) box_of<TUPLE>(a, item, bc, id);
        for (int e = TUPLE && a.wout ? tid : kBoxElems; e < kBoxElems; e += kThreads) {
            int q = e, dg[6];
            bool in = true;
#pragma unroll
            for (int d = 0; d < 6; ++d) {
                dg[d] = q % kBoxE;
                q /= kBoxE;
                in = in && dg[d] >= lo[d] && dg[d] < hi[d];
            }
            if (!in) continue;
            const double w = W[e];
            // occupied energies in index order, then the virtual ones subtracted
            const double D = eps[3][dg[3]] + eps[4][dg[4]] + eps[5][dg[5]] - eps[0][dg[0]] -
                             eps[1][dg[1]] - eps[2][dg[2]];
            sum += (w / D) * w;
            long long o = 0;
#pragma unroll
            for (int d = 5; d >= 0; --d)
                o = o * a.wdims[d] + (a.org[d] + bc[d] * kBoxE + dg[d] - a.lo[d]);
            a.wout[o] = w;
        }
        // fixed-order reduction: lanes by xor butterfly, then waves in order
#pragma unroll
        for (int m = 32; m >= 1; m >>= 1) sum += __shfl_xor(sum, m);
        if (lane == 0) red[wave] = sum;
        __syncthreads();
        if (tid == 0) {
            double t = red[0];
            for (int w = 1; w < kThreads / 64; ++w) t += red[w];
            if (TUPLE) {
                a.partial[item] = t;
            } else {
                int unused[6];
                BoxId id;
                box_of<TUPLE>(a, item, unused, id);
                // images that coincide store the same value twice
                for (int g = 0; g < 6; ++g) {
                    const long long slot = image_slot(id, g);
                    if (slot >= a.box0 && slot < a.box0 + a.nbox) a.partial[slot] = t;
                }
            }
        }
        item += stride;
        if (item >= end) break;
        if (TUPLE && a.wout) box_of<TUPLE>(a, item, bc, id);
    }
}

// out[0] += factor * sum of partial[0 .. n) in a fixed order: per-workgroup
// sums of contiguous ranges, then one workgroup over them.
__global__ __launch_bounds__(256) void triples_reduce_kernel(const double *partial, long long n,
                                                             long long chunk, double *sums) {
    __shared__ double red[4];
    const long long b0 = (long long)blockIdx.x * chunk;
    const long long b1 = b0 + chunk < n ? b0 + chunk : n;
    double s = 0.0;
    for (long long e = b0 + threadIdx.x; e < b1; e += blockDim.x) s += partial[e];
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) s += __shfl_xor(s, m);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) sums[blockIdx.x] = ((red[0] + red[1]) + red[2]) + red[3];
}

// One workgroup over the at most kTriplesSums sums: thread t its consecutive
// ones, then a fixed tree.  (One thread over all of them, a chain of 4096
// dependent loads and adds, took 214 us of every energy.)
__global__ __launch_bounds__(kFinalThreads) void triples_final_kernel(const double *sums, int n,
                                                                      double factor,
                                                                      double *out) {
    __shared__ double red[kFinalThreads];
    constexpr int per = kTriplesSums / kFinalThreads;
    const int t = threadIdx.x;
    double s = 0.0;
#pragma unroll
    for (int i = 0; i < per; ++i) s += t * per + i < n ? sums[t * per + i] : 0.0;
    red[t] = s;
    for (int m = kFinalThreads / 2; m >= 1; m >>= 1) {
        __syncthreads();
        if (t < m) red[t] += red[t + m];
    }
    if (t == 0) out[0] += factor * red[0];
}

} // namespace

hipError_t launch_triples_pack(const TriplesPackArgs &a, hipStream_t s) {
    if (a.total <= 0) return hipSuccess;
    const long long blocks = std::min<long long>((a.total + 255) / 256, 65536);
    triples_pack_kernel<<<(int)blocks, 256, 0, s>>>(a);
    return hipGetLastError();
}

hipError_t launch_triples_boxes(const TriplesArgs &a, hipStream_t s) {
    const bool one_list = a.tuple_mode || a.nlist;
    unsigned most = a.nlist; // work items of the longest list
    for (int x = 0; x < (one_list ? 1 : 8); ++x) most = std::max(most, a.end[x] - a.begin[x]);
    if (most == 0) return hipSuccess;
    const unsigned grid = one_list ? std::min(most, kTriplesGroups)
                                   : 8 * std::min(most, kTriplesGroups / 8);
    if (a.nkp < 4) return hipErrorInvalidValue;
    auto kernel = a.nkp % 3 == 0   ? a.tuple_mode ? triples_box_kernel<0, true> : triples_box_kernel<0, false>
                  : a.nkp % 3 == 1 ? a.tuple_mode ? triples_box_kernel<1, true> : triples_box_kernel<1, false>
                  : a.tuple_mode   ? triples_box_kernel<2, true>
                                   : triples_box_kernel<2, false>;
    kernel<<<grid, kThreads, 0, s>>>(a);
    return hipGetLastError();
}

hipError_t launch_triples_cut(const TriplesArgs &t, const double *PA, const double *PB, double *out,
                              hipStream_t s) {
    // enough workgroups for the largest of the twelve set arrays
    long long most = 0;
    for (int g = 0; g < 6; ++g) {
        const long long a = (long long)t.count[kPermHost[g][0]] * t.na1[g] * t.na2[g];
        const long long b = (long long)t.count[kPermHost[g][1]] * t.nb1[g] * t.nb2[g];
        most = std::max(most, std::max(a, b));
    }
    const long long blocks = (most * 8 * t.nkp * 64 + 255) / 256;
    triples_cut_kernel<<<dim3((unsigned)std::min<long long>(blocks, 4096), 12), 256, 0, s>>>(t, PA, PB,
                                                                                            out);
    return hipGetLastError();
}

hipError_t launch_triples_reduce(const double *partial, long long n, double *sums, double factor,
                                 double *out, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    const long long chunk = (n + kTriplesSums - 1) / kTriplesSums;
    const int blocks = (int)((n + chunk - 1) / chunk);
    triples_reduce_kernel<<<blocks, 256, 0, s>>>(partial, n, chunk, sums);
    triples_final_kernel<<<1, kFinalThreads, 0, s>>>(sums, blocks, factor, out);
    return hipGetLastError();
}

} // namespace sipgpu
