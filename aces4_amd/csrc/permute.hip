// permute.hip -- the permute super-instruction on gfx950.
//
// Semantics: tensor_block_copy_ of the reference (tensor_dil_omp.F90:438-660):
// out-of-place N-d transpose of a dense column-major block, old dim i going
// to new position dim_transp[i].  Bit-exact (pure data movement).
//
// Design.  After canonicalisation (plan_permute: extent-1 dims dropped, dims
// that stay adjacent merged) the block is viewed as a 2-D array (u, v):
//   u = the leading input dims (contiguous in the input, never the output's
//       fastest dim), v = the other dims in OUTPUT order (so consecutive v are
//       contiguous in the output).
// A 256-thread workgroup moves one TU x TV tile: it reads rows of u with
// consecutive lanes on consecutive input addresses, stages the tile in LDS
// (odd row pitch, so the transposed read is free of bank conflicts), and
// writes columns of v with consecutive lanes on consecutive output
// addresses.  The per-tile u/v offset tables are decoded once per tile into
// LDS, so the per-element cost is two LDS reads.  When the input's fastest
// dim is also the output's fastest ("row mode") no transpose is needed and
// the tile is copied straight through registers.
#include <algorithm>
#include <cstdint>

#include "kernels.h"
#include "plan.h"

namespace sipgpu {

namespace {

constexpr int kPermThreads = 256;
// Tiles of at most 2048 elements, u at most 32 wide: on 2-D to 6-D transposes
// (64^4 reversal, 40^4, 20^6, 120^3, 30^5) they beat 4096-element tiles on
// every shape, since more workgroups per CU keep more loads in flight (64^4 6.3
// against 4.7 TB/s).
constexpr int kPermItems = 8;              // elements per thread (at most)
constexpr int kPermMaxTV = 1024;
constexpr int kPermMaxTU = 32;             // transpose mode only
constexpr int64_t kLargeElems = 1 << 25;   // input and output fill the 256 MB cache twice
constexpr int kXcds = 8;                   // workgroup b runs on XCD b % 8

// Dynamic LDS of a launch: the staged tile (tile_cap doubles; none in row
// mode), then the tile's v input and output offsets (tv_cap ints each) and
// its u output offsets (kPermMaxTU ints).  Sized to the largest tile of the
// launch, so small tiles leave room for more workgroups per CU.
__host__ __device__ constexpr size_t perm_lds_bytes(int tile_cap, int tv_cap) {
    return (size_t)tile_cap * sizeof(double) + (size_t)(2 * tv_cap + kPermMaxTU) * sizeof(int);
}

template <bool STREAM>
__device__ __forceinline__ void put(double v, double *p) {
    if (STREAM)
        __builtin_nontemporal_store(v, p);
    else
        *p = v;
}

// Tile of workgroup `blk` of the permute `a` (at most kPermItems * kPermThreads
// elements), staged through the workgroup's LDS.
template <bool STREAM>
__device__ __forceinline__ void permute_tile(const PermArgs &a, int blk, double *lds,
                                             int tile_cap, int tv_cap) {
    double *tile = lds;
    int *sh_inV = reinterpret_cast<int *>(lds + tile_cap);
    int *sh_outV = sh_inV + tv_cap, *sh_outU = sh_outV + tv_cap;
    // the patch (workgroups of one XCD) and the tile in it
    const int r = (int)fastdiv(blk, a.round), q = blk - r * (int)a.round.d;
    const int at = r * kXcds + ((q - a.turn) & (kXcds - 1)), in_patch = q >> 3;
    const int pv = (int)fastdiv(at, a.patchesU), pu = at - pv * (int)a.patchesU.d;
    const int iv = (int)fastdiv(in_patch, a.patchU), iu = in_patch - iv * (int)a.patchU.d;
    const int bu = pu * (int)a.patchU.d + iu;
    const int bv = pv * (int)fastdiv(a.patch.d, a.patchU) + iv;
    if (bu >= a.tilesU || bv >= a.tilesV) return;
    const int u0 = bu * a.TU, v0 = bv * a.TV;
    const int tu = min(a.TU, a.sizeU - u0);
    const int tv = min(a.TV, a.sizeV - v0);
    const int tid = threadIdx.x;

    // Decode the tile's v offsets (input and output) and u output offsets.
    for (int i = tid; i < tv; i += kPermThreads) {
        int v = v0 + i, oin = 0, oout = 0;
        for (int d = 0; d < a.nV; ++d) {
            const int q = (int)fastdiv(v, a.extV[d]);
            const int r = v - q * (int)a.extV[d].d;
            oin += r * a.sinV[d];
            oout += r * a.soutV[d];
            v = q;
        }
        sh_inV[i] = oin;
        sh_outV[i] = oout;
    }
    if (!a.row_mode) {
        for (int i = tid; i < tu; i += kPermThreads) {
            int u = u0 + i, oout = 0;
            for (int d = 0; d < a.nU; ++d) {
                const int q = (int)fastdiv(u, a.extU[d]);
                oout += (u - q * (int)a.extU[d].d) * a.soutU[d];
                u = q;
            }
            sh_outU[i] = oout;
        }
    }
    __syncthreads();

    const int n = tu * tv;
    const double *__restrict__ in = a.in;
    double *__restrict__ out = a.out;
    double val[kPermItems];
    // Element e = tid + i * kPermThreads of the tile, as (v, u) = (e / tu,
    // e % tu) or (u, v) = (e / tv, e % tv): one division per thread, then
    // the stride kPermThreads is added in mixed radix (no division per item).
    const int qu = kPermThreads / tu, ru = kPermThreads - qu * tu;
    const int vu0 = tid / tu, uu0 = tid - vu0 * tu;
    if (a.row_mode) {
        // u is contiguous in both the input and the output.
        int vv = vu0, uu = uu0;
#pragma unroll
        for (int i = 0; i < kPermItems; ++i) {
            if (tid + i * kPermThreads < n) val[i] = in[u0 + uu + sh_inV[vv]];
            uu += ru;
            vv += qu;
            if (uu >= tu) { uu -= tu; ++vv; }
        }
        vv = vu0;
        uu = uu0;
#pragma unroll
        for (int i = 0; i < kPermItems; ++i) {
            if (tid + i * kPermThreads < n)
                put<STREAM>(val[i], &out[u0 + uu + sh_outV[vv]]);
            uu += ru;
            vv += qu;
            if (uu >= tu) { uu -= tu; ++vv; }
        }
        return;
    }
    const int pitch = a.pitch;
    {
        int vv = vu0, uu = uu0;
#pragma unroll
        for (int i = 0; i < kPermItems; ++i) {
            if (tid + i * kPermThreads < n) val[i] = in[u0 + uu + sh_inV[vv]];
            uu += ru;
            vv += qu;
            if (uu >= tu) { uu -= tu; ++vv; }
        }
        vv = vu0;
        uu = uu0;
#pragma unroll
        for (int i = 0; i < kPermItems; ++i) {
            if (tid + i * kPermThreads < n) tile[vv * pitch + uu] = val[i];
            uu += ru;
            vv += qu;
            if (uu >= tu) { uu -= tu; ++vv; }
        }
    }
    __syncthreads();
    const int qv = kPermThreads / tv, rv = kPermThreads - qv * tv;
    const int uv0 = tid / tv, vv0 = tid - uv0 * tv;
    int uu = uv0, vv = vv0;
#pragma unroll
    for (int i = 0; i < kPermItems; ++i) {
        if (tid + i * kPermThreads < n) val[i] = tile[vv * pitch + uu];
        vv += rv;
        uu += qv;
        if (vv >= tv) { vv -= tv; ++uu; }
    }
    uu = uv0;
    vv = vv0;
#pragma unroll
    for (int i = 0; i < kPermItems; ++i) {
        if (tid + i * kPermThreads < n)
            put<STREAM>(val[i], &out[sh_outU[uu] + sh_outV[vv]]);
        vv += rv;
        uu += qv;
        if (vv >= tv) { vv -= tv; ++uu; }
    }
}

template <bool STREAM>
__global__ __launch_bounds__(kPermThreads) void permute_kernel(PermArgs a, int tile_cap,
                                                               int tv_cap) {
    extern __shared__ double perm_lds[];
    permute_tile<STREAM>(a, blockIdx.x, perm_lds, tile_cap, tv_cap);
}

// Many permutes in one launch: workgroup b runs tile b - first[e] of entry
// e = entry[b] (a table of one int per workgroup, so a workgroup's set-up is
// two dependent loads, not a search).  The entry's arguments are read where
// they are: a local copy, indexed at run time, would be kept in private
// memory, 224 bytes a lane written and read per tile (144 blocks of 30 and 15,
// (3,4,1,2), 20.25 M elements: 127 us so, 84 now, 76 in patches).
__global__ __launch_bounds__(kPermThreads) void permute_batch_kernel(
    const PermArgs *__restrict__ args, const int *__restrict__ first,
    const int *__restrict__ entry, int tile_cap, int tv_cap) {
    extern __shared__ double perm_lds[];
    const int b = blockIdx.x;
    const int e = entry[b];
    const PermArgs &a = args[e];
    if (a.stream)
        permute_tile<true>(a, b - first[e], perm_lds, tile_cap, tv_cap);
    else
        permute_tile<false>(a, b - first[e], perm_lds, tile_cap, tv_cap);
}

// Tile extent for `size` elements with at most `cap` per tile: the count of
// tiles a cap-sized split needs, with the elements spread evenly over them
// (450 splits as 8 x 57, not 7 x 64 + 2).
int even_tile(int64_t size, int64_t cap) {
    const int64_t n = (size + cap - 1) / cap;
    return (int)((size + n - 1) / n);
}

// Sets the tile order to patches of su x sv tiles; the workgroups of one
// permute then number whole rounds of 8 patches, the first on XCD `turn` where
// the permute's first workgroup runs on XCD 0.  A permute of fewer than 8 tiles
// runs them in launch order: its round would be mostly empty workgroups (16384
// blocks of 2 x 3, 28 us against 144 with rounds; 4000 of 10^4, five tiles each,
// as (1,3,2,4) 119 against 163; 1000 of about 21 x 10 x 12 x 9, twelve tiles, 98
// with rounds and 106 without).
void patches(PermArgs &a, int su, int sv, int turn, int64_t &grid) {
    const int64_t nu = (a.tilesU + su - 1) / su, nv = (a.tilesV + sv - 1) / sv;
    a.patch = make_fastdiv((uint32_t)(su * sv));
    a.patchU = make_fastdiv((uint32_t)su);
    a.patchesU = make_fastdiv((uint32_t)nu);
    a.round = make_fastdiv((uint32_t)(kXcds * su * sv));
    const bool rounds = nu * nv * su * sv >= kXcds;
    a.turn = rounds ? turn : 0;
    grid = rounds ? (nu * nv + kXcds - 1) / kXcds * kXcds * su * sv : nu * nv;
}

constexpr int kLine = 16; // doubles

bool on_line(const void *p, int line = kLine) {
    return (reinterpret_cast<uintptr_t>(p) & (line * sizeof(double) - 1)) == 0;
}

// True if every row that a tile reads is whole cache lines: runs of U, which
// start at sums of the input strides of V.
bool whole_lines_in(const PermArgs &a) {
    bool ok = !a.row_mode && a.TU % kLine == 0 && a.sizeU % kLine == 0 && on_line(a.in);
    for (int i = 0; i < a.nV; ++i) ok = ok && a.sinV[i] % kLine == 0;
    return ok;
}

// True if the runs of V in the output (its leading dims as far as they follow
// each other there) are whole lines (or lines of another size), and so every row
// that a tile of a multiple of them writes.
bool whole_runs_out(const PermArgs &a, int line = kLine) {
    bool ok = !a.row_mode && on_line(a.out, line) && a.nV > 0;
    for (int i = 0; i < a.nU; ++i) ok = ok && a.soutU[i] % line == 0;
    int64_t run = 1;
    int d = 0;
    while (d < a.nV && a.soutV[d] == run) run *= a.extV[d++].d;
    for (; d < a.nV; ++d) ok = ok && a.soutV[d] % line == 0;
    return ok && run % line == 0;
}

// The order of a permute's tiles over the XCDs and how it stores.
//
// Rows of a tile that begin or end inside a cache line share it with the
// tile's neighbours, along U for the reads and along V for the writes.  In
// launch order the neighbours run on other XCDs, each with an L2 of its own,
// and the line is fetched (written) twice; patches of 8 x 8 tiles keep both
// neighbours on one XCD at about the same time.  Stores past the caches then
// only fit blocks that the 256 MB cache holds (30^5, 389 MB in all: 86 us
// against 94 stored through it); larger ones store through it, so that the
// halves of a line meet (113 x 97 x 109 x 101 reversed, 1.9 GB: launch order
// 543 us, patches 494, stored through the cache 425; 7001 x 5003 transposed
// 154 -> 142), unless what a tile writes begins and ends at half lines, the 64
// bytes that memory takes (36 x 14 x 18 x 18 x 20 x 16 reversed in part 163 us past
// the cache, 172 through it; 5934 x 6104 transposed 109 and 123; over 96 shapes of
// such halves 0.96, the worst 1.004, but over 30 batches 0.997 and 1.06: whole lines
// there; tiles that end at quarters of a line go either way, 0.9 to 1.3, and stay)
// or is whole rows (row mode: 63 x 82 x 81 x 94 as
// (1,3,4,2) 110 and 128; over 27 such shapes 0.97 of launch order, 1.09 through the
// cache).  Past the cache patches of 16 x 4 tiles are enough (over 96 such shapes
// 0.983 of 16 x 16).  Rows of whole lines on both sides have nothing to share and
// run in launch order with streaming stores (64^4 reversed 56 us, in patches 57).  A
// batch takes smaller patches, since its blocks have few tiles (144 blocks of 30,
// 15: 81 us with 8 x 8, 76 with 4 x 8).
void tile_order(bool large, bool batched, int turn, PermArgs &a, int64_t &grid) {
    const bool out = whole_runs_out(a) && a.TV % kLine == 0, lines = out && whole_lines_in(a);
    const bool halves = whole_runs_out(a, kLine / 2) && a.TV % (kLine / 2) == 0;
    a.stream = (batched ? out : halves) || a.row_mode || !large;
    // at least 64 patches of a single block (8 an XCD), and none in a batch's
    // smallest blocks, whose patches would not fill a round of the XCDs
    const int64_t tiles = (int64_t)a.tilesU * a.tilesV;
    const int64_t in_all = batched ? (tiles < 64 ? 1 : 32)
                                   : std::min<int64_t>(a.stream ? 64 : 256, tiles / 64);
    if (lines || in_all <= 1) return patches(a, 1, 1, turn, grid);
    const int64_t along_u = std::min<int64_t>(batched ? 4 : large ? 16 : 8, in_all);
    const int su = even_tile(a.tilesU, along_u);
    const int sv = even_tile(a.tilesV, std::max<int64_t>(1, in_all / su));
    patches(a, su, sv, turn, grid);
}

// Kernel arguments and workgroup count of one permute (an identity as a
// single contiguous run in row mode).
void fill_args(const PermutePlan &p, const double *in, double *out, PermArgs &a,
               int64_t &grid, bool large, bool batched, int turn) {
    const int tile_elems = kPermItems * kPermThreads;
    a = PermArgs{};
    a.in = in;
    a.out = out;
    if (p.identity) {
        a.nU = 1;
        a.extU[0] = make_fastdiv((uint32_t)p.size);
        a.soutU[0] = 1;
        a.nV = 0;
        a.sizeU = (int)p.size;
        a.sizeV = 1;
        a.row_mode = 1;
        a.TU = even_tile(p.size, tile_elems);
        a.TV = 1;
        a.pitch = a.TU;
        a.tilesU = (a.sizeU + a.TU - 1) / a.TU;
        a.tilesV = 1;
        a.stream = 1;
        patches(a, 1, 1, turn, grid);
        return;
    }
    a.nU = p.nU;
    a.nV = p.nV;
    for (int i = 0; i < p.nU; ++i) {
        a.extU[i] = make_fastdiv((uint32_t)p.ext[i]);
        a.soutU[i] = (int)p.sout[i];
    }
    // Input strides of the canonical dims are their column-major products.
    int64_t sin[kPermMaxDims];
    int64_t acc = 1;
    for (int i = 0; i < p.rank; ++i) { sin[i] = acc; acc *= p.ext[i]; }
    for (int i = 0; i < p.nV; ++i) {
        const int d = p.vdim[i];
        a.extV[i] = make_fastdiv((uint32_t)p.ext[d]);
        a.sinV[i] = (int)sin[d];
        a.soutV[i] = (int)p.sout[d];
    }
    a.sizeU = (int)p.sizeU;
    a.sizeV = (int)p.sizeV;
    a.row_mode = p.row_mode ? 1 : 0;
    a.TU = even_tile(p.sizeU, p.row_mode ? tile_elems : kPermMaxTU);
    a.TV = even_tile(p.sizeV, std::max<int64_t>(1, std::min<int64_t>(tile_elems / a.TU,
                                                                      kPermMaxTV)));
    if (a.TV > kLine && whole_runs_out(a)) a.TV -= a.TV % kLine; // tiles end where lines do
    a.pitch = p.row_mode ? a.TU : (a.TU | 1);
    const int64_t tilesU = (a.sizeU + a.TU - 1) / a.TU;
    const int64_t tilesV = (a.sizeV + a.TV - 1) / a.TV;
    grid = tilesU * tilesV;
    if (grid >= ((int64_t)1 << 31)) return; // refused by the callers
    a.tilesU = (int)tilesU;
    a.tilesV = (int)tilesV;
    tile_order(large, batched, turn, a, grid);
}

} // namespace

int64_t permute_args(const PermutePlan &p, const double *in, double *out, PermArgs &a) {
    int64_t grid = 0;
    fill_args(p, in, out, a, grid, p.size >= kLargeElems, false, 0);
    return grid;
}

hipError_t launch_permute(const PermutePlan &p, const double *in, double *out,
                          hipStream_t stream) {
    if (p.size <= 0) return hipSuccess;
    if (p.identity)
        return hipMemcpyAsync(out, in, (size_t)p.size * sizeof(double),
                              hipMemcpyDeviceToDevice, stream);
    PermArgs a;
    const int64_t grid = permute_args(p, in, out, a);
    if (grid <= 0 || grid >= ((int64_t)1 << 31)) return hipErrorInvalidValue;
    const int tile_cap = a.row_mode ? 0 : a.TV * a.pitch;
    const size_t lds = perm_lds_bytes(tile_cap, a.TV);
    if (a.stream)
        permute_kernel<true><<<(unsigned)grid, kPermThreads, lds, stream>>>(a, tile_cap, a.TV);
    else
        permute_kernel<false><<<(unsigned)grid, kPermThreads, lds, stream>>>(a, tile_cap, a.TV);
    return hipGetLastError();
}

int64_t permute_batch_args(const PermutePlan *plans, const double *const *in,
                           double *const *out, int n, PermArgs *args, int *first,
                           int *tile_cap, int *tv_cap) {
    int64_t total = 0, all = 0;
    int turn = 0;
    for (int e = 0; e < n; ++e) all += plans[e].size;
    *tile_cap = 0;
    *tv_cap = 1;
    for (int e = 0; e < n; ++e) {
        int64_t g = 0;
        if (plans[e].size > 0) {
            const int from = (int)((turn + kXcds - total % kXcds) % kXcds);
            fill_args(plans[e], in[e], out[e], args[e], g, all >= kLargeElems, true, from);
            if (!args[e].row_mode) *tile_cap = std::max(*tile_cap, args[e].TV * args[e].pitch);
            *tv_cap = std::max(*tv_cap, args[e].TV);
            // the next entry's patches go on with the next XCD
            const int64_t row = args[e].patchesU.d, sv = args[e].patch.d / args[e].patchU.d;
            turn = (int)((turn + row * ((args[e].tilesV + sv - 1) / sv)) % kXcds);
        } else {
            args[e] = PermArgs{};
        }
        first[e] = (int)std::min<int64_t>(total, INT32_MAX);
        total += g;
    }
    first[n] = (int)std::min<int64_t>(total, INT32_MAX);
    return total;
}

hipError_t launch_permute_batch(const PermArgs *args, const int *first, const int *entry,
                                int grid, int tile_cap, int tv_cap, hipStream_t stream) {
    if (grid <= 0) return hipSuccess;
    permute_batch_kernel<<<(unsigned)grid, kPermThreads, perm_lds_bytes(tile_cap, tv_cap),
                           stream>>>(args, first, entry, tile_cap, tv_cap);
    return hipGetLastError();
}

} // namespace sipgpu
