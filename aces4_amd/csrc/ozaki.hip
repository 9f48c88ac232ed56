// ozaki.hip -- split-precision contraction: FP64 products emulated exactly
// with INT8 MFMA (Ozaki scheme II, integer/CRT form).
//
// For D(m, n) = sum_k A(k, m) B(k, n) (A = the left operand, B = the right,
// read through the contraction's offset tables):
//   1. every row m of A (column n of B) gets a power-of-two scale so that
//      A_int = rint(A * 2^sA_m) is an integer with |A_int| <= 2^(P-1);
//   2. the integer product C = sum_k A_int B_int is computed modulo N
//      pairwise-coprime moduli p_i <= 255, one INT8 GEMM each, with exact
//      INT32 accumulation (|residue| <= 127, so K * 127^2 < 2^31);
//   3. C is recovered exactly from its residues (explicit CRT, 128-bit
//      integers) and D = C * 2^-(sA_m + sB_n), rounded once to FP64.
// The only rounding is step 1 (relative 2^-P per element); P follows from N
// and the largest K so that |C| <= M/4, M = prod p_i.  Inputs must be finite.
//
// Kernels, in launch order: exponent fill; row/column maxima -> exponents;
// FP64 -> residue panels (the operand permutation is applied here, once per
// block, through 64 x 64 LDS tiles read along whichever index is adjacent in
// memory); the INT8 GEMM per modulus over each task's virtual K (16-byte
// chunks of the pairs' panels, so K is padded per pair to 16 only), whose
// epilogue reduces the tile to t_i = (C mod p_i) u_i mod p_i; and the
// reconstruction, which walks each result block in its memory order.
#include "kernels.h"
#include "ozaki.h"

#include <climits>

namespace sipgpu {

namespace {

typedef int int32x4 __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(1))) int8_t gi8_t;

__global__ void fill_int_kernel(int *p, int n, int v) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        p[i] = v;
}

// Zeroes the kOzZero bytes at the start of each plane (16 lanes x 16 bytes).
__global__ void zero_heads_kernel(int8_t *planes, long long plane_bytes, int nplanes) {
    static_assert(kOzZero == 256, "16 lanes of 16 bytes per plane");
    const int p = blockIdx.x * 4 + (threadIdx.x >> 4);
    if (p < nplanes)
        *reinterpret_cast<int4 *>(planes + p * plane_bytes + (threadIdx.x & 15) * 16) =
            int4{0, 0, 0, 0};
}

// Rows [x0, x0 + 32) x k [k0, k0 + 128) of block b: each thread loads 16
// values along the index that is adjacent in memory (32 lanes on 32
// consecutive rows, or 128 on consecutive k); entries outside the block read
// as 0.  Thread t holds (row, k) = (t % 32, t / 32 + 8 j) when rows are
// adjacent, else (t / 128 + 2 j, t % 128).  Places outside the block load its
// last element's instead, so that nothing branches and all table entries,
// then all values, are in flight together.
struct SubTile {
    double v[16];
};

__device__ __forceinline__ void fetch_subtile(const OzBlock &b, const int32_t *tab, int x0, int k0,
                                              int tid, SubTile &t) {
    typedef const __attribute__((address_space(1))) double gdouble_t;
    gdouble_t *data = (gdouble_t *)b.data;
    const bool xf = b.xfast;
    // this thread's index along the adjacent side, and its 16 along the other
    const int fast = xf ? x0 + (tid & 31) : k0 + (tid & 127);
    const int slow = xf ? k0 + (tid >> 5) : x0 + (tid >> 7), step = xf ? 8 : 2;
    const int nfast = xf ? b.X : b.K, nslow = xf ? b.K : b.X;
    const int32_t *ftab = tab + (xf ? b.xtab : b.ktab), *stab = tab + (xf ? b.ktab : b.xtab);
    const int off = ftab[min(fast, nfast - 1)];
    int at[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) at[j] = stab[min(slow + step * j, nslow - 1)] + off;
    double v[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) v[j] = data[at[j]];
#pragma unroll
    for (int j = 0; j < 16; ++j) t.v[j] = fast < nfast && slow + step * j < nslow ? v[j] : 0.0;
}

__device__ __forceinline__ void store_subtile(const OzBlock &b, int tid, const SubTile &t,
                                              double (*S)[kOzTileK + 1]) {
    if (b.xfast) {
#pragma unroll
        for (int j = 0; j < 16; ++j) S[tid & 31][(tid >> 5) + 8 * j] = t.v[j];
    } else {
#pragma unroll
        for (int j = 0; j < 16; ++j) S[(tid >> 7) + 2 * j][tid & 127] = t.v[j];
    }
}

// One workgroup per 32-row tile of a block: max |value| of each row over
// the block's K, as a binary exponent folded into the row's component with
// atomicMax (order-independent, so the result is deterministic).  Maxima
// stay in registers across the K sweep; one LDS reduction per tile folds them
// per row.  Bound by the reads: the full ring batch (0.32 GB) in 80 us, four
// workgroups per CU with 16 loads a thread in flight; 128 us with a branch at
// every load.
__global__ __launch_bounds__(256, 4) void row_exponent_kernel(OzConvArgs a, const OzConvTile *items,
                                                           int nitems) {
    __shared__ double part[kOzTileX][129];
    const int tid = threadIdx.x;
    for (int it = blockIdx.x; it < nitems; it += gridDim.x) {
        const OzConvTile w = items[it];
        const OzBlock b = a.blocks[w.block];
        double mx[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) mx[j] = 0.0;
#pragma unroll 1
        for (int k0 = 0; k0 < b.K; k0 += kOzTileK) {
            SubTile t;
            fetch_subtile(b, a.tab, w.x0, k0, tid, t);
#pragma unroll
            for (int j = 0; j < 16; ++j) mx[j] = fmax(mx[j], fabs(t.v[j]));
        }
        // rows adjacent: thread holds row tid%32 for 16 k; else 16 rows
        __syncthreads();
        if (b.xfast) {
            double m = 0.0;
#pragma unroll
            for (int j = 0; j < 16; ++j) m = fmax(m, mx[j]);
            part[tid & 31][tid >> 5] = m;
        } else {
#pragma unroll
            for (int j = 0; j < 16; ++j) part[(tid >> 7) + 2 * j][tid & 127] = mx[j];
        }
        __syncthreads();
        if (tid < kOzTileX) {
            const int cols = b.xfast ? 8 : 128;
            double m = 0.0;
            for (int c = 0; c < cols; ++c) m = fmax(m, part[tid][c]);
            const int x = w.x0 + tid;
            if (x < b.X && m > 0.0) {
                int e;
                frexp(m, &e); // m = f * 2^e, f in [0.5, 1)
                atomicMax(&a.expo[b.exp_off + x], e);
            }
        }
    }
}

// t_i = (v mod p) u mod p in [0, p) of an INT32 accumulator |v| < 2^31:
// v = h 2^17 + l with l in [0, 2^17), so h c17 + l + p 2^17 (c17 = 2^17 mod
// p) is congruent to v, positive and below 2^26; two Barrett steps with
// bar = floor(2^32 / p) (each leaves r in [0, 2p)) and the multiplication
// by u (< p) finish it in 32-bit integer arithmetic.
__device__ __forceinline__ uint32_t crt_digit(int v, int p, int c17, int u, uint32_t bar) {
    const uint32_t t = (uint32_t)((v >> 17) * c17 + (v & 0x1ffff)) + ((uint32_t)p << 17);
    uint32_t c = t - __umulhi(t, bar) * (uint32_t)p;
    if (c >= (uint32_t)p) c -= p;
    uint32_t tt = c * (uint32_t)u;
    tt -= __umulhi(tt, bar) * (uint32_t)p;
    if (tt >= (uint32_t)p) tt -= p;
    return tt;
}

// Persistent workgroups over 32 x 128 conversion tiles: the next tile's
// values are loaded into registers while the current one (transposed
// through LDS) is converted to balanced residues (|r| <= 127) for every
// modulus and written to the block's panel in each modulus plane, the 16-byte
// pieces of 16 rows next to each other (a unit, 256 bytes).  Panel bytes for k
// in [K, Kp) are written as zeros.
//
// A residue costs two four-byte dot products, an FP32 quotient and one 24-bit
// multiply-add (FP32 and 24-bit products run at full rate, the high half of a
// 32-bit product at a quarter of it): the full ring batch (40 million operand
// elements, 14 moduli, 0.9 GB) takes 225 us; panels of rows instead of units
// 297, and with Barrett reduction of three limbs and a branch at every load 406.
__global__ __launch_bounds__(256, 4) void to_residues_kernel(OzConvArgs a) {
    __shared__ double S[kOzTileX][kOzTileK + 1];
    const int tid = threadIdx.x;
    int it = blockIdx.x;
    if (it >= a.nitems) return;
    SubTile next;
    OzConvTile w = a.items[it];
    OzBlock b = a.blocks[w.block];
    fetch_subtile(b, a.tab, w.x0, w.k0, tid, next);
    for (; it < a.nitems; it += gridDim.x) {
        __syncthreads(); // the previous tile's LDS reads are done
        store_subtile(b, tid, next, S);
        __syncthreads();
        const OzConvTile cw = w;
        const OzBlock cb = b;
        const int nit = it + gridDim.x;
        if (nit < a.nitems) {
            w = a.items[nit];
            b = a.blocks[w.block];
            fetch_subtile(b, a.tab, w.x0, w.k0, tid, next);
        }
        const int xx = tid & 31, kc = (tid >> 5) * 16; // 16 lanes: the 256 bytes of a unit
        const int x = cw.x0 + xx, k = cw.k0 + kc;
        if (x >= cb.X || k >= cb.Kp) continue;
        const int e = a.expo[cb.exp_off + x];
        const int shift = e == INT_MIN ? 0 : (a.c.P - 1) - e;
        // each scaled value, rounded to an integer V (|V| <= 2^51; the sum with
        // 1.5 2^52 rounds to nearest even and leaves V in the low bits), as seven
        // digits base 256 in [-128, 127]: the bytes of V + 128 (1 + 256 + ..
        // + 256^5), the six low ones less 128
        int lo[16], hi[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const double v = e == INT_MIN ? 0.0 : ldexp(S[xx][kc + j], shift);
            const unsigned long long digits =
                (unsigned long long)__double_as_longlong(v + 0x1.8p52) +
                (0x0000808080808080ull - 0x4338000000000000ull);
            lo[j] = (int)((uint32_t)digits ^ 0x80808080u);
            hi[j] = (int)((uint32_t)(digits >> 32) ^ 0x00008080u);
        }
        const int row = cb.row0 + x;
        int8_t *dst = a.planes + cb.panel_off + (long long)(row >> 4) * cb.Kp * kPanelRows +
                      (k / kOzChunk) * (kPanelRows * kOzChunk) + (row & 15) * kOzChunk;
        for (int i = 0; i < a.c.n; ++i) {
            const int c0 = a.c.d0[i], c1 = a.c.d1[i], np = -a.c.p[i];
            const float rp = a.c.rpf[i];
            uint32_t word[4];
#pragma unroll
            for (int j = 0; j < 16; j += 4) {
                uint32_t res[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    // t = digits . (256^j mod p), |t| < 2^17, congruent to V; as the
                    // low bits of the float 1.5 2^23 + t, since 0x4b400000 is 1.5 2^23
                    const int t = __builtin_amdgcn_sdot4(
                        hi[j + q], c1,
                        __builtin_amdgcn_sdot4(lo[j + q], c0, 0x4b400000, false), false);
                    // round(t / p) in the low bits: the quotient is at least 1/510 from
                    // a half (p = 254: or on it, and either neighbour will do), its
                    // error below 2^-13, so |t - p round(t / p)| <= 127
                    const float f = __fmaf_rn(__int_as_float(t) - 0x1.8p23f, rp, 0x1.8p23f);
                    // the two 0x4b400000 leave the low byte as it is
                    res[q] = (uint32_t)(t + __mul24(__float_as_int(f), np));
                }
                word[j >> 2] = __builtin_amdgcn_perm(res[1], res[0], 0x0c0c0400u) |
                               __builtin_amdgcn_perm(res[3], res[2], 0x04000c0cu);
            }
            *reinterpret_cast<int32x4 *>(dst + (long long)i * a.plane_bytes) =
                int32x4{(int)word[0], (int)word[1], (int)word[2], (int)word[3]};
        }
    }
}

// INT8 GEMM over residue panels, a tile of one modulus per entry of the list.  Workgroup tile
// BM x BN (4 waves, 2 x 2, each (BM/2) x (BN/2)); the task's virtual K runs
// in stages of 128 bytes = 8 chunks, double-buffered in LDS; loads run two
// stages ahead through two register sets (16 bytes per lane each): the
// loads of stage s + 2 are in flight while stage s is multiplied, and
// stage s + 1 is written to the other buffer after it.  LDS rows hold 8 chunk
// slots, chunk c of row r in slot c ^ (r & 7), so both the stores (one wave
// = 8 whole rows) and the fragment reads (16 rows x 4 chunks) spread over
// all banks.  Rows past the task's M / N read row M-1 /
// N-1 and are never stored; chunks past the pairs' K read the plane's zero
// bytes.  MFMA v_mfma_i32_16x16x64_i8: lane l holds row l%16, bytes
// 16*(l/16) .. +15 of a 64-byte k step; accumulator register r of lane l is
// C(4*(l/16) + r, l%16).
template <int BM, int BN, int WM, int WN, int MINB>
__global__ __launch_bounds__(64 * WM * WN, MINB) void gemm_i8_kernel(OzGemmArgs a) {
    constexpr int NT = 64 * WM * WN; // threads
    constexpr int TM = BM / WM, TN = BN / WN, FM = TM / 16, FN = TN / 16;
    constexpr int KS = kOzStage, CH = kOzStageChunks;
    // 8-row load instructions per wave per stage
    constexpr int IA = BM / (8 * WM * WN), IB = BN / (8 * WM * WN);
    static_assert(CH == 8 && KS == 128, "a stage is 8 chunks of 16 bytes");
    static_assert(IA * 8 * WM * WN == BM && IB * 8 * WM * WN == BN && TM % 16 == 0 &&
                      TN % 16 == 0, "tile shape");
    constexpr int kWin = 512; // chunk entries per LDS window (64 stages)
    static_assert(kWin % (2 * CH) == 0, "a window holds whole pairs of stages");
    __shared__ __attribute__((aligned(1024))) int8_t As[2][BM * KS];
    __shared__ __attribute__((aligned(1024))) int8_t Bs[2][BN * KS];
    __shared__ __attribute__((aligned(16))) OzChunkRef Es[kWin];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave % WM, wn = wave / WM;
    const int li = lane & 15, lk = lane >> 4;
    const int g = (lane & 7) ^ (lane >> 3); // chunk of the stage this lane loads
    for (int t = blockIdx.x; t < a.ntiles; t += gridDim.x) {
        const OzUnit unit = a.units[t];
        if (unit.task < 0) continue;
        const OzTask task = a.tasks[unit.task];
        int mt, nt, mod;
        oz_unit(unit, task.M, BM, mt, nt, mod);
        const int p = a.c.p[mod], u = a.c.u[mod], c17 = a.c.c17[mod];
        const uint32_t bar = a.c.bar[mod];
        gi8_t *plane = (gi8_t *)(a.planes + (long long)mod * a.plane_bytes);
        const int m0 = mt * BM, n0 = nt * BN;
        int ra[IA], rb[IB];
#pragma unroll
        for (int i = 0; i < IA; ++i) ra[i] = min(m0 + 8 * (wave * IA + i) + (lane >> 3), task.M - 1);
#pragma unroll
        for (int i = 0; i < IB; ++i) rb[i] = min(n0 + 8 * (wave * IB + i) + (lane >> 3), task.N - 1);

        int32x4 acc[FM][FN];
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) acc[i][j] = int32x4{0, 0, 0, 0};

        const OzChunkRef *ch = a.chunks + task.chunk0;
        const int nst = task.nchunks / CH; // even: the planner pads to pairs of stages
        // two register sets: the loads of stage s + 2 are issued while stage s
        // is multiplied and land in LDS after stage s + 1
        int32x4 xa[IA], xb[IB], ya[IA], yb[IB];
        auto put = [&](int buf, const int32x4 *va, const int32x4 *vb) {
#pragma unroll
            for (int i = 0; i < IA; ++i)
                *reinterpret_cast<int32x4 *>(&As[buf][(wave * IA + i) * 1024 + lane * 16]) = va[i];
#pragma unroll
            for (int i = 0; i < IB; ++i)
                *reinterpret_cast<int32x4 *>(&Bs[buf][(wave * IB + i) * 1024 + lane * 16]) = vb[i];
        };
        // B fragments in groups of FH (the 64 x 128 wave tiles read them in
        // two halves, which keeps the second prefetch register set in budget)
        constexpr int FH = FN > 4 ? 4 : FN;
        auto compute = [&](int buf) {
            const int8_t *sa = As[buf], *sb = Bs[buf];
#pragma unroll
            for (int ks = 0; ks < KS / 64; ++ks) {
                const int slot = ((ks * 4 + lk) ^ (li & 7)) * 16;
                int32x4 fa[FM];
#pragma unroll
                for (int i = 0; i < FM; ++i)
                    fa[i] = *reinterpret_cast<const int32x4 *>(sa + (wm * TM + i * 16 + li) * KS + slot);
#pragma unroll
                for (int j0 = 0; j0 < FN; j0 += FH) {
                    int32x4 fb[FH];
#pragma unroll
                    for (int j = 0; j < FH; ++j)
                        fb[j] = *reinterpret_cast<const int32x4 *>(
                            sb + (wn * TN + (j0 + j) * 16 + li) * KS + slot);
#pragma unroll
                    for (int i = 0; i < FM; ++i)
#pragma unroll
                        for (int j = 0; j < FH; ++j)
                            acc[i][j0 + j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(
                                fa[i], fb[j], acc[i][j0 + j], 0, 0, 0);
                }
            }
        };

        // loads are unconditional (stage indices are clamped, so the last
        // stages are fetched again) so the staged registers need no merge
        // copies, which would wait on them
        // Chunk entries are staged in LDS, a window of kWin entries at a time,
        // and each lane reads its own with ds_read: waiting for an entry then
        // waits on the LDS counter only, never on the operand loads in flight.
        struct Sel {
            uint32_t a, b;
            int stride;
        };
        auto load_window = [&](int st0) {
            __syncthreads(); // nobody still reads the previous window
            const int c0 = st0 * CH, n = min(kWin, task.nchunks - c0);
            for (int i = tid; i < n; i += NT)
                *reinterpret_cast<int32x4 *>(&Es[i]) =
                    *reinterpret_cast<const int32x4 *>(&ch[c0 + i]);
            __syncthreads();
        };
        auto entry = [&](int st) {
            const int idx = (min(st, nst - 1) * CH + g) % kWin;
            const OzChunkRef e = Es[idx];
            return Sel{e.a, e.b, e.stride};
        };
        auto fetch2 = [&](const Sel &e, int32x4 *va, int32x4 *vb) {
#pragma unroll
            for (int i = 0; i < IA; ++i)
                va[i] = *reinterpret_cast<const __attribute__((address_space(1))) int32x4 *>(
                    plane + oz_row(e.a, ra[i], e.stride));
#pragma unroll
            for (int i = 0; i < IB; ++i)
                vb[i] = *reinterpret_cast<const __attribute__((address_space(1))) int32x4 *>(
                    plane + oz_row(e.b, rb[i], e.stride));
        };
        load_window(0);
        fetch2(entry(0), xa, xb);
        fetch2(entry(1), ya, yb);
        put(0, xa, xb);
        __syncthreads();
        for (int s = 0; s < nst; s += 2) {
            // entries of stages s + 2, s + 3 are in the next window (a window
            // holds an even number of stages, so they share one)
            if (s + 2 < nst && ((s + 2) * CH) % kWin == 0) load_window(s + 2);
            // stage s from buffer 0; stage s + 1 waits in (ya, yb)
            fetch2(entry(s + 2), xa, xb);
            __builtin_amdgcn_sched_barrier(0); // keep the loads ahead of the MFMAs
            compute(0);
            put(1, ya, yb);
            __syncthreads();
            // stage s + 1 from buffer 1; stage s + 2 waits in (xa, xb)
            fetch2(entry(s + 3), ya, yb);
            __builtin_amdgcn_sched_barrier(0);
            compute(1);
            put(0, xa, xb); // after the last pair of stages this writes a copy nothing reads
            __syncthreads();
        }

        // t = (C mod p) u mod p of the tile into this modulus' result plane,
        // in the task's element order
        uint8_t *res = a.res_planes + (long long)mod * a.res_plane_bytes + task.res_off;
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                const int n = n0 + wn * TN + j * 16 + li;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int m = m0 + wm * TM + i * 16 + 4 * lk + r;
                    if (m < task.M && n < task.N) {
                        const uint32_t tt = crt_digit(acc[i][j][r], p, c17, u, bar);
                        const long long idx = task.nfast ? (long long)m * task.N + n
                                                         : (long long)n * task.M + m;
                        res[idx] = (uint8_t)tt;
                    }
                }
            }
    }
}

// The INT8 GEMM with a 256 x 256 workgroup tile, eight waves of 64 x 128.
//
// Operands go from memory into LDS directly (buffer_load_dwordx4 .. lds: no
// registers, no LDS store instructions), 64 bytes of virtual K a stage, through
// four stage buffers of 32 KiB: the loads of stage s + 3 are issued while
// stage s is multiplied.  A wave waits for its own loads of stage s (those of
// the two stages behind it stay in flight), then one barrier says that
// everybody's have landed and that nobody still reads stage s - 1, whose
// buffer the new loads fill.  A unit of a buffer is 16 rows x 64 bytes in MFMA
// operand order (lane l: row l % 16, bytes 16 (l / 16) ..), so both the loads
// and the fragment reads are linear in the lane.  The buffers are separate
// variables: the compiler then knows that a read of one does not depend on the
// loads into the others.  A lane holds the chunk entries of the next four
// stages.
//
// The product is formed transposed (B as the MFMA's row operand), so a lane's
// four accumulators are four consecutive columns of one row and leave as one
// 4-byte store.
//
// Bound by the card's power: the full ring batch (2.55e12 INT8 operations in
// 14 moduli) takes 1.27 ms, 2.0e15 operations a second, what a library's large
// INT8 product reaches here.  Operands staged through registers, with one LDS
// latency every eight MFMAs, took 0.32 ms longer.
__global__ __launch_bounds__(512, 1) void gemm_i8_wide_kernel(OzGemmArgs a) {
    constexpr int BT = kOzBigTile, FM = 4, FN = 8; // wave grid 4 x 2
    constexpr int KS = 64, CH = KS / kOzChunk, kUnit = 16 * KS;
    __shared__ __attribute__((aligned(1024))) int8_t S0[2 * BT * KS], S1[2 * BT * KS],
        S2[2 * BT * KS], S3[2 * BT * KS];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave & 3, wn = wave >> 2;
    const int li = lane & 15, lk = lane >> 4;
    const OzUnit unit = a.units[blockIdx.x];
    if (unit.task < 0) return;
    const OzTask task = a.tasks[unit.task];
    int mt, nt, mod;
    oz_unit(unit, task.M, BT, mt, nt, mod);
    const int p = a.c.p[mod], u = a.c.u[mod], c17 = a.c.c17[mod];
    const uint32_t bar = a.c.bar[mod];
    // (buffer loads: the compiler takes a global load into LDS for a flat access
    // and then waits for all loads at once)
    const __amdgpu_buffer_rsrc_t plane = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<int8_t *>(a.planes) + (long long)mod * a.plane_bytes, 0,
        (int)(uint32_t)a.plane_bytes, 0x00020000);

    const int m0 = mt * BT, n0 = nt * BT;
    // this wave loads four of the stage's 32 units: waves 0-3 those of A,
    // waves 4-7 those of B; a lane's rows, clamped into the panel
    const bool side_b = wave >= 4;
    int row[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = ((wave & 3) * 4 + i) * 16 + li;
        row[i] = side_b ? min(n0 + r, task.N - 1) : min(m0 + r, task.M - 1);
    }
    const int nst = task.nchunks / CH; // a multiple of four (the planner pads)
    // this lane's chunk entry (unit, stride) of stage st on its wave's side (past
    // the last one: that one's again, whose loads nothing reads)
    typedef int32_t int32x2 __attribute__((ext_vector_type(2)));
    typedef const __attribute__((address_space(1))) int32x2 gentry_t;
    gentry_t *ch = (gentry_t *)(a.chunks + task.chunk0 + lk) + (side_b ? 1 : 0);
    auto entry = [&](int st) { return ch[min(st, nst - 1) * CH * 2]; };
    auto fill = [&](int8_t *S, const int32x2 &e) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                plane, (__attribute__((address_space(3))) void *)(S + (wave * 4 + i) * kUnit), 16,
                (int)oz_row(e[0], row[i], e[1]), 0, 0, 0);
    };
    int32x4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = int32x4{0, 0, 0, 0};
    // stage st from `cur`; the loads of stage st + 3, whose entry is in `e`, go
    // to `next`, then e becomes the entry of stage st + 7
    auto stage = [&](const int8_t *cur, int8_t *next, int32x2 &e, int st) {
        // vmcnt <= 10, lgkmcnt 0: this wave's loads of stage st have landed (each
        // stage issues four and an entry; those of two stages are behind them)
        // and its reads of stage st - 1 are done.  (A fence would wait for all
        // loads; the empty statements keep the compiler from moving any.)
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0x007a);
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        fill(next, e);
        asm volatile("" ::: "memory");
        e = entry(st + 7);
        __builtin_amdgcn_sched_barrier(0);
        const int8_t *sa = cur + wm * FM * kUnit + lane * 16;
        const int8_t *sb = cur + BT * KS + wn * FN * kUnit + lane * 16;
        // all fragments of the stage at once, the first MFMAs' first: one LDS
        // latency a stage instead of one every eight MFMAs
        int32x4 fa[FM], fb[FN];
        fb[0] = *reinterpret_cast<const int32x4 *>(sb);
#pragma unroll
        for (int i = 0; i < FM; ++i) fa[i] = *reinterpret_cast<const int32x4 *>(sa + i * kUnit);
#pragma unroll
        for (int j = 1; j < FN; ++j) fb[j] = *reinterpret_cast<const int32x4 *>(sb + j * kUnit);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int i = 0; i < FM; ++i)
                acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fb[j], fa[i], acc[i][j], 0, 0, 0);
    };
    if (nst > 0) {
        // issued in the order of the loop's stages: its waits count loads
        const int32x2 e0 = entry(0), e1 = entry(1), e2 = entry(2);
        int32x2 e6 = entry(6), e3, e4, e5;
        asm volatile("" ::: "memory");
        fill(S0, e0);
        asm volatile("" ::: "memory");
        e3 = entry(3);
        asm volatile("" ::: "memory");
        fill(S1, e1);
        asm volatile("" ::: "memory");
        e4 = entry(4);
        asm volatile("" ::: "memory");
        fill(S2, e2);
        asm volatile("" ::: "memory");
        e5 = entry(5);
        asm volatile("" ::: "memory");
        for (int st = 0; st < nst; st += 4) {
            stage(S0, S3, e3, st);
            stage(S1, S0, e4, st + 1);
            stage(S2, S1, e5, st + 2);
            stage(S3, S2, e6, st + 3);
        }
    }
    // t = (C mod p) u mod p of the tile into this modulus' result plane, in
    // the task's element order
    uint8_t *res = a.res_planes + (long long)mod * a.res_plane_bytes + task.res_off;
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        const int m = m0 + (wm * FM + i) * 16 + li;
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            const int n = n0 + (wn * FN + j) * 16 + 4 * lk;
            uint32_t word = 0;
#pragma unroll
            for (int r = 0; r < 4; ++r) word |= crt_digit(acc[i][j][r], p, c17, u, bar) << (8 * r);
            if (m >= task.M || n >= task.N) continue;
            if (task.nfast && n + 4 <= task.N) {
                __builtin_memcpy(res + (long long)m * task.N + n, &word, 4);
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (n + r < task.N)
                        res[task.nfast ? (long long)m * task.N + n + r
                                       : (long long)(n + r) * task.M + m] = (uint8_t)(word >> (8 * r));
            }
        }
    }
    __builtin_amdgcn_s_waitcnt(0); // no load into LDS outlives the workgroup
}

// 128-bit helpers on {low, high} 64-bit halves (two's complement, mod 2^128).
struct U128 {
    unsigned long long lo, hi;
};

// A signed 128-bit value correctly rounded to FP64.
__device__ __forceinline__ double to_double(U128 v) {
    const bool neg = (long long)v.hi < 0;
    if (neg) {
        v.lo = ~v.lo + 1;
        v.hi = ~v.hi + (v.lo == 0 ? 1ull : 0ull);
    }
    double d;
    if (v.hi == 0) {
        d = (double)v.lo;
    } else {
        // top 64 bits, with a sticky bit for everything below them: one
        // rounding of the 64-bit value is then the correct rounding of v
        const int sh = __clzll((long long)v.hi);
        unsigned long long top = sh ? (v.hi << sh) | (v.lo >> (64 - sh)) : v.hi;
        const unsigned long long rest = sh ? v.lo << sh : v.lo;
        if (rest) top |= 1ull;
        d = ldexp((double)top, 64 - sh);
    }
    return neg ? -d : d;
}

// One workgroup per kOzRecChunk result elements of a task, four to a thread,
// walked in the task's element order (the destination's memory order where it
// has a unit-stride index).  Explicit CRT: with t_i = r_i u_i mod p_i,
// C = sum_i t_i (M/p_i) - q M for q = round(sum_i t_i / p_i); |C| <= M/4 keeps
// that sum a quarter away from the rounding boundary, so 1/p_i in 16 bits
// (0.03 off over 14 moduli) gives q.  C is formed exactly modulo 2^128
// (|C| < 2^111), rounded once to FP64 and scaled by the operands' powers of
// two.
//
// Both sums are byte dot products: the planes' words of four elements are
// transposed into words of four moduli's t_i each, q takes the place after
// the last modulus, and byte b of every M/p_i and of -M gives the sum S_b
// (< 2^20) of weight 256^b.
// Bound by instruction issue: 64 dot products an element, about as many more
// to put the sums together and to find the destination.  A full ring batch
// (15 blocks of up to 450 x 900, 20 million elements, 14 moduli, 0.6 GB): 189
// us; with 128-bit products per modulus (64-bit integer and FP64 units) 282.
// One round of 1024 elements a workgroup, all planes loaded at once: a batch
// of 4800 elements takes 7 us instead of 20, which were load latencies.
template <int NW>
__global__ __launch_bounds__(256) void reconstruct_kernel(OzRecArgs a) {
    typedef double f64x2 __attribute__((ext_vector_type(2), aligned(8)));
    typedef __attribute__((address_space(1))) double gdouble_t;
    typedef __attribute__((address_space(1))) f64x2 gf64x2_t;
    const OzRecItem w = a.items[blockIdx.x / kOzRecPer];
    const OzTask task = a.tasks[w.task];
    const int first = w.e0 + (int)(blockIdx.x % kOzRecPer) * kOzRecChunk;
    const int e1 = min(first + kOzRecChunk, task.M * task.N);
    const int e0 = first + 4 * (int)threadIdx.x;
    if (e0 >= e1) return;
    // one 32-bit load per plane for the thread's four elements, all before any
    // is used (task regions start 16-byte aligned and planes end 16 bytes past
    // the last region, so the word never leaves the plane)
    const uint8_t *res = a.res_planes + task.res_off + e0;
    uint32_t w4[4 * NW];
#pragma unroll
    for (int i = 0; i < 4 * NW; ++i)
        w4[i] = i < 4 * (NW - 1) || i < a.c.n
                    ? *reinterpret_cast<const uint32_t *>(res + (long long)i * a.res_plane_bytes)
                    : 0u;
    // destinations and exponents (past the end the last element's again, which
    // is not stored)
    gdouble_t *dst[4];
    int beta[4], ea[4], eb[4];
    {
        const int fast = task.nfast ? task.N : task.M;
        int slow = e0 / fast, quick = e0 - slow * fast;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int m = task.nfast ? slow : quick, n = task.nfast ? quick : slow;
            ea[q] = a.expo[task.expA + m];
            eb[q] = a.expo[task.expB + n];
            dst[q] = (gdouble_t *)oz_dest(task, a.subs, a.tab, m, n, beta[q]);
            if (e0 + q + 1 < e1 && ++quick == fast) quick = 0, ++slow;
        }
    }
    // byte k of t[q][g]: t_i of element q, modulus i = 4 g + k
    uint32_t t[4][NW];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        uint32_t s0 = 1u << 15, s1 = 0u;
#pragma unroll
        for (int g = 0; g < NW; ++g) {
            const uint32_t sel = 0x0c0c0400u + 0x0101u * q;
            t[q][g] = __builtin_amdgcn_perm(w4[4 * g + 1], w4[4 * g], sel) |
                      __builtin_amdgcn_perm(w4[4 * g + 3], w4[4 * g + 2], sel) << 16;
            s0 = __builtin_amdgcn_udot4(t[q][g], a.c.inv[0][g], s0, false);
            s1 = __builtin_amdgcn_udot4(t[q][g], a.c.inv[1][g], s1, false);
        }
        t[q][NW - 1] |= ((s0 + (s1 << 8)) >> 16) << (8 * (a.c.n & 3));
    }
    uint32_t pr[4][8]; // S_2k + 256 S_2k+1, weight 2^16k
#pragma unroll
    for (int k = 0; k < 8; ++k) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            uint32_t even = 0u, odd = 0u;
            // M < 2^112: bytes 14 and 15 are those of -M alone
#pragma unroll
            for (int g = k < 7 ? 0 : NW - 1; g < NW; ++g) {
                even = __builtin_amdgcn_udot4(t[q][g], a.c.crt[2 * k][g], even, false);
                odd = __builtin_amdgcn_udot4(t[q][g], a.c.crt[2 * k + 1][g], odd, false);
            }
            pr[q][k] = even + (odd << 8);
        }
        __builtin_amdgcn_sched_barrier(0); // the constants in turn: all at once spill
    }
    double v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        auto two = [](uint32_t x, uint32_t y) {
            return (unsigned long long)x + ((unsigned long long)y << 16);
        };
        const unsigned long long low = two(pr[q][0], pr[q][1]), mid = two(pr[q][2], pr[q][3]);
        U128 C{low + (mid << 32),
               two(pr[q][4], pr[q][5]) + (two(pr[q][6], pr[q][7]) << 32) + (mid >> 32)};
        C.hi += C.lo < low ? 1ull : 0ull;
        v[q] = 0.0;
        if (ea[q] != INT_MIN && eb[q] != INT_MIN)
            v[q] = ldexp(to_double(C), -((a.c.P - 1) - ea[q] + ((a.c.P - 1) - eb[q])));
    }
    if (e0 + 4 <= e1 && dst[1] == dst[0] + 1 && dst[2] == dst[0] + 2 && dst[3] == dst[0] + 3 &&
        beta[0] == beta[1] && beta[0] == beta[2] && beta[0] == beta[3]) {
        gf64x2_t *p = (gf64x2_t *)dst[0];
        f64x2 x = {v[0], v[1]}, y = {v[2], v[3]};
        if (beta[0]) x += p[0], y += p[1];
        p[0] = x, p[1] = y;
    } else {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (e0 + q >= e1) break;
            *dst[q] = beta[q] ? v[q] + *dst[q] : v[q];
        }
    }
}

unsigned grid_for(long long items, long long cap) {
    return (unsigned)(items < cap ? items : cap);
}

} // namespace

hipError_t oz_fill_int(int *p, int n, int v, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(fill_int_kernel, dim3(grid_for((n + 255) / 256, 4096)), dim3(256), 0, s, p,
                       n, v);
    return hipGetLastError();
}

hipError_t oz_zero_heads(int8_t *planes, long long plane_bytes, int nplanes, hipStream_t s) {
    if (nplanes <= 0) return hipSuccess;
    hipLaunchKernelGGL(zero_heads_kernel, dim3((nplanes + 3) / 4), dim3(64), 0, s, planes,
                       plane_bytes, nplanes);
    return hipGetLastError();
}

hipError_t oz_row_exponents(const OzConvArgs &a, const OzConvTile *row_items, int nrow_items,
                            hipStream_t s) {
    if (nrow_items <= 0) return hipSuccess;
    hipLaunchKernelGGL(row_exponent_kernel, dim3(grid_for(nrow_items, 65535)), dim3(256), 0, s, a,
                       row_items, nrow_items);
    return hipGetLastError();
}

hipError_t oz_to_residues(const OzConvArgs &a, hipStream_t s) {
    if (a.nitems <= 0) return hipSuccess;
    hipLaunchKernelGGL(to_residues_kernel, dim3(grid_for(a.nitems, 4 * 256)), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t oz_gemm(const OzGemmArgs &a, hipStream_t s) {
    if (a.ntiles <= 0) return hipSuccess;
    if (a.tile == kOzBigTile) return oz_gemm_big(a, s);
    if (a.tile == kOzWideTile) {
        gemm_i8_wide_kernel<<<dim3(a.ntiles), 512, 0, s>>>(a);
        return hipGetLastError();
    }
    hipLaunchKernelGGL((gemm_i8_kernel<kOzBM, kOzBN, 2, 2, 2>), dim3(grid_for(a.ntiles, kOzMaxGrid)),
                       dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t oz_reconstruct(const OzRecArgs &a, hipStream_t s) {
    if (a.nitems <= 0) return hipSuccess;
    const dim3 grid(a.nitems * kOzRecPer);
    const int words = a.c.n / 4 + 1; // of four: the moduli and q
    if (words > 4) return hipErrorInvalidValue;
    if (words == 4)
        hipLaunchKernelGGL(reconstruct_kernel<4>, grid, dim3(256), 0, s, a);
    else if (words == 3)
        hipLaunchKernelGGL(reconstruct_kernel<3>, grid, dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL(reconstruct_kernel<2>, grid, dim3(256), 0, s, a);
    return hipGetLastError();
}

} // namespace sipgpu
