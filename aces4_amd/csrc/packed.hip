// packed.hip -- the FP64 contraction on packed operand panels.
//
// For large batches the operand permutations are applied once per block
// instead of once per tile: every operand instance (block + its k / x
// tables) is packed into a panel of X rows (a merged task's instances one
// after another in one panel) by K rounded up to 8, zero filled, and the
// grouped GEMM runs over each task's virtual K -- its pairs' panels one after
// another, 8 k a stage -- with no table lookups in the K loop.  The product is
// scattered into the destination block through its tables, accumulating when
// the task does.
//
// A panel is made of 1 KiB units of 16 rows x 8 k in the operand order of
// v_mfma_f64_16x16x4_f64 (lane l holds A(i = l%16, k = l/16); register r of
// lane l holds C(4r + l/16, l%16)): element (row i, k) sits at 2 (i + 16 (k %
// 4)) + k / 4, so one 16-byte load per lane, 1 KiB contiguous per wave, gives
// a wave its operand for two MFMAs.  Unit (row block, k block) of a panel is
// number row block * (Kp / 8) + k block.
#include "kernels.h"
#include "ozaki.h"

namespace sipgpu {

namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef double f64x2 __attribute__((ext_vector_type(2)));
typedef const __attribute__((address_space(1))) int8_t gi8_t;
typedef const __attribute__((address_space(4))) OzChunkRef cref_t;

// Workgroups over 32 x 128 tiles of operand blocks, each done as two halves
// of 64 k (half the LDS of a whole tile, so twice the workgroups per CU keep
// their loads in flight): read along the index adjacent in memory,
// transposed through LDS, written unit by unit.
__global__ __launch_bounds__(256) void pack_kernel(OzConvArgs a) {
    constexpr int HK = kOzTileK / 2;
    __shared__ __attribute__((aligned(16))) double S[kOzTileX][HK + 2];
    const int tid = threadIdx.x;
    for (int it = blockIdx.x; it < a.nitems; it += gridDim.x) {
        const OzConvTile w = a.items[it];
        const OzBlock b = a.blocks[w.block];
#pragma unroll 1
        for (int half = 0; half < 2; ++half) {
            const int kb = w.k0 + half * HK;
            double v[8];
            if (b.xfast) {
                const int x = w.x0 + (tid & 31);
                const bool xin = x < b.X;
                const int xo = xin ? a.tab[b.xtab + x] : 0;
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int k = kb + (tid >> 5) + 8 * j;
                    v[j] = (xin && k < b.K) ? b.data[a.tab[b.ktab + k] + xo] : 0.0;
                }
            } else {
                const int k = kb + (tid & 63);
                const bool kin = k < b.K;
                const int ko = kin ? a.tab[b.ktab + k] : 0;
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int x = w.x0 + (tid >> 6) + 4 * j;
                    v[j] = (kin && x < b.X) ? b.data[ko + a.tab[b.xtab + x]] : 0.0;
                }
            }
            __syncthreads(); // the previous LDS reads are done
            if (b.xfast) {
#pragma unroll
                for (int j = 0; j < 8; ++j) S[tid & 31][(tid >> 5) + 8 * j] = v[j];
            } else {
#pragma unroll
                for (int j = 0; j < 8; ++j) S[(tid >> 6) + 4 * j][tid & 63] = v[j];
            }
            __syncthreads();
            // 16 bytes (k, k + 4) per thread, rows fastest: 16 rows x 4 k are
            // the 1 KiB of a unit, in address order
            const int nk = b.Kp / kPanelK;
            double *dst = reinterpret_cast<double *>(a.planes + b.panel_off);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int e = j * 256 + tid;
                const int xx = (e & 15) + 16 * ((e >> 9) & 1), kl = (e >> 4) & 3, ku = (e >> 6) & 7;
                const int x = w.x0 + xx, kk = 8 * ku + kl;
                if (x < b.X && kb + kk < b.Kp) {
                    const int row = b.row0 + x;
                    const long long unit = (long long)(row >> 4) * nk + (kb >> 3) + ku;
                    *reinterpret_cast<f64x2 *>(dst + unit * 128 + 2 * ((row & 15) + 16 * kl)) =
                        f64x2{S[xx][kk], S[xx][kk + 4]};
                }
            }
        }
    }
}

// Grouped FP64 GEMM over packed panels.  Workgroup tile BM x BN = 128 x 128
// (4 waves, 2 x 2, each 64 x 64: 16 accumulator fragments) or 64 x 64 (each
// wave 32 x 32: for small batches, whose tiles are cut into K segments:
// a segment's partial sums are a quarter of the bytes).  Operands go from the
// panels straight into registers: no LDS, no barrier, so a wave waits for its
// own loads alone, which run one stage (32 MFMAs of 64 cycles) ahead in a
// second register set.  Chunk entries are wave-uniform and come through the
// scalar cache.  What bounds it is the FP64 matrix rate at the clock that the
// card's power leaves: 4500^3 in 450 x 450 blocks 3.03 ms with the operands
// staged through LDS (matrix units busy 82%), 2.82 so (91%; 93% and 2.06 GHz on
// the block-sparse ladder, 7.31 -> 7.04 ms).  Rows past the task's M / N lie in its last row block or
// repeat it and are never stored.
// SKIP: heed the chunks' k-step counts (a pair's last 8 k may hold four or
// fewer: their second MFMAs would multiply zeros).
template <int BM, int BN, bool SKIP>
__global__ __launch_bounds__(256, 2) void gemm_f64_packed_kernel(OzGemmArgs a) {
    constexpr int WM = 2, WN = 2;
    constexpr int TM = BM / WM, TN = BN / WN, FM = TM / 16, FN = TN / 16;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave % WM, wn = wave / WM;
    const int li = lane & 15, lk = lane >> 4;
    gi8_t *plane = (gi8_t *)a.planes;

    const int u0 = a.wg_first ? a.wg_first[blockIdx.x] : (int)blockIdx.x;
    const int u1 = a.wg_first ? a.wg_first[blockIdx.x + 1] : min((int)blockIdx.x + 1, a.ntiles);
    for (int t = u0; t < u1; ++t) {
        const OzTile tile = a.tiles[t];
        if (tile.task < 0) continue;
        const OzTask task = a.tasks[tile.task];
        const int m0 = tile.mt * BM, n0 = tile.nt * BN;
        // this wave's row blocks of the operands, clamped into the panels
        int ra[FM], rb[FN];
#pragma unroll
        for (int i = 0; i < FM; ++i) ra[i] = (min(m0 + wm * TM + i * 16, task.M - 1)) >> 4;
#pragma unroll
        for (int j = 0; j < FN; ++j) rb[j] = (min(n0 + wn * TN + j * 16, task.N - 1)) >> 4;

        f64x4 acc[FM][FN];
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) acc[i][j] = f64x4{0.0, 0.0, 0.0, 0.0};

        cref_t *ch = (cref_t *)(a.chunks + task.chunk0);
        const int sb = tile.s0, se = tile.s1; // stages of this unit
        f64x2 fa[2][FM], fb[2][FN];
        int steps[2]; // MFMA k-steps of the stage
        // stage s into register set `set` (past the unit's last stage that
        // one again: the loads stay unconditional, nothing reads them)
        auto fetch = [&](int set, int s) {
            const int at = min(s, se - 1);
            const uint32_t ea = ch[at].a, eb = ch[at].b;
            const int stride = ch[at].stride;
            steps[set] = SKIP ? ch[at].aux : 2;
#pragma unroll
            for (int i = 0; i < FM; ++i)
                fa[set][i] = *reinterpret_cast<const __attribute__((address_space(1))) f64x2 *>(
                    plane + ((long long)ea + (long long)ra[i] * stride) * kPanelUnit + lane * 16);
#pragma unroll
            for (int j = 0; j < FN; ++j)
                fb[set][j] = *reinterpret_cast<const __attribute__((address_space(1))) f64x2 *>(
                    plane + ((long long)eb + (long long)rb[j] * stride) * kPanelUnit + lane * 16);
        };
        auto mma = [&](int set) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                if (SKIP && h >= steps[set]) break;
#pragma unroll
                for (int i = 0; i < FM; ++i)
#pragma unroll
                    for (int j = 0; j < FN; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[set][i][h], fb[set][j][h],
                                                                         acc[i][j], 0, 0, 0);
            }
        };
        if (sb < se) {
            fetch(0, sb);
            int s = sb;
            for (; s + 1 < se; s += 2) {
                fetch(1, s + 1);
                mma(0);
                fetch(0, s + 2);
                mma(1);
            }
            if (s < se) mma(0);
        }

        if (tile.part >= 0) {
            // one K segment of a split tile: raw accumulators, register order;
            // elements outside the task (which the fixup skips) are not written
            double *w = a.work + (long long)tile.part * kOzWorkSlot;
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j) {
                    const bool nin = n0 + wn * TN + j * 16 + li < task.N;
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (nin && m0 + wm * TM + i * 16 + 4 * r + lk < task.M)
                            w[(((wave * FM + i) * FN + j) * 4 + r) * 64 + lane] = acc[i][j][r];
                }
            continue;
        }
        // scatter into the destination block(s), 16 elements at a time:
        // their destinations first, then all loads (beta), then the stores,
        // so the loads overlap instead of waiting behind each other's stores
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            const int n = n0 + wn * TN + j * 16 + li;
            const bool nin = n < task.N;
            const int no = (task.rmap < 0 && nin) ? a.tab[task.nD + n] : 0;
            double *p[FM * 4];
            int bt[FM * 4];
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int m = m0 + wm * TM + i * 16 + 4 * r + lk;
                    const int q = i * 4 + r;
                    p[q] = nullptr;
                    bt[q] = 0;
                    if (nin && m < task.M) {
                        if (task.rmap < 0) {
                            p[q] = task.D + a.tab[task.mD + m] + no;
                            bt[q] = task.beta;
                        } else {
                            p[q] = oz_dest(task, a.subs, a.tab, m, n, bt[q]);
                        }
                    }
                }
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (p[i * 4 + r] && bt[i * 4 + r]) acc[i][j][r] += *p[i * 4 + r];
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (p[i * 4 + r]) *p[i * 4 + r] = acc[i][j][r];
        }
    }
}

// Split tiles: one thread per element of a split tile (BM * BN / 256
// workgroups of 256 per tile) sums the tile's segments in segment order --
// the layout the GEMM wrote: element e = (((wave * FM + i) * FN + j) * 4 + r)
// * 64 + lane holds fragment (i, j, r) of that wave and lane -- and stores
// the sum like the GEMM epilogue.  One element per thread keeps thousands of
// the dependent destination lookups in flight.
template <int BM, int BN>
__global__ __launch_bounds__(256) void fixup_f64_kernel(OzGemmArgs a) {
    constexpr int TM = BM / 2, TN = BN / 2, FM = TM / 16, FN = TN / 16;
    constexpr int LFM = FM == 4 ? 2 : 1, LFN = FN == 4 ? 2 : 1; // log2
    static_assert((FM == 4 || FM == 2) && (FN == 4 || FN == 2), "tile shape");
    constexpr int kPer = BM * BN / 256; // workgroups per tile
    const long long nwork = (long long)a.nfix * kPer;
    for (long long w = blockIdx.x; w < nwork; w += gridDim.x) {
        const OzTile f = a.fix[w / kPer];
        const int e = (int)(w % kPer) * 256 + threadIdx.x;
        const int lane = e & 63, r = (e >> 6) & 3, j = (e >> 8) & (FN - 1);
        const int i = (e >> (8 + LFN)) & (FM - 1);
        const int wave = e >> (8 + LFN + LFM), wm = wave & 1, wn = wave >> 1;
        const OzTask task = a.tasks[f.task];
        const int m = f.mt * BM + wm * TM + i * 16 + 4 * r + (lane >> 4);
        const int n = f.nt * BN + wn * TN + j * 16 + (lane & 15);
        if (m >= task.M || n >= task.N) continue;
        const double *w0 = a.work + (long long)f.part * kOzWorkSlot + e;
        // segments summed in order; loaded eight at a time so the loads are
        // in flight together
        double v = 0.0;
        for (int q0 = 0; q0 < f.s0; q0 += 8) {
            double x[8];
#pragma unroll
            for (int q = 0; q < 8; ++q)
                x[q] = q0 + q < f.s0 ? w0[(long long)(q0 + q) * kOzWorkSlot] : 0.0;
#pragma unroll
            for (int q = 0; q < 8; ++q)
                if (q0 + q < f.s0) v = q0 + q == 0 ? x[q] : v + x[q];
        }
        int beta;
        double *p = oz_dest(task, a.subs, a.tab, m, n, beta);
        if (beta) v += *p;
        *p = v;
    }
}

} // namespace

hipError_t oz_fixup_f64(const OzGemmArgs &a, hipStream_t s) {
    if (a.nfix <= 0) return hipSuccess;
    const int edge = a.tile == kOzSmallTile ? kOzSmallTile : kOzBM;
    const long long work = (long long)a.nfix * (edge * edge / 256);
    const dim3 grid((unsigned)(work < 1048576 ? work : 1048576));
    if (a.tile == kOzSmallTile)
        hipLaunchKernelGGL((fixup_f64_kernel<kOzSmallTile, kOzSmallTile>), grid, dim3(256), 0, s,
                           a);
    else
        hipLaunchKernelGGL((fixup_f64_kernel<kOzBM, kOzBN>), grid, dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t oz_pack(const OzConvArgs &a, hipStream_t s) {
    if (a.nitems <= 0) return hipSuccess;
    hipLaunchKernelGGL(pack_kernel, dim3(a.nitems < 65535 ? a.nitems : 65535), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t oz_gemm_f64(const OzGemmArgs &a, hipStream_t s) {
    if (a.ntiles <= 0) return hipSuccess;
    const dim3 grid(a.wg_first ? a.nwg : a.ntiles);
    const bool small = a.tile == kOzSmallTile;
    auto kernel = small ? (a.skip_halves ? gemm_f64_packed_kernel<kOzSmallTile, kOzSmallTile, true>
                                         : gemm_f64_packed_kernel<kOzSmallTile, kOzSmallTile, false>)
                        : (a.skip_halves ? gemm_f64_packed_kernel<kOzBM, kOzBN, true>
                                         : gemm_f64_packed_kernel<kOzBM, kOzBN, false>);
    kernel<<<grid, 256, 0, s>>>(a);
    return hipGetLastError();
}

} // namespace sipgpu
