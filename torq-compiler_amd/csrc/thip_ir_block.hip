// gfx950 kernel of a whole inverted-residual block: the pointwise convolution that widens the channels, the 3 x 3 depthwise
// convolution, the pointwise one that narrows them again, and the residual add behind it, as one launch.
#include "thip_ir_depthwise.h"
#include "thip_kernels_common.h"

#include <utility>

namespace thip {

// The packed requant tails only (the planner takes no other record into a block).
template <typename F>
__device__ __forceinline__ void withPackedRequant(const WideRequant &w, F &&f) {
    if (w.packShift <= 0) f(std::integral_constant<int, 4>{});
    else f(std::integral_constant<int, 5>{});
}

// f(0) .. f(n - 1), at most as many as the sequence holds, each argument a constant of its own.
template <int... R, typename F>
__device__ __forceinline__ void firstOf(std::integer_sequence<int, R...>, int n, F &&f) {
    (void)((R < n && (f(std::integral_constant<int, R>{}), true)) && ...);
}

// Output rows of a lane, and tiles of 32 input pixels of a wave: what the registers hold (two waves a SIMD, 256 each), of which
// 4 OT a row are sums of the last convolution and one a tile says where its cells are.
constexpr int irBlockRows(int OT, int S) { return OT == 1 ? 10 : OT == 2 ? (S == 1 ? 7 : 5) : OT == 3 ? 4 : OT == 4 ? 3 : 2; }
constexpr int irBlockTiles(int S) { return S == 1 ? 6 : 10; }

// ---------------------------------------------------------------------------
// ir_block_i8: a workgroup makes all channels of a strip of output rows of one image.
//
// It walks over the wide channels in chunks of 32, and per chunk:
// Phase 1, the widening convolution: the pixels under the strip's windows are rows of a [pixels][K] matrix, 32 of them a tile, straight from memory
// in MFMA operand layout; requantised, the chunk's 32 channels of a pixel go to LDS as a cell of 16 bytes in each of
// two planes (channel 8 a + 4 j + e is byte 4 a + e of plane j). Cells outside the image hold the depthwise op's zero point.
// Phase 2, the depthwise convolution as a product: 16 channels x 16 neighbouring pixels of a row are one v_mfma_i32_16x16x64_i8 per
// window row, K = (tap, channel) with the taps' weights on the diagonals of 16 x 16 blocks (the fourth block is zero); its right operand is the
// 16 bytes of a cell as they lie.  Fifteen sixteenths of these products are zeros, but the vector pipes, which bound this path,
// have none of it: no byte transposes and no dot products.  The two planes' results of a lane are 8 neighbouring channels of a pixel, which is
// the right operand of v_mfma_i32_16x16x32_i8: phase 3, the narrowing convolution, adds the chunk's share to sums in registers.
// Chunks alternate between two LDS buffers: a wave widens the next one before it convolves this one, one barrier separates them, and each phase's
// weights are fetched during the other.
// RUNS: a convolution over few channels in the widening one's place (the first layer of an image network), as in ir_expand_dw_i8, to one chunk at most: there
// are no sums to keep, so four waves a SIMD overlap one another's phases, and a strip may be a block of columns of its rows.
//
// Why: apart, the depthwise result (2.3 MB per image of a 224 x 224 mobile network) is written and read back by a launch of its own.  Bound by
// vector instructions and MFMAs that two waves a SIMD overlap in part: an instruction takes the SIMD 4.3 to 4.6 cycles (a wave alone issues one in 5 to 5.7), which is 58 % of the cycles
// (75 % of a first layer's, at four waves), and MFMAs 15 to 20 %.  Measured one behind another, us, the two launches / this one:
//   batch 256  224x224x3 -> 112x112x32 -> 16 98 / 71, 112x112x16 -> 96 stride 2 -> 32 98 / 95, 56x56x32 -> 144 -> 32 and the add 88 / 83,
//              its stride 2 45 / 39, 28x28x32 -> 192 -> 32 35 / 25
//   batch 32   24.6 / 13.4, 21.5 / 17.5, 21.6 / 17.5, 12.8 / 12.5, 11.2 / 11.0
//   batch 1    10.0 / 5.4; 8.1 / 8.1, 8.4 / 9.0, 7.8 / 9.9, 7.9 / 9.8 (left to the two launches)
// and left at any batch: 14x14x64 -> 384 -> 64 21.1 / 33.3 (223 images), 14x14x96 -> 576 -> 96 38.5 / 53, whose chunks are too small for what each costs.  Tried on it: four waves a SIMD
// (their registers hold half the rows, the chunks' constants are fetched twice as often: 85 -> 103), waves that only widen beside waves that
// only convolve (94), the next row's cells and products, or the next tile's, ahead of this one's requant (85; 56x56x32 -> 144 -> 32 89.7 -> 92.3).
// ---------------------------------------------------------------------------
template <int KS, int S, bool RUNS, int OT, int DW>
__global__ __launch_bounds__(256, RUNS ? 4 : 2) void ir_block_i8(IrBlockArgs p, FastDiv divRegion, FastDiv divColumns) {
    constexpr int RT = irBlockRows(OT, S), T = irBlockTiles(S);
    extern __shared__ __attribute__((aligned(16))) int8_t cells[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // neighbouring strips on one XCD: they share rows of the input
    int n, oy0, ox0;
    {
        const int nb = (int)gridDim.x, pid = (int)blockIdx.x;
        const int per = nb / 8, rem = nb % 8, xcd = pid % 8, idx = pid / 8;
        const int lin = xcd * per + (xcd < rem ? xcd : rem) + idx;
        const int rest = lin / p.columnBlocks;
        ox0 = (lin - rest * p.columnBlocks) * p.blockColumns;
        n = rest / p.strips;
        oy0 = (rest - n * p.strips) * p.stripRows;
    }
    const int rows = p.OH - oy0 < p.stripRows ? p.OH - oy0 : p.stripRows, columns = p.OW - ox0 < p.blockColumns ? p.OW - ox0 : p.blockColumns;
    const int iyFirst = oy0 * S - p.PT, ixFirst = ox0 * S - p.PL;
    const int iyLo = iyFirst < 0 ? 0 : iyFirst, iyEnd = iyFirst + (rows - 1) * S + 3, iyHi = iyEnd < p.H ? iyEnd : p.H;
    const int ixLo = p.columnBlocks == 1 ? 0 : ixFirst;  // column 0 of the region
    const int pixels = (iyHi - iyLo) * p.regionColumns;
    const int cellCols = p.cellCols, cellRowBytes = cellCols * 16, trash = p.cellRows * cellRowBytes, planeBytes = trash + 16;
    const int chunks = (p.C + 31) / 32, bufferBytes = chunks > 1 ? 2 * planeBytes : 0;

    // ---- phase 1's pixels ----
    const int fr = lane & 31, half = lane >> 5;
    // where the cell of pixel m of the region is, for the lane's plane; pixels that have none share one behind the others
    auto cellOf = [&](int m, int &iy, int &ix) {
        const int r = (int)fastDiv((uint32_t)m, divRegion);
        iy = iyLo + r;
        ix = ixLo + m - r * p.regionColumns;
        const int cellCol = ix - ixFirst;
        const bool ok = m < pixels && (unsigned)ix < (unsigned)p.W && (unsigned)cellCol < (unsigned)cellCols;
        return half * planeBytes + (ok ? (iy - iyFirst) * cellRowBytes + cellCol * 16 : trash);
    };
    const int imageBytes = RUNS ? p.IH * p.IW * p.IC : p.H * p.W * p.K;
    const int8_t *x = p.x + (size_t)n * imageBytes + (RUNS ? 0 : iyLo * p.W * p.K);
    const int64_t before = (int64_t)n * imageBytes, behind = p.xBytes - before - 16;
    const int runLo = before < 1024 ? -(int)before : -1024, runHi = behind < 0x7fffffff ? (int)behind : 0x7fffffff;
    const int runRow = p.IW * p.IC;
    int khOff[KS];  // from a window's first row to the lane's; beyond the window its first one again, against zero weights
#pragma unroll
    for (int s = 0; s < KS; s++) khOff[s] = (2 * s + half < p.CKH ? 2 * s + half : 0) * runRow;
    struct Tile {
        int cell, y, at;  // RUNS: its window's first row, and where in a row it starts
    };
    int cellAt[RUNS ? 1 : T];
    if constexpr (!RUNS) {
        int iy, ix;
#pragma unroll
        for (int t = 0; t < T; t++) cellAt[t] = cellOf((t * 4 + wave) * 32 + fr, iy, ix);
    }
    // tile t of the wave: where its cells are, and its pixels under way; behind the last pixel, that one again
    auto loadTile = [&](auto tag, v4i(&a)[KS]) {
        Tile e{};
        const int t = tag, m = (t * 4 + wave) * 32 + fr;
        if constexpr (RUNS) {
            int iy, ix;
            e.cell = cellOf(m, iy, ix);
            e.y = iy * p.CS - p.CPT;
            e.at = (ix * p.CS - p.CPL) * p.IC;
            const int first = e.y * runRow + e.at;
#pragma unroll
            for (int s = 0; s < KS; s++) {
                const int off = first + khOff[s];
                a[s] = ((const UnalignedV4 *)(x + (off < runLo ? runLo : off > runHi ? runHi : off)))->v;
            }
        } else {
            e.cell = cellAt[t];
            const uint32_t from = (uint32_t)((m < pixels ? m : pixels - 1) * p.K);
#pragma unroll
            for (int s = 0; s < KS; s++) a[s] = *(const v4i *)(x + (from + (32 * s + 16 * half < p.K ? 32 * s + 16 * half : 0)));  // beyond K: against zero weights
        }
        return e;
    };

    // ---- a chunk's constants ----
    const int slot = lane & 15, group = lane >> 4;
    v4i w[KS], scale1[4];
    v16i bias1;
    // addresses: a uniform base that moves with the chunk and an offset of the lane's that does not
    auto at = [](const void *base, uint32_t offset) { return (const int8_t *)base + offset; };
    const uint32_t widenRow = (uint32_t)(fr * p.Kp + 16 * half), narrowRow = (uint32_t)((4 * OT * (slot >> 2) + (slot & 3)) * p.Kp3 + 8 * group);
    auto loadWiden = [&](int chunk) {
        const int ch0 = chunk * 32;
        const int8_t *rows = p.wexp + (size_t)ch0 * p.Kp;
#pragma unroll
        for (int s = 0; s < KS; s++) w[s] = *(const v4i *)at(rows + 32 * s, widenRow);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const v4i b4 = *(const v4i *)at(p.bias1 + ch0 + 8 * q, 16u * half);
            scale1[q] = *(const v4i *)at(p.scale1 + ch0 + 8 * q, 16u * half);
#pragma unroll
            for (int e = 0; e < 4; e++) bias1[4 * q + e] = b4[e];
        }
    };
    uint32_t taps[2][3];
    v4i bias2[2], scale2[2];
    long wproj[OT];
    // the lane's output channels are 4 OT group + 4 t + e: neighbours, so its row of tile t of the weights is that of channel
    // 4 OT (slot / 4) + 4 t + slot % 4.  Depthwise channels beyond C, half a chunk, are made of the chunk's first ones: they meet
    // zero weights.
    auto loadDepthwise = [&](int chunk) {
        const int ch0 = chunk * 32;
        const bool whole = ch0 + 32 <= p.C;
        const uint32_t tapAt = 4 * depthwiseTapAt(whole, slot), channelAt = whole || group < 2 ? 32u * group : 0u;
#pragma unroll
        for (int j = 0; j < 2; j++) {
#pragma unroll
            for (int kh = 0; kh < 3; kh++) taps[j][kh] = *(const uint32_t *)at(p.wdw + (size_t)kh * p.C + ch0 + 4 * j, tapAt);
            bias2[j] = *(const v4i *)at(p.bias2 + ch0 + 4 * j, channelAt);
            scale2[j] = *(const v4i *)at(p.scale2 + ch0 + 4 * j, channelAt);
        }
#pragma unroll
        for (int t = 0; t < OT; t++) wproj[t] = *(const long *)at(p.wproj + ch0 + (size_t)(4 * t) * p.Kp3, narrowRow);
    };
    v4i a0[KS], a1[KS];
    loadWiden(0);
    Tile e0 = loadTile(std::integral_constant<int, 0>{}, a0), e1;

    // ---- the lane's pixels of phase 2 ----
    const int item = wave * 16 + slot;
    const int seg = (int)fastDiv((uint32_t)item, divColumns), column = item - seg * p.blockColumns, oyA = seg * p.segmentRows;
    int left = rows - oyA < p.segmentRows ? rows - oyA : p.segmentRows;  // rows of its segment
    if (seg >= p.segments || column >= columns || left < 0) left = 0;
    // the cell under the lane's tap of the first row; a lane without rows reads those of segment 0
    const int src0 = (left > 0 ? (oyA * S * cellCols + column * S) * 16 : 0) + (group < 3 ? group : 2) * 16;
    // its results: `step` bytes from row to row
    const size_t firstOut = (((size_t)n * p.OH + oy0) * p.OW + ox0) * p.O;
    const uint32_t laneOut = (uint32_t)((oyA * p.OW + column) * p.O + 4 * OT * group), step = (uint32_t)(p.OW * p.O);

    {
        const int zp4 = (int)((uint32_t)(p.zp & 0xff) * 0x01010101u), bytes = 2 * planeBytes + bufferBytes;
        for (int i = tid * 16; i < bytes; i += 4096) *(v4i *)(cells + i) = v4i{zp4, zp4, zp4, zp4};
    }
    __syncthreads();

    const WideRequant w1 = wideRequant(p.rq1), w2 = wideRequant(p.rq2), w3 = wideRequant(p.rq3);
    auto widenTile = [&](const Tile &e, v4i(&a)[KS], int8_t *buffer) {
        if constexpr (RUNS) {
            // runs that reach into the padding, or that were read elsewhere than they lie (at the tensor's two ends), are put right
            const int first = e.y * runRow + e.at, last = first + (p.CKH - 1) * runRow;
            const bool wanted = e.cell != half * planeBytes + trash;
            const bool bad = e.y < 0 || e.y + p.CKH > p.IH || e.at < 0 || e.at + p.runBytes > runRow || last > runHi;
            if (__ballot(bad && wanted) != 0) {
                const uint32_t zp4 = (uint32_t)(p.czp & 0xff) * 0x01010101u;
                if (__ballot((first < runLo || last > runHi) && wanted) != 0) {
#pragma unroll
                    for (int s = 0; s < KS; s++) {
                        const int kh = 2 * s + half < p.CKH ? 2 * s + half : 0, off = first + khOff[s];
                        // a row of the window outside the image is all padding
                        a[s] = fixRun16(a[s], off - (off < runLo ? runLo : off > runHi ? runHi : off), -e.at, (unsigned)(e.y + kh) >= (unsigned)p.IH ? 0 : runRow - e.at, zp4);
                    }
                } else {
                    // masks of the bytes inside the row, the same for every row of the window: a quarter of fixRun16's instructions, in half of the tiles of a right-hand
                    // block (224x224x3 -> 112x112x32 -> 16, 256 images: 97 us with fixRun16, 90 so, the narrow convolution as it was)
                    uint32_t in[4];
#pragma unroll
                    for (int d = 0; d < 4; d++) {
                        const int past = 8 * (4 * d + 4 - (runRow - e.at));  // bits of the dword behind the row
                        in[d] = (uint32_t)(0xffffffffull >> (past < 0 ? 0 : past > 32 ? 32 : past));
                    }
                    if (__ballot(e.at < 0) != 0) {
#pragma unroll
                        for (int d = 0; d < 4; d++) {
                            const int before = 8 * (-e.at - 4 * d);
                            in[d] &= (uint32_t)(0xffffffffull << (before < 0 ? 0 : before > 32 ? 32 : before));
                        }
                    }
#pragma unroll
                    for (int s = 0; s < KS; s++) {
                        const int kh = 2 * s + half < p.CKH ? 2 * s + half : 0;
                        const bool row = (unsigned)(e.y + kh) < (unsigned)p.IH;
#pragma unroll
                        for (int d = 0; d < 4; d++) {
                            const uint32_t keep = row ? in[d] : 0u;
                            a[s][d] = (int)(((uint32_t)a[s][d] & keep) | (zp4 & ~keep));
                        }
                    }
                }
            }
        }
        v16i acc = bias1;
#pragma unroll
        for (int s = 0; s < KS; s++) acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(w[s], a[s], acc, 0, 0, 0);
        v4i o;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const v4i t0 = {acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
            o[q] = (int)requantPack4<4>(t0, scale1[q], 0, p.rq1, w1);
        }
        *(v4i *)(buffer + e.cell) = o;
    };
    // The wave's tiles, the next one's pixels under way; dense ones end with the first tile's again, for the next chunk.
    auto widen = [&](int8_t *buffer) {
        const int mine = (pixels - wave * 32 + 127) / 128;
        if constexpr (RUNS) {
            for (int t = 0; t < mine; t += 2) {
                e1 = loadTile(t + 1, a1);
                widenTile(e0, a0, buffer);
                if (t + 1 >= mine) break;
                e0 = loadTile(t + 2, a0);
                widenTile(e1, a1, buffer);
            }
        } else {
            firstOf(std::make_integer_sequence<int, T>{}, mine, [&](auto tag) {
                constexpr int t = decltype(tag)::value;
                constexpr int next = t + 1 < T ? t + 1 : 0;
                if constexpr (t % 2 == 0) {
                    e1 = loadTile(std::integral_constant<int, next>{}, a1);
                    widenTile(e0, a0, buffer);
                } else {
                    e0 = loadTile(std::integral_constant<int, next>{}, a0);
                    widenTile(e1, a1, buffer);
                }
                __builtin_amdgcn_sched_barrier(0);
            });
            e0 = loadTile(std::integral_constant<int, 0>{}, a0);
        }
    };
    // one output row of the lane's 4 OT channels, its requant, the add and the store
    auto finishRow = [&](auto mode, auto adds, int r, const v4i(&sums)[OT], const v4i(&scale3)[OT], const uint32_t(&other)[OT]) {
        if (r < left) {
#pragma unroll
            for (int t = 0; t < OT; t++) {
                uint32_t o = requantPack4<decltype(mode)::value>(sums[t], scale3[t], 0, p.rq3, w3);
                if (decltype(adds)::value) o = residualAdd4<true>(o, other[t], p.addSkipFirst != 0, p.addW0, p.addW1, 0, 1, 0, p.arq, p.addFolded);
                *(uint32_t *)(p.out + firstOut + (laneOut + r * step + 4 * t)) = o;
            }
        }
    };
    // f(mode, adds): which requant the narrow convolution has and whether an add follows, asked once: branches in every row keep a wave from issuing (256 images,
    // us, in every row / once: 224x224x3 -> 112x112x32 -> 16 90.4 / 80.8, 56x56x32 -> 144 -> 32 and the add 89.7 / 86.0, 28x28x32 -> 192 -> 32 30.0 / 28.9)
    auto withFinish = [&](auto &&f) {
        withPackedRequant(w3, [&](auto mode) {
            if (p.skip) f(mode, std::true_type{});
            else f(mode, std::false_type{});
        });
    };
    auto loadSkip = [&](auto adds, int r, uint32_t(&other)[OT]) {
#pragma unroll
        for (int t = 0; t < OT; t++) other[t] = decltype(adds)::value && r < left ? *(const uint32_t *)(p.skip + firstOut + (laneOut + r * step + 4 * t)) : 0u;
    };
    v4i bias3[OT], scale3[OT];
    auto loadNarrow = [&](const int32_t *from, v4i(&to)[OT]) {
#pragma unroll
        for (int t = 0; t < OT; t++) to[t] = *(const v4i *)(from + 4 * OT * group + 4 * t);
    };
    // f(row, the narrowing convolution's operand): output rows of the strip one by one
    auto depthwise = [&](const int8_t *buffer, auto &&f) {
        v4i wd[2][3], ring[3][2];
        depthwiseWeights(taps, slot, group, wd);
        const int8_t *src = buffer + src0;
        auto row = [&](v4i(&o)[2]) { depthwiseRow(src, planeBytes, cellRowBytes, o); };
        row(ring[0]);
        if (S == 1) row(ring[1]);
        firstOf(std::make_integer_sequence<int, RT>{}, p.segmentRows, [&](auto tag) {
            constexpr int r = decltype(tag)::value, i0 = r * S % 3, i1 = (i0 + 1) % 3, i2 = (i0 + 2) % 3;
            if (S == 2) row(ring[i1]);
            row(ring[i2]);
            f(tag, __builtin_bit_cast(long, depthwiseResults<DW>(wd, ring[i0], ring[i1], ring[i2], bias2, scale2, p.rq2, w2)));
        });
    };

    if constexpr (RUNS) {
        widen(cells);
        loadDepthwise(0);
        loadNarrow(p.bias3, bias3);
        loadNarrow(p.scale3, scale3);
        __syncthreads();
        withFinish([&](auto mode, auto adds) {
            depthwise(cells, [&](auto tag, long o) {
                constexpr int r = decltype(tag)::value;
                uint32_t other[OT];
                loadSkip(adds, r, other);
                v4i sums[OT];
#pragma unroll
                for (int t = 0; t < OT; t++) sums[t] = __builtin_amdgcn_mfma_i32_16x16x32_i8(wproj[t], o, bias3[t], 0, 0, 0);
                finishRow(mode, adds, r, sums, scale3, other);
            });
        });
    } else {
        v4i sum[RT][OT];
        loadNarrow(p.bias3, bias3);
#pragma unroll
        for (int r = 0; r < RT; r++) {
#pragma unroll
            for (int t = 0; t < OT; t++) sum[r][t] = bias3[t];
        }
        widen(cells);
        loadDepthwise(0);
        if (chunks > 1) loadWiden(1);
        __syncthreads();
        for (int c = 0; c < chunks; c++) {
            if (c + 1 < chunks) widen(cells + (~c & 1) * bufferBytes);
            if (c + 2 < chunks) loadWiden(c + 2);
            depthwise(cells + (c & 1) * bufferBytes, [&](auto tag, long o) {
                constexpr int r = decltype(tag)::value;
#pragma unroll
                for (int t = 0; t < OT; t++) sum[r][t] = __builtin_amdgcn_mfma_i32_16x16x32_i8(wproj[t], o, sum[r][t], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            });
            if (c + 1 < chunks) loadDepthwise(c + 1);
            __syncthreads();
        }
        loadNarrow(p.scale3, scale3);
        withFinish([&](auto mode, auto adds) {
            uint32_t other[RT][OT];
#pragma unroll
            for (int r = 0; r < RT; r++) loadSkip(adds, r, other[r]);
#pragma unroll
            for (int r = 0; r < RT; r++) finishRow(mode, adds, r, sum[r], scale3, other[r]);
        });
    }
}

constexpr size_t kIrBlockMaxLds = 80 * 1024;  // two workgroups a CU

static bool packedRequant(const Requant &rq, int mostShift) {
    return (rq.shift == 32 || (rq.shift > 32 && rq.pre_shift == 0 && rq.t0_clamp == 0)) && rq.shift <= mostShift && rq.out_max == 127 && rq.out_min >= -128 && rq.out_min <= 127 && rq.out_zp >= -32768 &&
           rq.out_zp <= 32767;
}

// The depthwise op's 9 taps leave scales that start above 1/2 here and there, for all channels of an op a shift below 32 then: mode 3.
static bool preShiftedRequant(const Requant &rq) {
    return rq.shift >= 3 && rq.shift < 32 && rq.pre_shift == 33 - rq.shift && rq.t0_clamp == 0 && rq.out_min >= -128 && rq.out_max <= 127 && rq.out_min <= rq.out_max && rq.out_zp >= -32768 &&
           rq.out_zp <= 32767;
}

// The time of a launch, us: of a workgroup alone on its CU a start, its chunks, each of which costs something whatever its size, then a share a tile
// of a wave and a share an output row, and at the end the add of its rows; of those that share a CU more.  Fitted to 789 blocks by every height of strips (few
// channels: 111 first layers), half of them of mobile networks and the others of 16 .. 96 channels in and out, 1 .. 6 times as many wide ones, 7 .. 112 pixels, 1 .. 256 images:
// half of 1828 within 5 %, nine in ten within 18 %, those of 96 channels in up to 40 % low; strips by it take 0.3 % longer than the best.
static double irBlockTime(const IrBlockArgs &a) {
    struct Cost {
        double launch, start, chunk, tile, tileK, row, rowO, add, shared;
        int perCu;
    };
    constexpr Cost dense{2.61, 1.41, 0.439, 0.174, 0.062, 0.051, 0.045, 0.086, 0.508, 2}, runs{2.62, 0.97, 0.01, 0.361, 0.067, 0.085, 0.067, 0.0, 0.434, 4};
    const Cost &c = a.CKH > 0 ? runs : dense;
    const int KS = a.CKH > 0 ? (a.CKH + 1) / 2 : (a.K + 31) / 32, OT = (a.O + 15) / 16, imageRows = a.cellRows < a.H ? a.cellRows : a.H;
    const long long blocks = (long long)a.N * a.strips * a.columnBlocks, room = 256LL * c.perCu, rest = blocks % room;
    const int tiles = (imageRows * a.regionColumns + 127) / 128, chunks = (a.C + 31) / 32;
    const double alone = c.start + chunks * (c.chunk + tiles * (c.tile + c.tileK * (KS - 1)) + a.segmentRows * (c.row + c.rowO * OT)) + (a.skip ? a.segmentRows * OT * c.add : 0.0);
    auto together = [&](long long n) { return n > 0 ? alone * (1 + c.shared * (double)(n - 1)) : 0.0; };
    return c.launch + (double)(blocks / room) * together(c.perCu) + together((rest + 255) / 256);
}

// The time of ir_expand_dw_i8, by its own estimate, and the pointwise convolution behind it, us, by millions of depthwise and narrow values and wide channels: nine in
// ten of the 1828 within 6 %.  The choice by the two costs 0.2 % of the better one's time over them and 1.3 at most, always two launches 6 %, always one 43 %; 45 of
// them are more than 3 % behind the other way.  First layers are all one launch (two: 1.7 times the time).
static double irPairTime(const IrBlockArgs &a) {
    IrExpandDwArgs f{};
    f.N = a.N; f.H = a.H; f.W = a.W; f.K = a.K; f.C = a.C; f.OH = a.OH; f.OW = a.OW; f.S = a.S; f.PT = a.PT; f.PL = a.PL; f.CKH = a.CKH;
    const double out = 1e-6 * a.N * a.OH * a.OW;
    const double narrow = a.CKH > 0 ? 2.4 + out * (0.229 * a.C + 0.562 * a.O) : 2.42 + out * (0.234 * a.C + 0.409 * a.O) + 0.0018 * a.C + (a.skip ? 0.157 + 0.267 * out * a.O : 0.0);
    return irExpandDwTime(&f) + narrow;
}

bool planIrBlock(IrBlockArgs *args) {
    IrBlockArgs &a = *args;
    const bool runs = a.CKH > 0;
    if (!a.x || !a.wexp || !a.bias1 || !a.scale1 || !a.wdw || !a.bias2 || !a.scale2 || !a.wproj || !a.bias3 || !a.scale3 || !a.out) return false;
    if (a.N <= 0 || a.H <= 0 || a.W <= 0 || a.C <= 0 || a.C % 16 != 0 || a.C > kIrMaxChannels || a.OH <= 0 || a.OW <= 0 || a.O <= 0 || a.O % 16 != 0) return false;
    if ((a.S != 1 && a.S != 2) || a.PT < 0 || a.PT > 2 || a.PL < 0 || a.PL > 2) return false;
    if ((a.OH - 1) * a.S - a.PT >= a.H || (a.OW - 1) * a.S - a.PL >= a.W) return false;
    if (!packedRequant(a.rq1, 40) || !(packedRequant(a.rq2, 40) || preShiftedRequant(a.rq2)) || !packedRequant(a.rq3, 45)) return false;
    const int KS = runs ? (a.CKH + 1) / 2 : (a.K + 31) / 32, OT = (a.O + 15) / 16;
    if (runs ? a.CKH > 4 || OT > 2 || a.C > 32 : a.K <= 0 || a.K % 16 != 0 || KS > 3 || a.OW > 64) return false;
    if (OT > 6) return false;
    if (a.Kp < KS * 32 || a.Np < (a.C + 31) / 32 * 32 || a.Kp3 < (a.C + 31) / 32 * 32 || a.Kp3 % 8 != 0) return false;
    if (runs) {
        if (a.IH <= 0 || a.IW <= 0 || a.IC <= 0 || a.CS <= 0 || a.CPT < 0 || a.CPL < 0 || a.runBytes <= 0 || a.runBytes > 16 || a.runBytes % a.IC != 0) return false;
        if (a.xBytes != (int64_t)a.N * a.IH * a.IW * a.IC || a.xBytes < 16 || (long long)a.IH * a.IW * a.IC > (1LL << 27)) return false;
    } else if ((uintptr_t)a.x & 15 || (long long)a.H * a.W * a.K >= (1LL << 31)) {
        return false;
    }
    if (((uintptr_t)a.wexp | (uintptr_t)a.bias1 | (uintptr_t)a.scale1 | (uintptr_t)a.wdw | (uintptr_t)a.bias2 | (uintptr_t)a.scale2 | (uintptr_t)a.wproj | (uintptr_t)a.bias3 |
         (uintptr_t)a.scale3) & 15) return false;
    if (((uintptr_t)a.out | (uintptr_t)a.skip) & 3) return false;
    a.addFolded = 0;
    if (a.skip && !residualAddFolded(a.addW0, a.addW1, a.addBias, a.addScale, a.arq, &a.addFolded)) return false;

    a.columnBlocks = (a.OW + 63) / 64;
    a.blockColumns = (a.OW + a.columnBlocks - 1) / a.columnBlocks;
    a.segments = 64 / a.blockColumns;
    a.cellCols = (a.blockColumns - 1) * a.S + 3;
    a.regionColumns = a.columnBlocks == 1 ? a.W : a.cellCols;
    const int buffers = a.C > 32 ? 2 : 1, mostRows = irBlockRows(OT, a.S);
    auto cellRowsOf = [&](int rows) { return (rows - 1) * a.S + 3; };
    auto setRows = [&](int segmentRows) {
        a.segmentRows = segmentRows;
        a.stripRows = segmentRows * a.segments;
        a.strips = (a.OH + a.stripRows - 1) / a.stripRows;
        a.cellRows = cellRowsOf(a.stripRows);
    };
    auto fits = [&](int segmentRows, int segments) {
        const int cellRows = cellRowsOf(segments * segmentRows), imageRows = cellRows < a.H ? cellRows : a.H;
        return (runs || (long long)imageRows * a.regionColumns <= irBlockTiles(a.S) * 128) && ((size_t)cellRows * a.cellCols + 1) * 32 * buffers <= (runs ? kIrBlockMaxLds / 2 : kIrBlockMaxLds);
    };
    if (a.segments > a.OH) a.segments = a.OH;
    while (a.segments > 1 && !fits(1, a.segments)) a.segments--;
    if (!fits(1, a.segments)) return false;
    // strips as high as the estimate says; of equal ones the lowest that make as many strips
    double best = 0;
    int segmentRows = 0;
    for (int tried = 1; tried <= mostRows && (tried == 1 || (tried - 1) * a.segments < a.OH) && fits(tried, a.segments); tried++) {
        setRows(tried);
        const double time = irBlockTime(a);
        if (segmentRows == 0 || time < best) {
            best = time;
            segmentRows = tried;
        }
    }
    setRows(segmentRows);
    return (long long)a.N * a.strips * a.columnBlocks < (1LL << 31) && (long long)a.OH * a.OW * a.O < (1LL << 31);
}

bool irBlockFits(const IrBlockArgs &in) {
    IrBlockArgs a = in;
    return planIrBlock(&a);
}

bool irBlockBetter(const IrBlockArgs &in) {
    IrBlockArgs a = in;
    return planIrBlock(&a) && irBlockTime(a) < 0.97 * irPairTime(a);
}

static size_t irBlockLds(const IrBlockArgs &a) { return ((size_t)a.cellRows * a.cellCols + 1) * 32 * (a.C > 32 ? 2 : 1); }

template <int KS, int S, bool RUNS, int OT, int DW>
static hipError_t launchBlockDw(const IrBlockArgs &a, const LaunchCtx &ctx) {
    auto kernel = ir_block_i8<KS, S, RUNS, OT, DW>;
    static std::once_flag once;
    static hipError_t configured = hipSuccess;
    std::call_once(once, [&] { configured = hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kIrBlockMaxLds); });
    if (configured != hipSuccess) return configured;
    THIP_ENQUEUE(ctx, kernelLabel("ir_block_i8", {KS, S, (int)RUNS, OT, DW}), kernel, dim3((unsigned)(a.N * a.strips * a.columnBlocks)), dim3(256), irBlockLds(a), a,
                 makeFastDiv((uint32_t)a.regionColumns), makeFastDiv((uint32_t)a.blockColumns));
    return hipGetLastError();
}

template <int KS, int S, bool RUNS, int OT>
static hipError_t launchBlock(const IrBlockArgs &a, const LaunchCtx &ctx) {
    return a.rq2.shift < 32 ? launchBlockDw<KS, S, RUNS, OT, 3>(a, ctx) : launchBlockDw<KS, S, RUNS, OT, 4>(a, ctx);
}

template <int KS, int S>
static hipError_t launchBlockO(const IrBlockArgs &a, const LaunchCtx &ctx) {
    switch ((a.O + 15) / 16) {
    case 1: return launchBlock<KS, S, false, 1>(a, ctx);
    case 2: return launchBlock<KS, S, false, 2>(a, ctx);
    case 3: return launchBlock<KS, S, false, 3>(a, ctx);
    case 4: return launchBlock<KS, S, false, 4>(a, ctx);
    case 5: return launchBlock<KS, S, false, 5>(a, ctx);
    default: return launchBlock<KS, S, false, 6>(a, ctx);
    }
}

template <int S>
static hipError_t launchBlockS(const IrBlockArgs &a, const LaunchCtx &ctx) {
    if (a.CKH > 0) {
        if (a.O <= 16) return a.CKH <= 2 ? launchBlock<1, S, true, 1>(a, ctx) : launchBlock<2, S, true, 1>(a, ctx);
        return a.CKH <= 2 ? launchBlock<1, S, true, 2>(a, ctx) : launchBlock<2, S, true, 2>(a, ctx);
    }
    switch ((a.K + 31) / 32) {
    case 1: return launchBlockO<1, S>(a, ctx);
    case 2: return launchBlockO<2, S>(a, ctx);
    default: return launchBlockO<3, S>(a, ctx);
    }
}

hipError_t launchIrBlock(const IrBlockArgs &in, const LaunchCtx &ctx) {
    IrBlockArgs a = in;
    if (!planIrBlock(&a)) return hipErrorInvalidValue;
    return a.S == 1 ? launchBlockS<1>(a, ctx) : launchBlockS<2>(a, ctx);
}

}  // namespace thip
