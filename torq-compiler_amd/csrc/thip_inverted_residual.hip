// gfx950 kernel of the front half of an inverted-residual block: the pointwise convolution that widens the channels and the
// 3 x 3 depthwise convolution behind it as one launch, the widened image never leaving LDS.
#include "thip_inverted_residual.h"
#include "thip_ir_depthwise.h"
#include "thip_kernels_common.h"

#include <math.h>

namespace thip {

// The requant tails that need 32-bit arithmetic only (withPackMode without its 64-bit one; the planner keeps such records
// apart).
template <typename F>
__device__ __forceinline__ void withNarrowPackMode(const WideRequant &w, F &&f) {
    if (w.packed && w.packShift <= 0) f(std::integral_constant<int, 4>{});
    else if (w.packed) f(std::integral_constant<int, 5>{});
    else if (w.plain) f(std::integral_constant<int, 2>{});
    else if (w.preOnly) f(std::integral_constant<int, 3>{});
    else f(std::integral_constant<int, 1>{});
}

// Columns of cells under the windows of one output row.
static inline int irCellColumns(int OW, int S) { return (OW - 1) * S + 3; }

// ---------------------------------------------------------------------------
// ir_expand_dw_i8: a workgroup makes 32 channels of a strip of output rows of one image.
//
// Phase 1, the pointwise convolution: the strip's input pixels are rows of a dense [pixels][K] matrix; a wave takes 32 of
// them at a time straight from memory in MFMA operand layout (K <= 192: at most six loads per lane, prefetched one tile ahead), the
// 32 channels' weights stay in registers, and the requantised bytes go to LDS as cells of 16 bytes [row][column] in each of two planes (channel
// 8 a + 4 j + e is byte 4 a + e of plane j). Cells outside the image hold the depthwise op's zero point.
// RUNS: a convolution over few channels instead (the first layer of an image network): K is one 16-byte run per window row, and the pixels are gathered from the image.
// Phase 2, the depthwise convolution as a product, as in ir_block_i8: 16 channels x 16 pixels are one v_mfma_i32_16x16x64_i8 per window row with
// the taps on the diagonals of 16 x 16 blocks. A lane owns a column of a segment of the strip's rows, of any image of the workgroup's, and walks down it: two 16-byte
// loads from LDS a row, and its group's 8 neighbouring channels of a pixel are one 8-byte store.
//
// Why: apart, the two launches write the widened image and read it back (3.3 MB per image of a 224 x 224 mobile network, 6.7 MB of
// its 11 MB of traffic), and at small batches each costs a dependent launch. About half of the cycles are vector instructions (5 per widened and 5 per depthwise
// byte; with byte transposes and v_dot4_i32_i8 in phase 2 it was 9 per depthwise byte); the rest goes where a workgroup's phases and the launch's last round of workgroups wait.
// us, in a trace of the network, with v_dot4_i32_i8 / now:
//   batch 256  14x14x64 -> 384 17.4 / 14.6, 14x14x96 -> 576 24.6 / 21.7, its stride 2 17.3 / 15.0, 7x7x160 -> 960 17.0 / 14.5
// and one behind another, in time from one to the next
//   batch 32   7x7x160 -> 960 8.0 / 5.3, 14x14x96 -> 576 7.9 / 7.4, its stride 2 6.4 / 5.7, 14x14x64 -> 384 6.0 / 6.0, 28x28x32 -> 192 7.9 / 6.9
//   batch 1    14x14x64 -> 384 3.9 / 4.0
// the whole network at 256 images 716 -> 695, and 676 -> 672 with strips and images by irTime (at 32 in host memory and at one the runs of one build differ by as much as it gave). Tried: phase 2's constants under way from the start on (registers spill from K = 96
// on: 23.8 -> 25.5), the requants' constants from the host (no change, and spills), more tiles prefetched (no change).
// ---------------------------------------------------------------------------
template <int KS, int S, bool RUNS>
__global__ __launch_bounds__(256, KS <= 3 ? 4 : 3) void ir_expand_dw_i8(IrExpandDwArgs p, FastDiv divW, FastDiv divH, FastDiv divCols, FastDiv divSegments) {
    extern __shared__ __attribute__((aligned(16))) int8_t cells[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // channel chunks of a strip are neighbours on one XCD: they read the same pixels and write pieces of the same lines
    int chunk, strip, n;
    {
        const int nb = (int)gridDim.x, pid = (int)blockIdx.x;
        const int per = nb / 8, rem = nb % 8, xcd = pid % 8, idx = pid / 8;
        const int lin = xcd * per + (xcd < rem ? xcd : rem) + idx;
        const int chunks = (p.C + kIrChunk - 1) / kIrChunk;
        const int rest = lin / chunks;
        chunk = lin - rest * chunks;
        n = rest / p.strips;
        strip = rest - n * p.strips;
    }
    n *= p.images;
    const int ch0 = chunk * kIrChunk;
    const IrStrip part = irStrip(p, n, strip);
    const int images = part.images, oy0 = part.oy0, iyFirst = part.iyFirst, iyLo = part.iyLo, cellRows = part.cellRows, pixels = part.pixels;
    const int cellCols = p.cellCols;

    // ---- phase 1 ----
    const int fr = lane & 31, half = lane >> 5;
    v4i w[KS];
    v16i bias;
    v4i scale[4];
    {
        const int8_t *wrow = p.wexp + (size_t)(ch0 + fr) * p.Kp + 16 * half;
#pragma unroll
        for (int s = 0; s < KS; s++) w[s] = *(const v4i *)(wrow + 32 * s);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const v4i b4 = *(const v4i *)(p.bias1 + ch0 + 8 * q + 4 * half), s4 = *(const v4i *)(p.scale1 + ch0 + 8 * q + 4 * half);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                bias[4 * q + e] = b4[e];
            }
            scale[q] = s4;
        }
    }
    const int imageBytes = RUNS ? p.IH * p.IW * p.IC : 0;
    const int8_t *x = RUNS ? p.x + (size_t)n * imageBytes : p.x + ((size_t)n * p.H + iyLo) * p.W * p.K;
    // offsets from x at which 16 bytes lie inside the tensor
    const int64_t before = (int64_t)n * imageBytes, behind = p.xBytes - before - 16;
    const int runLo = before < 1024 ? -(int)before : -1024, runHi = behind < 0x7fffffff ? (int)behind : 0x7fffffff;
    // bytes of K a lane has no chunk for meet zero weights: it re-reads its first chunk of the pixel
    int kOff[KS];
#pragma unroll
    for (int s = 0; s < KS; s++) kOff[s] = 32 * s + 16 * half < p.K ? 32 * s + 16 * half : 0;
    const int tiles = (pixels + 31) / 32;
    // RUNS: where the runs of the strip's pixel (r, c) start, from x; kh past the window meets zero weights
    auto runOffsets = [&](int r, int c, int(&off)[KS], int *iyTop, int *ixLeft) {
        const int image = p.images > 1 ? (int)fastDiv((uint32_t)r, divH) : 0;
        const int iy = (r - image * p.H + iyLo) * p.CS - p.CPT, ix = c * p.CS - p.CPL;
#pragma unroll
        for (int s = 0; s < KS; s++) {
            const int kh = 2 * s + half < p.CKH ? 2 * s + half : 0;
            off[s] = image * imageBytes + ((iy + kh) * p.IW + ix) * p.IC;
        }
        if (iyTop) *iyTop = iy;
        if (ixLeft) *ixLeft = ix;
    };
    auto clampRun = [&](int off) { return off < runLo ? runLo : off > runHi ? runHi : off; };
    // Puts a tile's runs that were read at a clamped offset, or that reach into the padding, right. The loads themselves are branch-free:
    // with gatherRun's cases around them the compiler waits for each before the next, and the prefetch is none
    // (224x224x3 -> 112x112x32 and its depthwise convolution, 256 images: 104.8 us so, 97.3 now).
    auto fixRuns = [&](int r, int c, v4i(&a)[KS]) {
        int off[KS], iy, ix;
        runOffsets(r, c, off, &iy, &ix);
        const int row = p.IW * p.IC, at = ix * p.IC;
        const uint32_t zp4 = (uint32_t)(p.czp & 0xff) * 0x01010101u;
        // bytes [lo, hi) of a run lie inside its row
        const int lo = at < 0 ? -at : 0, room = row - at;
#pragma unroll
        for (int s = 0; s < KS; s++) {
            const int kh = 2 * s + half < p.CKH ? 2 * s + half : 0;
            const int hi = (unsigned)(iy + kh) >= (unsigned)p.IH ? 0 : room;
            a[s] = fixRun16(a[s], off[s] - clampRun(off[s]), lo, hi, zp4);
        }
    };
    // the wave's first pixel, and its tiles' pixels behind it
    auto walkFrom = [&](int imageStep, int rowStep, int columnStep, int first) {
        const int m = wave * 32 + fr;
        const int r = (int)fastDiv((uint32_t)m, divW), image = p.images > 1 ? (int)fastDiv((uint32_t)r, divH) : 0;
        return irWalkFrom(p, m, r, image, imageStep, rowStep, columnStep, first);
    };
    const int cellRowBytes = cellCols * kIrPitch, cellImageBytes = cellRows * cellRowBytes;
    const int planeBytes = images * cellImageBytes;
    IrWalk cell = walkFrom(cellImageBytes, cellRowBytes, kIrPitch, (iyLo - iyFirst) * cellRowBytes + p.PL * kIrPitch + half * planeBytes);
    const int runRow = RUNS ? p.CS * p.IW * p.IC : 0, runColumn = RUNS ? p.CS * p.IC : 0;
    IrWalk run{};
    int khOff[KS];
    if constexpr (RUNS) {
        run = walkFrom(imageBytes, runRow, runColumn, ((iyLo * p.CS - p.CPT) * p.IW - p.CPL) * p.IC);
#pragma unroll
        for (int s = 0; s < KS; s++) khOff[s] = (2 * s + half < p.CKH ? 2 * s + half : 0) * p.IW * p.IC;
    }
    // every run that starts inside this workgroup's images can be read as 16 bytes
    const bool roomBehind = runHi >= images * imageBytes;
    uint32_t next = (uint32_t)((wave * 32 + fr) * p.K);
    const uint32_t last = (uint32_t)((pixels - 1) * p.K);
    // the wave's next tile; past the last pixel, the last one again or (RUNS) whatever lies there
    auto loadTile = [&](v4i(&a)[KS]) {
        if constexpr (RUNS) {
#pragma unroll
            for (int s = 0; s < KS; s++) a[s] = ((const UnalignedV4 *)(x + clampRun(run.at + khOff[s])))->v;
            irWalkOn(p, run, imageBytes, runRow, runColumn);
        } else {
            const int8_t *src = x + (next < last ? next : last);
#pragma unroll
            for (int s = 0; s < KS; s++) a[s] = *(const v4i *)(src + kOff[s]);
            next += 128u * (uint32_t)p.K;
        }
    };
    v4i a0[KS], a1[KS];
    loadTile(a0);
    {
        const int zp4 = (int)((uint32_t)(p.zp & 0xff) * 0x01010101u);
        for (int i = tid * 16; i < 2 * planeBytes; i += 4096) *(v4i *)(cells + i) = v4i{zp4, zp4, zp4, zp4};
    }
    __syncthreads();
    const WideRequant w1 = wideRequant(p.rq1);
    withNarrowPackMode(w1, [&](auto tag) {
        constexpr int kMode = decltype(tag)::value;
        auto computeTile = [&](int t, v4i(&a)[KS]) {
            const int m = t * 32 + fr;
            if constexpr (RUNS) {
                const int iy = (cell.row + iyLo) * p.CS - p.CPT, at = (cell.column * p.CS - p.CPL) * p.IC;
                const bool bad = !roomBehind || iy < 0 || iy + p.CKH > p.IH || at < 0 || at + p.runBytes > p.IW * p.IC;
                // rows past the last pixel are stored nowhere
                if (__ballot(bad && m < pixels) != 0 && m < pixels) {
                    const int r = (int)fastDiv((uint32_t)m, divW);
                    fixRuns(r, m - r * p.W, a);
                }
            }
            v16i acc = bias;
#pragma unroll
            for (int s = 0; s < KS; s++) acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(w[s], a[s], acc, 0, 0, 0);
            int8_t *dst = cells + cell.at;
            const bool inside = irHasCell(p, part, m, cell);
            irWalkOn(p, cell, cellImageBytes, cellRowBytes, kIrPitch);
            if (!inside) return;
            v4i o;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const v4i t0 = {acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
                o[q] = (int)requantPack4<kMode>(t0, scale[q], 0, p.rq1, w1);
            }
            *(v4i *)dst = o;
        };
        for (int t = wave; t < tiles; t += 8) {
            loadTile(a1);
            computeTile(t, a0);
            if (t + 4 >= tiles) break;
            loadTile(a0);
            computeTile(t + 4, a1);
        }
    });
    // phase 2's weights and constants, under way while other waves widen: their registers are not free before
    const int slot = lane & 15, group = lane >> 4;
    // channels beyond C, half a chunk, are made of the chunk's first ones and stored nowhere
    const bool whole = ch0 + 32 <= p.C, stored = whole || group < 2;
    const uint32_t tapAt = depthwiseTapAt(whole, slot), channelAt = stored ? 8 * group : 0;
    uint32_t taps[2][3];
    v4i bias2[2], scale2[2];
#pragma unroll
    for (int j = 0; j < 2; j++) {
#pragma unroll
        for (int kh = 0; kh < 3; kh++) taps[j][kh] = (uint32_t)(p.wdw + (size_t)kh * p.C + ch0 + 4 * j)[tapAt];
        bias2[j] = *(const v4i *)(p.bias2 + ch0 + 4 * j + channelAt);
        scale2[j] = *(const v4i *)(p.scale2 + ch0 + 4 * j + channelAt);
    }
    __syncthreads();

    // ---- phase 2 ----
    v4i wd[2][3];
    depthwiseWeights(taps, slot, group, wd);
    const WideRequant w2 = wideRequant(p.rq2);
    const int items = p.OW * p.segments * images, count = irWalkedRows(p, part);
    const uint32_t step = (uint32_t)(p.OW * p.C);
    int8_t *out = p.out + ((size_t)n * p.OH + oy0) * p.OW * p.C;
    withNarrowPackMode(w2, [&](auto tag) {
        constexpr int kMode = decltype(tag)::value;
        for (int first = wave * 16; first < items; first += 64) {
            const int item = first + slot;
            int seg = 0, image = 0, ox = item;
            if (p.segments * p.images > 1) {
                seg = (int)fastDiv((uint32_t)item, divCols);
                ox -= seg * p.OW;
            }
            if (p.images > 1) {
                image = (int)fastDiv((uint32_t)seg, divSegments);
                seg -= image * p.segments;
            }
            const IrColumn column = irColumn(p, part, S, item < items, image, seg, ox);
            const int left = stored ? column.left : 0;
            const int8_t *src = cells + column.first + (group < 3 ? group : 2) * kIrPitch;
            uint32_t dst = (uint32_t)(((image * p.OH + column.oy) * p.OW + ox) * p.C + ch0 + 8 * group);
            v4i ring[3][2];
            auto row = [&](v4i(&o)[2]) { depthwiseRow(src, planeBytes, cellRowBytes, o); };
            auto emit = [&](int r, const v4i(&r0)[2], const v4i(&r1)[2], const v4i(&r2)[2]) {
                const v2i o = depthwiseResults<kMode>(wd, r0, r1, r2, bias2, scale2, p.rq2, w2);
                if (r < left) ((UnalignedV2 *)(out + dst))->v = o;
                dst += step;
            };
            row(ring[0]);
            if (S == 1) {
                row(ring[1]);
                for (int r = 0;;) {
                    row(ring[2]);
                    emit(r, ring[0], ring[1], ring[2]);
                    if (++r >= count) break;
                    row(ring[0]);
                    emit(r, ring[1], ring[2], ring[0]);
                    if (++r >= count) break;
                    row(ring[1]);
                    emit(r, ring[2], ring[0], ring[1]);
                    if (++r >= count) break;
                }
            } else {
                for (int r = 0;;) {
                    row(ring[1]);
                    row(ring[2]);
                    emit(r, ring[0], ring[1], ring[2]);
                    if (++r >= count) break;
                    row(ring[1]);
                    row(ring[0]);
                    emit(r, ring[2], ring[1], ring[0]);
                    if (++r >= count) break;
                }
            }
        }
    });
}

constexpr size_t kIrMaxLds = 64 * 1024;
constexpr int kIrMaxImages = 12;  // of a workgroup

bool irExpandDwFits(int K, int runRows, int OW, int stride, int PT, int PL) {
    // a window of three rows with at most two above the image reaches into it
    return PT >= 0 && PT <= 2 && PL >= 0 && PL <= 2 && (runRows > 0 ? runRows <= 4 : K > 0 && K % 16 == 0 && K <= 192) && (stride == 1 || stride == 2) && irLds(1, 3, irCellColumns(OW, stride)) <= kIrMaxLds;
}

bool irExpandDwBetter(int64_t wide, int OW, int stride) {
    // Rows of which LDS holds no two windows leave strips of one row, whose pixels are widened three times (stride 2: half of them twice).  At
    // stride 1 two launches are ahead of that: over 97 drawn layers of 511 .. 680 columns they cost 1.5 % of the better one's time, one launch
    // 30 % (1x5x640x16 -> 32 10.7 / 7.1 us, 8x64x600x64 -> 128 46.1 / 38.0).  At stride 2 only where there is little work: over 124 layers of
    // 205 .. 340 columns this line costs 2.8 %, always one launch 10 %, always two 16 % (1x16x320x16 -> 32 9.0 / 7.1, 8x64x340x64 -> 128 23.0 / 30.3).
    if (irLds(1, 3 + stride, irCellColumns(OW, stride)) <= kIrMaxLds) return true;
    return stride == 2 && wide >= 2000000;
}

template <int KS, int S, bool RUNS = false>
static hipError_t launchIr(const IrExpandDwArgs &a, const LaunchCtx &ctx) {
    const long long blocks = (long long)((a.N + a.images - 1) / a.images) * a.strips * ((a.C + kIrChunk - 1) / kIrChunk);
    if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
    THIP_ENQUEUE(ctx, kernelLabel("ir_expand_dw_i8", {KS, S, (int)RUNS}), (ir_expand_dw_i8<KS, S, RUNS>), dim3((unsigned)blocks), dim3(256), irLaunchLds(a), a,
                 makeFastDiv((uint32_t)a.W), makeFastDiv((uint32_t)a.H), makeFastDiv((uint32_t)a.OW), makeFastDiv((uint32_t)a.segments));
    return hipGetLastError();
}

template <int S>
static hipError_t launchIrS(const IrExpandDwArgs &a, const LaunchCtx &ctx) {
    if (a.CKH > 0) return a.CKH <= 2 ? launchIr<1, S, true>(a, ctx) : launchIr<2, S, true>(a, ctx);
    switch ((a.K + 31) / 32) {
    case 1: return launchIr<1, S>(a, ctx);
    case 2: return launchIr<2, S>(a, ctx);
    case 3: return launchIr<3, S>(a, ctx);
    case 4: return launchIr<4, S>(a, ctx);
    case 5: return launchIr<5, S>(a, ctx);
    case 6: return launchIr<6, S>(a, ctx);
    default: return hipErrorInvalidValue;
    }
}

// What follows from `images` and `stripRows`: strips, and segments of a strip's rows so that a wave's 16 columns and its rows fill four waves.
static void irLayout(IrExpandDwArgs *args, int images, int stripRows) {
    IrExpandDwArgs &a = *args;
    a.images = images;
    a.strips = (a.OH + stripRows - 1) / stripRows;
    a.stripRows = stripRows;
    const int columns = a.OW * images;
    a.segments = columns >= 64 ? 1 : 64 / columns;
    if (a.segments > stripRows) a.segments = stripRows;
    a.segmentRows = (stripRows + a.segments - 1) / a.segments;
    a.segments = (stripRows + a.segmentRows - 1) / a.segmentRows;
}

// The time of a launch, us: of a workgroup alone on its CU a start, the cells it clears, the tiles of pixels and the rows of 16 results of a wave; of
// those that share a CU, as many as its registers and LDS hold, each one more; and the rounds of these.  Fitted to 9316 launches of 992 layers, by
// every height of strips and up to 12 images a workgroup: 1 .. 256 images of 4 .. 112 pixels a side, 16 .. 192 channels in and 1 .. 6 times as many wide
// ones, both strides, half of them of mobile networks; `runs` to 140 first layers.  Nine in ten of the launches near a layer's best are within 11 %.  The choice by it
// takes 0.6 % longer than the best, strips of 40 KB in at least 512 workgroups (and images by their rounds) 6 %; in turn with that, 472 other layers took
// 0.946 of the time, three of them more than 3 % longer, 7 % at most.  us, by that / now: 7x7x160 -> 960, 16 images 8.0 / 4.7,
// 10x10x80 -> 480, 14 images 6.0 / 4.4, 14x14x64 -> 384, 126 images 12.0 / 9.3, 16 images 5.7 / 4.9, 32 images 6.04 / 6.02 (two strips of an image before, two images now).
static double irTime(const IrExpandDwArgs &a) {
    struct Cost {
        double launch, start, fill, tile, tileK, row, more, moreFill, moreTile, moreTileK, moreRow;
    };
    constexpr Cost dense{2.72, 1.04, 0.126, 0.092, 0.039, 0.165, 0.59, 0.047, 0.0, 0.074, 0.075}, runs{3.03, 0.90, 0.221, 0.406, 0.241, 0.153, 0.75, 0.0, 0.0, 0.116, 0.073};
    const Cost &c = a.CKH > 0 ? runs : dense;
    const int KS = a.CKH > 0 ? (a.CKH + 1) / 2 : (a.K + 31) / 32, cellRows = irCellRows(a, a.images, a.stripRows);
    int rows = a.strips == 1 ? cellRows - a.PT : cellRows;
    if (rows > a.H) rows = a.H;
    const size_t lds = irLaunchLds(a);
    const int byLds = (int)(160 * 1024 / (lds + 1024)), perCu = byLds < (KS <= 3 ? 4 : 3) ? byLds : KS <= 3 ? 4 : 3;
    const long long blocks = (long long)((a.N + a.images - 1) / a.images) * a.strips * ((a.C + kIrChunk - 1) / kIrChunk), room = 256LL * perCu, rest = (blocks % room + 255) / 256;
    const double tiles = (double)(((long long)a.images * rows * a.W + 31) / 32), items = (a.OW * a.segments * a.images + 15) / 16, kb4 = (double)lds / 4096;
    const double alone = c.start + kb4 * c.fill + ceil(tiles / 4) * (c.tile + c.tileK * (KS - 1)) + ceil(items / 4) * a.segmentRows * c.row;
    const double more = c.more + kb4 * c.moreFill + tiles / 4 * (c.moreTile + c.moreTileK * (KS - 1)) + items / 4 * a.segmentRows * c.moreRow;
    return c.launch + (double)(blocks / room) * (alone + (perCu - 1) * more) + (rest > 0 ? alone + (double)(rest - 1) * more : 0.0);
}

static bool chooseIrLayout(IrExpandDwArgs *args) {
    IrExpandDwArgs &a = *args;
    a.cellCols = irCellColumns(a.OW, a.S);
    // Strips of rows, or whole images, as the estimate has them, heights a fifth apart: neighbouring ones hardly differ.  Both ways end where a
    // launch takes half as long again as the best one: it only gets longer behind that.
    constexpr long long enough = 20000;  // workgroups: strips that make more of them gain nothing
    const long long perStrip = (long long)a.N * ((a.C + kIrChunk - 1) / kIrChunk);
    double best = -1.0;
    int images = 0, stripRows = 0;
    auto consider = [&](int n, int rows) {
        irLayout(&a, n, rows);
        if (irLaunchLds(a) > kIrMaxLds) return true;
        const double time = irTime(a);
        if (best < 0.0 || time < best) {
            best = time;
            images = n;
            stripRows = rows;
        }
        return time < 1.5 * best;
    };
    const int fitting = ((int)(kIrMaxLds / irLds(1, 1, a.cellCols)) - 3) / a.S + 1;
    for (int rows = a.OH < fitting ? a.OH : fitting; rows >= 1;) {
        const int strips = (a.OH + rows - 1) / rows, even = (a.OH + strips - 1) / strips;
        if (!consider(1, even) || (best >= 0.0 && perStrip * strips > enough)) break;
        rows = even > 6 ? even * 4 / 5 : even - 1;
    }
    for (int n = 2; n <= kIrMaxImages && n <= a.N && irLds(n, irCellRows(a, n, a.OH), a.cellCols) <= kIrMaxLds && consider(n, a.OH); n++) {}
    if (best < 0.0) return false;
    irLayout(&a, images, stripRows);
    return true;
}

bool planIrExpandDw(IrExpandDwArgs *args) {
    IrExpandDwArgs &a = *args;
    if (!a.x || !a.wexp || !a.bias1 || !a.scale1 || !a.wdw || !a.bias2 || !a.scale2 || !a.out) return false;
    if (a.N <= 0 || a.H <= 0 || a.W <= 0 || a.C <= 0 || a.C % 16 != 0 || a.OH <= 0 || a.OW <= 0) return false;
    if (!irExpandDwFits(a.K, a.CKH, a.OW, a.S, a.PT, a.PL) || a.Kp < (a.CKH > 0 ? (a.CKH + 1) / 2 * 32 : (a.K + 31) / 32 * 32) || a.Np < (a.C + 31) / 32 * 32) return false;
    if (a.CKH > 0) {
        // the runs of every output pixel start inside the image or its padding (the kernel checks every byte against the image)
        if (a.IH <= 0 || a.IW <= 0 || a.IC <= 0 || a.CS <= 0 || a.CPT < 0 || a.CPL < 0 || a.runBytes <= 0 || a.runBytes > 16 || a.runBytes % a.IC != 0) return false;
        if (a.xBytes != (int64_t)a.N * a.IH * a.IW * a.IC || a.xBytes < 16) return false;
        // a workgroup's images and the padding around them, in 31 bits
        if ((long long)a.IH * a.IW * a.IC > (1LL << 27)) return false;
    } else if ((uintptr_t)a.x & 15) {
        return false;
    }
    if (((uintptr_t)a.wexp | (uintptr_t)a.bias1 | (uintptr_t)a.scale1 | (uintptr_t)a.wdw | (uintptr_t)a.bias2 | (uintptr_t)a.scale2) & 15) return false;
    if (((uintptr_t)a.out) & 3 || (a.CKH == 0 && (long long)a.H * a.W * a.K >= (1LL << 31))) return false;
    // every window starts inside the image or its padding and none needs a row the strip does not make
    if ((a.OH - 1) * a.S - a.PT >= a.H || (a.OW - 1) * a.S - a.PL >= a.W) return false;
    a.cellCols = irCellColumns(a.OW, a.S);
    if ((long long)a.C > kIrMaxChannels) return false;
    if (a.images == 0 && a.stripRows == 0) {
        if (!chooseIrLayout(&a)) return false;
    } else {
        if (a.images < 1 || a.images > kIrMaxImages || a.images > a.N || a.stripRows < 1 || a.stripRows > a.OH || (a.images > 1 && a.stripRows != a.OH)) return false;
        irLayout(&a, a.images, a.stripRows);
        if (irLaunchLds(a) > kIrMaxLds) return false;
    }
    // 128 pixels on, in images, rows and columns
    a.stepImages = a.images > 1 ? 128 / (a.H * a.W) : 0;
    a.stepRows = (128 - a.stepImages * a.H * a.W) / a.W;
    a.stepColumns = (128 - a.stepImages * a.H * a.W) % a.W;
    return true;
}

double irExpandDwTime(IrExpandDwArgs *args) {
    IrExpandDwArgs &a = *args;
    return a.N > 0 && a.H > 0 && a.W > 0 && a.C > 0 && a.OH > 0 && a.OW > 0 && irExpandDwFits(a.K, a.CKH, a.OW, a.S, a.PT, a.PL) && chooseIrLayout(&a) ? irTime(a) : HUGE_VAL;
}

hipError_t launchIrExpandDw(const IrExpandDwArgs &in, const LaunchCtx &ctx) {
    IrExpandDwArgs a = in;
    if (!planIrExpandDw(&a)) return hipErrorInvalidValue;
    return a.S == 1 ? launchIrS<1>(a, ctx) : launchIrS<2>(a, ctx);
}

}  // namespace thip
