// gfx950 kernel of the front half of an inverted-residual block: the pointwise convolution that widens the channels and the
// 3 x 3 depthwise convolution behind it as one launch, the widened image never leaving LDS.
#include "thip_inverted_residual.h"
#include "thip_kernels_common.h"

namespace thip {

// The requant tails that need 32-bit arithmetic only (withRequantMode without its 64-bit one; the planner keeps such records
// apart).
template <typename F>
__device__ __forceinline__ void withNarrowRequantMode(const WideRequant &w, F &&f) {
    if (w.plain) f(std::integral_constant<int, 2>{});
    else if (w.preOnly) f(std::integral_constant<int, 3>{});
    else f(std::integral_constant<int, 1>{});
}

// Columns of cells under the windows of one output row, in whole column groups of the threads.
static inline int irCellColumns(int OW, int S) { return S == 1 ? 2 * ((OW + 1) / 2) + 2 : 2 * OW + 1; }

// ---------------------------------------------------------------------------
// ir_expand_dw_i8: a workgroup makes 32 channels of a strip of output rows of one image.
//
// Phase 1, the pointwise convolution: the strip's input pixels are rows of a dense [pixels][K] matrix; a wave takes 32 of
// them at a time straight from memory in MFMA operand layout (K <= 192: at most six loads per lane, prefetched one tile ahead), the
// 32 channels' weights stay in registers, and the requantised bytes go to LDS as cells [row][column][32 channels]. Cells outside the
// image hold the depthwise op's zero point.
// RUNS: a convolution over few channels instead (the first layer of an image network): K is one 16-byte run per window row, and the pixels are gathered from the image.
// Phase 2, the depthwise convolution: a thread owns four channels of two output columns (one at stride 2) and walks down rows:
// per input row three to four dwords from LDS, a byte transpose so that a dword holds one channel at neighbouring
// columns, and one v_dot4_i32_i8 per window row, channel and output. No address clamping and no padding selects are left in the loop.
//
// Why: apart, the two launches write the widened image and read it back (3.3 MB per image of a 224 x 224 mobile network, 6.7 MB of
// its 11 MB of traffic), and at small batches each costs a dependent launch. Bound by the vector pipes: about 5 instructions
// per widened byte and 9 per depthwise byte, most of them the requants.  Measured, us, the two launches / this one:
//   batch 256  112x112x16 -> 96 stride 2 151 / 99, 56x56x32 -> 144 80 / 69, 28x28x32 -> 192 42 / 26, 14x14x96 -> 576 34 / 25
//   batch 32   112x112x16 -> 96 stride 2 30.9 / 18.5, 56x56x32 -> 144 24.2 / 15.9, 14x14x96 -> 576 10.0 / 8.0
//   batch 1    56x56x32 -> 144 6.8 / 4.8, 14x14x96 -> 576 6.7 / 3.8, 7x7x160 -> 960 6.8 / 4.1
// and since, with pixels and cells reached by a walk instead of divisions and 32-bit offsets of the results (in a trace of the network,
// batch 256): 224x224x3 -> 112x112x32 104.9 -> 94.9, 112x112x16 -> 96 stride 2 115.1 -> 108.6, 56x56x32 -> 144 80.0 -> 77.2. The busy
// cycles are 90 % vector instructions there; more tiles prefetched, or strips of 26, 32 or 53 KB, change nothing.
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
    const int images = part.images, oy0 = part.oy0, rows = part.rows, iyFirst = part.iyFirst, iyLo = part.iyLo, cellRows = part.cellRows, pixels = part.pixels;
    const int cellCols = p.cellCols;

    // ---- phase 1 ----
    const int fr = lane & 31, half = lane >> 5;
    v4i w[KS];
    v16i bias;
    int scale[16];
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
                scale[4 * q + e] = s4[e];
            }
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
    IrWalk cell = walkFrom(cellImageBytes, cellRowBytes, kIrPitch, (iyLo - iyFirst) * cellRowBytes + p.PL * kIrPitch + 4 * half);
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
        const int words = images * cellRows * cellCols * (kIrPitch / 4);
        for (int i = tid * 4; i < words; i += 1024) *(v4i *)(cells + (size_t)i * 4) = v4i{zp4, zp4, zp4, zp4};  // LDS is rounded up to 16 bytes
    }
    __syncthreads();
    const WideRequant w1 = wideRequant(p.rq1);
    withNarrowRequantMode(w1, [&](auto tag) {
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
#pragma unroll
            for (int q = 0; q < 4; q++) {
                int32_t v[4];
#pragma unroll
                for (int e = 0; e < 4; e++) v[e] = requantT0<kMode>(acc[4 * q + e], scale[4 * q + e], 0, p.rq1, w1);
                *(uint32_t *)(dst + 8 * q) = packBytes(v[0], v[1], v[2], v[3]);
            }
        };
        for (int t = wave; t < tiles; t += 8) {
            loadTile(a1);
            computeTile(t, a0);
            if (t + 4 >= tiles) break;
            loadTile(a0);
            computeTile(t + 4, a1);
        }
    });
    __syncthreads();

    // ---- phase 2 ----
    constexpr int P = S == 1 ? 2 : 1;  // output columns of a thread
    const int c4 = tid & 7, slot = tid >> 3;
    if (ch0 + 4 * c4 >= p.C) return;
    const int ch = ch0 + 4 * c4;
    int wk[3][4], wks[3][4];
#pragma unroll
    for (int kh = 0; kh < 3; kh++) {
        const v4i w4 = *(const v4i *)(p.wdw + (size_t)kh * p.C + ch);
#pragma unroll
        for (int c = 0; c < 4; c++) {
            wk[kh][c] = w4[c];
            wks[kh][c] = (int)((uint32_t)w4[c] << 8);
        }
    }
    const v4i bias2 = *(const v4i *)(p.bias2 + ch), scale2 = *(const v4i *)(p.scale2 + ch);
    const WideRequant w2 = wideRequant(p.rq2);
    const int colGroups = (p.OW + P - 1) / P, items = colGroups * p.segments * images;
    const int rowBytes = cellCols * kIrPitch;
    int8_t *out = p.out + ((size_t)n * p.OH + oy0) * p.OW * p.C;
    withNarrowRequantMode(w2, [&](auto tag) {
        constexpr int kMode = decltype(tag)::value;
        for (int item = slot; item < items; item += 32) {
            int seg = 0, image = 0, j = item;
            if (p.segments * p.images > 1) {
                seg = (int)fastDiv((uint32_t)item, divCols);
                j -= seg * colGroups;
            }
            if (p.images > 1) {
                image = (int)fastDiv((uint32_t)seg, divSegments);
                seg -= image * p.segments;
            }
            const int oyA = seg * p.segmentRows, oyB = oyA + p.segmentRows < rows ? oyA + p.segmentRows : rows;
            if (oyA >= oyB) continue;
            const int ox = j * P;
            const int8_t *src = cells + ((image * cellRows + oyA * S) * cellCols + ox * S) * kIrPitch + 4 * c4;
            uint32_t dst = (uint32_t)(((image * p.OH + oyA) * p.OW + ox) * p.C + ch);
            const bool second = P == 2 && ox + 1 < p.OW;
            uint32_t ring[3][4];
            auto row = [&](uint32_t(&o)[4]) {
                const uint32_t x0 = *(const uint32_t *)src, x1 = *(const uint32_t *)(src + kIrPitch), x2 = *(const uint32_t *)(src + 2 * kIrPitch);
                const uint32_t x3 = S == 1 ? *(const uint32_t *)(src + 3 * kIrPitch) : x2;  // stride 2: its weight is zero
                const uint32_t lo01 = __builtin_amdgcn_perm(x1, x0, 0x05010400u), hi01 = __builtin_amdgcn_perm(x1, x0, 0x07030602u);
                const uint32_t lo23 = S == 1 ? __builtin_amdgcn_perm(x3, x2, 0x05010400u) : x2, hi23 = S == 1 ? __builtin_amdgcn_perm(x3, x2, 0x07030602u) : x2;
                o[0] = __builtin_amdgcn_perm(lo23, lo01, S == 1 ? 0x05040100u : 0x0c040100u);
                o[1] = __builtin_amdgcn_perm(lo23, lo01, S == 1 ? 0x07060302u : 0x0c050302u);
                o[2] = __builtin_amdgcn_perm(hi23, hi01, S == 1 ? 0x05040100u : 0x0c060100u);
                o[3] = __builtin_amdgcn_perm(hi23, hi01, S == 1 ? 0x07060302u : 0x0c070302u);
                src += rowBytes;
            };
            auto emit = [&](const uint32_t(&r0)[4], const uint32_t(&r1)[4], const uint32_t(&r2)[4]) {
                int32_t v[P][4];
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    int32_t acc = __builtin_amdgcn_sdot4((int)r0[c], wk[0][c], bias2[c], false);
                    acc = __builtin_amdgcn_sdot4((int)r1[c], wk[1][c], acc, false);
                    acc = __builtin_amdgcn_sdot4((int)r2[c], wk[2][c], acc, false);
                    v[0][c] = requantT0<kMode>(acc, scale2[c], 0, p.rq2, w2);
                    if (P == 2) {
                        acc = __builtin_amdgcn_sdot4((int)r0[c], wks[0][c], bias2[c], false);
                        acc = __builtin_amdgcn_sdot4((int)r1[c], wks[1][c], acc, false);
                        acc = __builtin_amdgcn_sdot4((int)r2[c], wks[2][c], acc, false);
                        v[P - 1][c] = requantT0<kMode>(acc, scale2[c], 0, p.rq2, w2);
                    }
                }
                *(uint32_t *)(out + dst) = packBytes(v[0][0], v[0][1], v[0][2], v[0][3]);
                if (second) *(uint32_t *)(out + (dst + (uint32_t)p.C)) = packBytes(v[P - 1][0], v[P - 1][1], v[P - 1][2], v[P - 1][3]);
                dst += (uint32_t)(p.OW * p.C);
            };
            if (S == 1) {
                row(ring[0]);
                row(ring[1]);
                for (int oy = oyA;;) {
                    row(ring[2]);
                    emit(ring[0], ring[1], ring[2]);
                    if (++oy >= oyB) break;
                    row(ring[0]);
                    emit(ring[1], ring[2], ring[0]);
                    if (++oy >= oyB) break;
                    row(ring[1]);
                    emit(ring[2], ring[0], ring[1]);
                    if (++oy >= oyB) break;
                }
            } else {
                row(ring[0]);
                for (int oy = oyA;;) {
                    row(ring[1]);
                    row(ring[2]);
                    emit(ring[0], ring[1], ring[2]);
                    if (++oy >= oyB) break;
                    row(ring[1]);
                    row(ring[0]);
                    emit(ring[2], ring[1], ring[0]);
                    if (++oy >= oyB) break;
                }
            }
        }
    });
}

static size_t irLds(int images, int cellRows, int cellCols) { return ((size_t)images * cellRows * cellCols * kIrPitch + 15) / 16 * 16; }
constexpr size_t kIrMaxLds = 64 * 1024;

bool irExpandDwFits(int K, int runRows, int OW, int stride, int PT, int PL) {
    // a window of three rows with at most two above the image reaches into it
    return PT >= 0 && PT <= 2 && PL >= 0 && PL <= 2 && (runRows > 0 ? runRows <= 4 : K > 0 && K % 16 == 0 && K <= 192) && (stride == 1 || stride == 2) && irLds(1, 3, irCellColumns(OW, stride)) <= kIrMaxLds;
}

template <int KS, int S, bool RUNS = false>
static hipError_t launchIr(const IrExpandDwArgs &a, const LaunchCtx &ctx) {
    const long long blocks = (long long)((a.N + a.images - 1) / a.images) * a.strips * ((a.C + kIrChunk - 1) / kIrChunk);
    if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
    THIP_ENQUEUE(ctx, kernelLabel("ir_expand_dw_i8", {KS, S, (int)RUNS}), (ir_expand_dw_i8<KS, S, RUNS>), dim3((unsigned)blocks), dim3(256), irLds(a.images, irCellRows(a, a.images, a.stripRows), a.cellCols), a,
                 makeFastDiv((uint32_t)a.W), makeFastDiv((uint32_t)a.H), makeFastDiv((uint32_t)(S == 1 ? (a.OW + 1) / 2 : a.OW)), makeFastDiv((uint32_t)a.segments));
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

bool planIrExpandDw(IrExpandDwArgs *args) {
    IrExpandDwArgs &a = *args;
    if (!a.x || !a.wexp || !a.bias1 || !a.scale1 || !a.wdw || !a.bias2 || !a.scale2 || !a.out) return false;
    if (a.N <= 0 || a.H <= 0 || a.W <= 0 || a.C <= 0 || a.C % 16 != 0 || a.OH <= 0 || a.OW <= 0) return false;
    if (!irExpandDwFits(a.K, a.CKH, a.OW, a.S, a.PT, a.PL) || a.Kp < (a.CKH > 0 ? (a.CKH + 1) / 2 * 32 : (a.K + 31) / 32 * 32) || a.Np < (a.C + 31) / 32 * 32) return false;
    if (a.CKH > 0) {
        // the runs of every output pixel start inside the image or its padding (the kernel checks every byte against the image)
        if (a.IH <= 0 || a.IW <= 0 || a.IC <= 0 || a.CS <= 0 || a.CPT < 0 || a.CPL < 0 || a.runBytes <= 0 || a.runBytes > 16 || a.runBytes % a.IC != 0) return false;
        if (a.xBytes != (int64_t)a.N * a.IH * a.IW * a.IC || a.xBytes < 16) return false;
        // a workgroup's eight images and the padding around them, in 31 bits
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
    // Four workgroups per CU (160 KB of LDS, 16 waves) overlap one another's phases: strips as high as 40 KB of cells hold
    // (56x56x32 -> 144, 256 images: 79 us at 20 KB, whose strips make more rows twice, 69 at 40, 76 at 64), lower where that
    // leaves fewer than two workgroups per CU (14x14x96 -> 576, 32 images: 8.0 us with at least 512, 9.1 with 1024), and down
    // to four rows; images that leave room share a workgroup (7x7x160 -> 960, 256 images: 37.3 us one by one, 17.3 by eight).
    // Images that share cost no rows twice, so where the registers (K <= 64) let eight workgroups run on a CU they get 20 KB each
    // (14x14x64 -> 384, 256 images: 23.4 -> 19.5 us; with K = 96 18.6 -> 21.0 at stride 2, with 160 18.7 -> 20.0, the other way).
    constexpr size_t ldsAim = 40 * 1024;
    constexpr long long wgAim = 512;
    const long long perStrip = (long long)a.N * ((a.C + kIrChunk - 1) / kIrChunk);
    int strips = 1;
    auto rowsOf = [&](int s) { return (a.OH + s - 1) / s; };
    auto lds = [&](int images, int s) { return irLds(images, irCellRows(a, images, rowsOf(s)), a.cellCols); };
    // phase 1's rounds of a workgroup's four waves: where not even every second CU has a workgroup they are the launch's time
    auto rounds = [&](int s) { return (((rowsOf(s) - 1) * a.S + 3) * a.W + 127) / 128; };
    while (rowsOf(strips) > 1 && (lds(1, strips) > ldsAim || (perStrip * strips < wgAim && rowsOf(strips) > 4) || (perStrip * strips < 128 && rounds(strips) > 2))) strips++;
    a.stripRows = rowsOf(strips);
    a.strips = (a.OH + a.stripRows - 1) / a.stripRows;
    a.images = 1;
    if (a.strips == 1) {
        const size_t aim = a.CKH == 0 && a.K <= 64 ? ldsAim / 2 : ldsAim;
        while (a.images < 8 && lds(a.images + 1, 1) <= aim && perStrip / (a.images + 1) >= 1024) a.images++;
    }
    // 128 pixels on, in images, rows and columns
    a.stepImages = a.images > 1 ? 128 / (a.H * a.W) : 0;
    a.stepRows = (128 - a.stepImages * a.H * a.W) / a.W;
    a.stepColumns = (128 - a.stepImages * a.H * a.W) % a.W;
    const int P = a.S == 1 ? 2 : 1, columns = (a.OW + P - 1) / P * a.images;
    a.segments = columns >= 32 ? 1 : 32 / columns;
    if (a.segments > a.stripRows) a.segments = a.stripRows;
    a.segmentRows = (a.stripRows + a.segments - 1) / a.segments;
    a.segments = (a.stripRows + a.segmentRows - 1) / a.segmentRows;
    return true;
}

hipError_t launchIrExpandDw(const IrExpandDwArgs &in, const LaunchCtx &ctx) {
    IrExpandDwArgs a = in;
    if (!planIrExpandDw(&a)) return hipErrorInvalidValue;
    return a.S == 1 ? launchIrS<1>(a, ctx) : launchIrS<2>(a, ctx);
}

}  // namespace thip
