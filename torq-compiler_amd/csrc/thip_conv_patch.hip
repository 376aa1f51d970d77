// gfx950 kernel of the int8 convolutions whose weights fit LDS next to a patch of the image: conv_patch_i8, every input pixel brought
// into LDS once for all taps.
#include "thip_kernels_common.h"

namespace thip {

// ---------------------------------------------------------------------------
// conv_patch_i8 (stride 1): a workgroup of eight waves keeps all weights of the convolution in LDS and walks over strips of output rows of an
// image: the strip's input pixels, padding in place, go to LDS; a wave then takes 64 output pixels by all NB * 32 channels at a time,
// both MFMA operands read from LDS, a tap being an offset from the pixel's place in the patch.
//
// Why: the ring kernel addresses the window in memory, so a 3x3 convolution brings every pixel from L2 into LDS nine times, and a tile
// column of 128 brings and multiplies 128 channels where there are 96 (56x56x96 -> 96, 32 images: 130 MB through LDS, 19.0 us; here 34
// MB and 15.3).
//
// What is left is serial in a workgroup, mostly one to a CU: weights and patch into LDS, the MFMA steps, the epilogue.  The sums start at
// the bias and the results are packed as requantPack4 says, as each of the two waves of a SIMD issues a vector instruction in 8 cycles at most (56x56x96: 15.8
// -> 15.4 us).  Weights in parts that are multiplied as they arrive (by LDS-DMA) are slower than all at once: 16.0 against 15.2.
//
// Pixels and weight rows are padded in LDS to pitches of 16-byte units that are no multiple of four, so that the eight
// lanes that a ds_read_b128 serves at a time hit all banks once.
// ---------------------------------------------------------------------------
struct ConvPatchPlan {
    int32_t rows, stripsPerImage, strips;  // output rows of a strip, strips of an image, of all
    int32_t cols;                          // columns of the patch
    int32_t pixelPitch, weightPitch;       // bytes
    int32_t patchBytes;                    // room for a strip's patch
    int32_t steps;                         // of 32 k, an even number
    size_t lds;
};

template <int NB, bool ANY>  // ANY: rows of no whole 16 channels
__global__ __launch_bounds__(512) void conv_patch_i8(IgemmArgs p, ConvPatchPlan q, FastDiv divPixel, FastDiv divCols, FastDiv divOW, FastDiv divRow) {
    extern __shared__ __attribute__((aligned(16))) int8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int fr = lane & 31, half = lane >> 5;
    int8_t *weights = smem, *patch = smem + NB * 32 * q.weightPitch;
    int32_t *ldsBias = (int32_t *)(patch + q.patchBytes), *ldsScale = ldsBias + NB * 32, *tap = ldsScale + NB * 32;
    const int pixelChunks = p.C / 16, rowChunks = 2 * q.steps;
    {
        const int total = NB * 32 * rowChunks;
        for (int i0 = tid; i0 < total; i0 += 512 * 4) {
            v4i v[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int i = i0 + 512 * u < total ? i0 + 512 * u : total - 1;
                const int n = (int)fastDiv((uint32_t)i, divRow);
                v[u] = *(const v4i *)(p.Bp + (size_t)n * p.Kp + (i - n * rowChunks) * 16);
            }
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int i = i0 + 512 * u < total ? i0 + 512 * u : total - 1;
                const int n = (int)fastDiv((uint32_t)i, divRow);
                *(v4i *)(weights + n * q.weightPitch + (i - n * rowChunks) * 16) = v[u];
            }
        }
        if (tid < NB * 32) {
            ldsBias[tid] = p.bias[tid];
            ldsScale[tid] = p.scale[tid];
        }
        // where the 16 channels of k-chunk i lie from a pixel's first tap; past K (zero weights) the first chunk again
        for (int i = tid; i < rowChunks; i += 512) {
            const int t = i * 16 < p.K ? (int)fastDiv((uint32_t)i, divPixel) : 0, c = i * 16 < p.K ? i - t * pixelChunks : 0;
            tap[i] = (t / p.KW * q.cols + t % p.KW) * q.pixelPitch + c * 16;
        }
    }
    const int zp4 = (int)((uint32_t)(p.input_zp & 0xff) * 0x01010101u);
    const WideRequant wrq = wideRequant(p.rq);
    const long long rnd = roundTerm(p.rq.shift);
    for (int strip = (int)blockIdx.x; strip < q.strips; strip += (int)gridDim.x) {
        const int image = strip / q.stripsPerImage, oy0 = (strip - image * q.stripsPerImage) * q.rows;
        const int rows = p.OH - oy0 < q.rows ? p.OH - oy0 : q.rows;
        const int8_t *x = p.A + (size_t)image * p.H * p.W * p.C;
        const int chunks = (rows - 1 + p.KH) * q.cols * pixelChunks;
        __syncthreads();  // the strip before has been read
        for (int i0 = tid; i0 < chunks; i0 += 512 * 8) {
            v4i v[8];
            int at[8];
            bool inside[8];
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const int i = i0 + 512 * u < chunks ? i0 + 512 * u : chunks - 1;
                const int pixel = (int)fastDiv((uint32_t)i, divPixel), c = i - pixel * pixelChunks;
                const int row = (int)fastDiv((uint32_t)pixel, divCols);
                const int iy = oy0 - p.PT + row, ix = pixel - row * q.cols - p.PL;
                inside[u] = (unsigned)iy < (unsigned)p.H && (unsigned)ix < (unsigned)p.W;
                at[u] = pixel * q.pixelPitch + c * 16;
                v[u] = *(const v4i *)(x + (inside[u] ? (uint32_t)((iy * p.W + ix) * p.C + c * 16) : 0u));
            }
#pragma unroll
            for (int u = 0; u < 8; u++) *(v4i *)(patch + at[u]) = inside[u] ? v[u] : v4i{zp4, zp4, zp4, zp4};
        }
        __syncthreads();
        const int pixels = rows * p.OW;
        int8_t *out = (int8_t *)p.out + ((size_t)image * p.OH + oy0) * p.OW * p.N;
        for (int t = wave; t * 64 < pixels; t += 8) {
            const int8_t *base[2];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                int m = t * 64 + 32 * i + fr;
                m = m < pixels ? m : pixels - 1;
                const int oy = (int)fastDiv((uint32_t)m, divOW), ox = m - oy * p.OW;
                base[i] = patch + (oy * q.cols + ox) * q.pixelPitch;
            }
            const int8_t *wbase = weights + fr * q.weightPitch + 16 * half;
            v16i acc[2][NB];
#pragma unroll
            for (int i = 0; i < 2; i++) {
#pragma unroll
                for (int j = 0; j < NB; j++) {
#pragma unroll
                    for (int g = 0; g < 4; g++) {
                        const v4i b4 = *(const v4i *)(ldsBias + 32 * j + 8 * g + 4 * half);
#pragma unroll
                        for (int e = 0; e < 4; e++) acc[i][j][4 * g + e] = b4[e];
                    }
                }
            }
            struct Operands {
                v4i a[2], w[NB];
            };
            // the offset of the step after next is read behind a step's operands: no read waits for another
            int off = tap[half];
            auto load = [&](int s, Operands &o) {
                s = s < q.steps ? s : q.steps - 1;
#pragma unroll
                for (int j = 0; j < NB; j++) o.w[j] = *(const v4i *)(wbase + 32 * j * q.weightPitch + 32 * s);
#pragma unroll
                for (int i = 0; i < 2; i++) o.a[i] = *(const v4i *)(base[i] + off);
                off = tap[2 * (s + 1 < q.steps ? s + 1 : s) + half];
            };
            auto multiply = [&](const Operands &o) {
#pragma unroll
                for (int j = 0; j < NB; j++) {
#pragma unroll
                    for (int i = 0; i < 2; i++) acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(o.w[j], o.a[i], acc[i][j], 0, 0, 0);
                }
            };
            Operands o0, o1;
            load(0, o0);
            // (an even number of steps: a way out between the two would keep the accumulators twice)
            for (int s = 0; s < q.steps; s += 2) {
                load(s + 1, o1);
                multiply(o0);
                load(s + 2, o0);
                multiply(o1);
            }
            withPackMode(wrq, [&](auto tag) {
                constexpr int kMode = decltype(tag)::value;
#pragma unroll
                for (int j = 0; j < NB; j++) {
                    v4i s4[4];
#pragma unroll
                    for (int g = 0; g < 4; g++) s4[g] = *(const v4i *)(ldsScale + 32 * j + 8 * g + 4 * half);
                    const int n = 32 * j + 16 * half;
#pragma unroll
                    for (int i = 0; i < 2; i++) {
                        uint32_t d[4];
#pragma unroll
                        for (int g = 0; g < 4; g++) {
                            const v4i t0 = {acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
                            d[g] = requantPack4<kMode>(t0, s4[g], rnd, p.rq, wrq);
                        }
                        const auto s02 = __builtin_amdgcn_permlane32_swap(d[0], d[2], false, false);
                        const auto s13 = __builtin_amdgcn_permlane32_swap(d[1], d[3], false, false);
                        const int m = t * 64 + 32 * i + fr;
                        const v4i v = {(int)s02[0], (int)s02[1], (int)s13[0], (int)s13[1]};
                        if (m < pixels && n < p.N) {
                            if (ANY) storeRow16(out + (size_t)m * p.N + n, v, p.N - n);
                            else *(v4i *)(out + (size_t)m * p.N + n) = v;
                        }
                        // Two tiles of channels: one after the other they need 123 registers in place of 171, and two workgroups share a CU where
                        // LDS has room (115x115x32 -> 48, batch 26, 24.4 -> 19.3 us; one tile fits anyway, and loses 8 % by it).
                        if (NB == 2) __builtin_amdgcn_sched_barrier(0);
                    }
                }
            });
        }
    }
}

constexpr size_t kPatchMaxLds = 160 * 1024;

// The pitch of rows of `bytes` (whole 16-byte units) in LDS.
static int paddedPitch(int bytes) { return bytes / 16 % 4 == 0 ? bytes + 16 : bytes; }

// Fills the plan; false where the kernel does not take the operands (whole 16-byte pieces of image and weights, results that begin at one, rows of
// which may be of any length: 3x3 115x115x32 -> 40, batch 26, 20.5 us, the ring kernel 21 - 29).
static bool planConvPatch(const IgemmArgs &a, ConvPatchPlan *q) {
    if (!a.A || !a.Bp || !a.bias || !a.scale || !a.out || (((uintptr_t)a.A | (uintptr_t)a.Bp | (uintptr_t)a.out) & 15)) return false;
    if (a.loader != kLoaderWindow || a.out_dtype != kDtypeI8 || a.skip || a.M <= 0 || a.N <= 0 || a.N > 96 || a.C < 16 || a.C % 16 != 0) return false;
    if (a.KH <= 0 || a.KW <= 0 || a.KH > 16 || a.KW > 16 || a.H <= 0 || a.W <= 0 || a.OH <= 0 || a.OW <= 0 || a.SH != 1 || a.SW != 1 || a.PT < 0 || a.PL < 0) return false;
    const long long frame = (long long)a.OH * a.OW, taps = (long long)a.KH * a.KW * a.C;
    if (a.M % frame != 0 || a.K != taps || taps > 8192 || (long long)a.H * a.W * a.C >= (1LL << 31)) return false;
    const long long images = a.M / frame;
    if (a.a_bytes != images * a.H * a.W * a.C) return false;
    const int nb = (a.N + 31) / 32, K64 = (a.K + 63) / 64 * 64;
    if (a.Kp < K64 || a.Kp % 16 != 0 || a.Np < nb * 32) return false;
    q->steps = K64 / 32;
    q->weightPitch = paddedPitch(K64);
    q->pixelPitch = paddedPitch(a.C);
    const long long cols = (long long)a.OW - 1 + a.KW, fixed = (long long)nb * 32 * (q->weightPitch + 8) + K64 / 16 * 4;
    const long long rowBytes = cols * q->pixelPitch, room = (long long)kPatchMaxLds - fixed;
    if (cols > 65536 || rowBytes * a.KH > room) return false;
    q->cols = (int)cols;
    long long most = room / rowBytes - a.KH + 1;
    if (most > a.OH) most = a.OH;
    // As many strips as fill the CUs without beginning another round (a strip for each CU
    // at least, rounded up, left a few CUs two: 605 drawn convolutions took 1.15 times as long, 53x53x64 -> 89, batch 19, 16.4 us in 266 strips, 11.7 in 209).
    const long long rounds = (images * ((a.OH + most - 1) / most) + 255) / 256;
    long long strips = 256 * rounds / images;
    if (strips > a.OH) strips = a.OH;
    q->rows = (int)((a.OH + strips - 1) / strips);
    q->stripsPerImage = (a.OH + q->rows - 1) / q->rows;
    const long long all = images * q->stripsPerImage;
    if (all > 0x3fffffff) return false;
    q->strips = (int)all;
    q->patchBytes = (int)((q->rows - 1 + a.KH) * rowBytes);
    q->lds = (size_t)(fixed + q->patchBytes);
    return true;
}

// Against the ring kernel's own tile, us (ring / patch), 3x3 unless it says 5x5, stride 1:
//   56x56x96 -> 96, batch 32 19.0 / 15.3; 112x112x32 -> 64, 32 24.3 / 17.4; 160x160x32 -> 16, 32 33.4 / 18.1; 80x80x80 -> 48, 32 21.3 / 17.3;
//   127x127x96 -> 80, 5 17.4 / 13.4; 28x28x96 -> 96, 64 11.4 / 10.7; 5x5 160x160x16 -> 32, 8 14.0 / 8.9; 5x5 64x64x48 -> 32, 16 11.6 / 7.8
// and where the rule below says no:
//   few pixels, whose strips are few or low   30x30x96 -> 96, 32 8.2 / 9.8; 160x160x64 -> 64, 2 (two rows each) 7.6 / 8.7
//   many channels out, few taps, many in      56x56x48 -> 128, 20 9.8 / 12.0; 2x2 100x100x96 -> 64, 20 15.2 / 21.5; 64x64x128 -> 64, 32 19.2 / 22.6
//   a second round of low strips              5x5 46x46x80 -> 33, 27 16.7 / 24.9; 7x7 40x40x80 -> 7, 40 26.0 / 42.4; 5x5 105x105x64 -> 53, 7 19.1 / 21.4
//   rows that only rounding up makes three    104x104x16 -> 45, 5 6.2 / 7.5
//   ragged results in two rounds or more      5x5 122x122x96 -> 28, 6 21.3 / 25.0; 93x93x112 -> 18, 9 23.4 / 26.8; 7x7 73x73x64 -> 5, 22 26.4 / 38.8
//   where the ring kernel's tiles are one     (43 drawn ones: up to 400 tiles 0.89 of its speed, to 512 1.00 in two rounds and 0.85 in three, beyond 1.21; whole results 1.06 and more)
// Over 605 drawn ones (16 .. 112 channels in, 1 .. 96 out, windows of 3, 5 and 7) the choice costs 1.1 % of the better one's time, always the ring kernel 20 %, always this one 3 %.
bool convPatchBetter(const IgemmArgs &a) {
    ConvPatchPlan q;
    if (a.C > 112 || a.KH * a.KW < 9 || a.M < 49152 || !planConvPatch(a, &q)) return false;
    const int rounds = (q.strips + 255) / 256;
    if (q.rows * a.KW < 9 || (long long)(a.M / a.OW) * a.KW < 1600LL * rounds) return false;
    if (rounds == 1) return true;
    return (q.rows >= a.KH || q.rows * a.OW > 160) && (a.N <= 32 || q.rows >= (a.KH < 4 ? a.KH : 4)) && (a.N % 16 == 0 || a.M > (rounds == 2 ? 102400 : 131072));
}

template <int NB, bool ANY>
static hipError_t launchPatch(const IgemmArgs &a, const ConvPatchPlan &q, const LaunchCtx &ctx) {
    auto kernel = conv_patch_i8<NB, ANY>;
    static std::once_flag once;
    static hipError_t configured = hipSuccess;
    std::call_once(once, [&] { configured = hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kPatchMaxLds); });
    if (configured != hipSuccess) return configured;
    const int perCu = (int)(kPatchMaxLds / q.lds) < 2 ? 1 : 2, grid = q.strips < 256 * perCu ? q.strips : 256 * perCu;
    THIP_ENQUEUE(ctx, kernelLabel("conv_patch_i8", {NB, (int)ANY}), kernel, dim3((unsigned)grid), dim3(512), q.lds, a, q, makeFastDiv((uint32_t)(a.C / 16)), makeFastDiv((uint32_t)q.cols),
                 makeFastDiv((uint32_t)a.OW), makeFastDiv((uint32_t)(2 * q.steps)));
    return hipGetLastError();
}

hipError_t launchConvPatch(const IgemmArgs &a, const LaunchCtx &ctx) {
    ConvPatchPlan q;
    if (!planConvPatch(a, &q)) return hipErrorInvalidValue;
    const bool any = a.N % 16 != 0;
    switch ((a.N + 31) / 32) {
    case 1: return any ? launchPatch<1, true>(a, q, ctx) : launchPatch<1, false>(a, q, ctx);
    case 2: return any ? launchPatch<2, true>(a, q, ctx) : launchPatch<2, false>(a, q, ctx);
    default: return any ? launchPatch<3, true>(a, q, ctx) : launchPatch<3, false>(a, q, ctx);
    }
}

}  // namespace thip
