// gfx950 kernel of the small int8 GEMMs and convolutions, those that a tile per workgroup leaves most of the chip idle for:
// igemm_direct_i8, operands straight from memory into MFMA registers, K split over the waves of a workgroup.
#include "thip_kernels_common.h"

namespace thip {

// ---------------------------------------------------------------------------
// igemm_direct_i8: the records of igemm_dense_i8 (dense operand, or a window over C % 16 == 0 channels addressed in place), one
// 32 x 32 tile per workgroup of NW waves.
//
// The ring kernel walks K one k-tile at a time, 0.2 us each (DMA, barrier, LDS, MFMA), so that a tile's time is its
// K whatever else the chip does: 49 x 960 -> 160 is three workgroups and 5.0 us, 28 x 5536 -> 144 12.4 us.  Here the waves
// take turns at four MFMA steps of 32 k, the 128 bytes of a cache line; a lane loads its 16 bytes of a pixel and of a weight row
// per step, all four steps before the first MFMA; nothing is staged and no barrier passed until the partial sums meet in LDS.  Four waves then finish four accumulator registers (four
// neighbouring channels of a pixel) each: sum in wave order, requant, residual add, one dword per lane.
//
// Bound by latency: one or two memory round trips, the LDS exchange and the launch.  A tile brings 64 bytes per k where a 64 x 64
// tile brings 32 per output: taken up to two workgroups per CU only (igemmDirectBetter).
//
// RAGGED: rows (pixels) of no whole 16-byte chunks, as they are in memory.  A row's last chunk reaches into the next row, where the weights have zeros; the
// last row's is read at the tensor's end and shifted.  1: rows of whole dwords, which a 16-byte load takes at no loss (1583 x 4184 -> 23 8.3 us;
// rows copied to whole chunks first 15.7).  2: any other, whose chunks are put together from the dwords they lie in: a wave's 16-byte load at odd
// addresses takes the CU 190 cycles in place of 30 (3 x 5637 -> 567 11.9 -> 9.0, 5x5 19x19x387 -> 134 31.7 -> 19.7).
// ---------------------------------------------------------------------------
template <bool WINDOW, int NW, int RAGGED>
__global__ __launch_bounds__(NW * 64) void igemm_direct_i8(IgemmArgs p, FastDiv divC, FastDiv divKW, FastDiv divFrame, FastDiv divOW) {
    constexpr int U = 4;  // steps in flight
    __shared__ v4i partial[NW][4][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int fr = lane & 31, half = lane >> 5;
    const int tilesM = (p.M + 31) / 32;
    const int m0 = ((int)blockIdx.x % tilesM) * 32, n0 = ((int)blockIdx.x / tilesM) * 32;
    const int mOwn = m0 + fr, m = mOwn < p.M ? mOwn : p.M - 1;
    // what the epilogue reads from memory, issued with the operands
    const int n = n0 + 8 * (wave & 3) + 4 * half;
    const v4i bias = *(const v4i *)(p.bias + n), scale = *(const v4i *)(p.scale + n);  // padded to Np
    const bool whole = n + 4 <= p.N;
    uint32_t other = 0;
    if (p.skip && whole) other = *(const uint32_t *)(p.skip + (size_t)m * p.N + n);

    int y0 = 0, x0 = 0;
    uint32_t imageRow = 0;
    const int pixel = RAGGED ? p.row_bytes : p.C;
    const int8_t *arow = p.A + (WINDOW || RAGGED ? 0 : (size_t)m * p.K);
    const uint32_t rowAt = RAGGED && !WINDOW ? (uint32_t)m * (uint32_t)pixel : 0u, last = RAGGED ? (uint32_t)p.a_bytes - 16u : 0u;
    if (WINDOW) {
        const int image = (int)fastDiv((uint32_t)m, divFrame), rem = m - image * (p.OH * p.OW);
        const int oy = (int)fastDiv((uint32_t)rem, divOW), ox = rem - oy * p.OW;
        y0 = oy * p.SH - p.PT;
        x0 = ox * p.SW - p.PL;
        imageRow = (uint32_t)image * (uint32_t)p.H;
    }
    const int8_t *wrow = p.Bp + (size_t)(n0 + fr) * p.Kp + 16 * half;
    const int zp4 = (int)((uint32_t)(p.input_zp & 0xff) * 0x01010101u);
    const int steps = (p.K + 31) / 32;
    // A chunk of RAGGED rows is asked for with load and finished with finish.  One that would end behind A is read before its place, at A's end.  RAGGED 2,
    // rows that are no whole dwords: read from the dword that it begins in, and the dword behind it (or A's last) too.
    struct Chunk {
        v4i v;
        uint32_t off, behind;
    };
    auto load = [&](Chunk &c, uint32_t off) {
        if (RAGGED) {
            uint32_t at = off < last ? off : last;
            if (RAGGED == 2) {
                at &= ~3u;
                c.behind = ((const UnalignedU32 *)(arow + (at < last - 4u ? at + 16u : last + 12u)))->v;
            }
            c.off = off;
            c.v = ((const UnalignedV4 *)(arow + at))->v;
        } else {
            c.v = *(const v4i *)(arow + off);
        }
    };
    auto finish = [&](const Chunk &c) {
        if (!RAGGED) return c.v;
        const uint32_t at = c.off < last ? c.off : last;
        v4i x = c.v;
        if (RAGGED == 2) {
            // at A's end the dword was read up to four bytes early
            const uint32_t base = at & ~3u, early = base + 4u > last ? base + 4u - last : 0u;
            const uint32_t w[5] = {(uint32_t)x[0], (uint32_t)x[1], (uint32_t)x[2], (uint32_t)x[3], (uint32_t)((uint64_t)c.behind >> (8 * early))};
#pragma unroll
            for (int e = 0; e < 4; e++) x[e] = (int)__builtin_amdgcn_alignbyte(w[e + 1], w[e], at & 3u);
        }
        if (c.off != at) x = fixRun16(x, (int)(c.off - at), 0, 16, 0u);
        return x;
    };
    v16i acc;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = 0;
    for (int s0 = wave * U; s0 < steps; s0 += NW * U) {
        Chunk a[U];
        v4i w[U];
        bool inside[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            // a step past the end re-reads the last one and is not used; a chunk past K (zero weights) re-reads the row's first
            const int s = s0 + u < steps ? s0 + u : steps - 1;
            const int k = 32 * s + 16 * half, kk = k < p.K ? k : 0;
            if (WINDOW) {
                const int tap = (int)fastDiv((uint32_t)kk, divC), c = kk - tap * p.C;
                const int kh = (int)fastDiv((uint32_t)tap, divKW), kw = tap - kh * p.KW;
                const int y = y0 + kh, x = x0 + kw;
                inside[u] = (unsigned)y < (unsigned)p.H && (unsigned)x < (unsigned)p.W;
                const uint32_t off = inside[u] ? ((imageRow + (uint32_t)y) * (uint32_t)p.W + (uint32_t)x) * (uint32_t)pixel + (uint32_t)c : 0u;
                load(a[u], off);
            } else {
                inside[u] = true;
                load(a[u], rowAt + (uint32_t)kk);
            }
            w[u] = *(const v4i *)(wrow + 32 * s);
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (s0 + u >= steps) break;
            v4i x = finish(a[u]);
            if (WINDOW) {
#pragma unroll
                for (int d = 0; d < 4; d++) x[d] = inside[u] ? x[d] : zp4;
            }
            acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(w[u], x, acc, 0, 0, 0);  // register 4 q + e: channel 8 q + 4 half + e of pixel fr
        }
    }
#pragma unroll
    for (int q = 0; q < 4; q++) partial[wave][q][lane] = v4i{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
    __syncthreads();
    if (wave >= 4) return;
    v4i sum = partial[0][wave][lane];
#pragma unroll
    for (int o = 1; o < NW; o++) sum += partial[o][wave][lane];
    if (mOwn >= p.M || n >= p.N) return;
    const long long rnd = roundTerm(p.rq.shift);
    const WideRequant wrq = wideRequant(p.rq);
    int32_t v[4];
    withRequantMode(wrq, [&](auto tag) {
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = requantT0<decltype(tag)::value>((int32_t)((uint32_t)sum[e] + (uint32_t)bias[e]), scale[e], rnd, p.rq, wrq);
    });
    if (p.skip) {
        const long long addRnd = roundTerm(p.arq.shift);
        const int32_t wm = p.add_skip_first ? p.add_w1 : p.add_w0, wo = p.add_skip_first ? p.add_w0 : p.add_w1;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int32_t b = whole ? (int32_t)(int8_t)(other >> (8 * e)) : (n + e < p.N ? (int32_t)p.skip[(size_t)m * p.N + n + e] : 0);
            v[e] = requant(v[e] * wm + b * wo, p.add_bias, p.add_scale, addRnd, p.arq);
        }
    }
    const size_t at = (size_t)m * p.N + n;
    if (p.out_dtype == kDtypeI8 && whole) {
        ((UnalignedU32 *)((int8_t *)p.out + at))->v = packBytes(v[0], v[1], v[2], v[3]);
    } else {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            if (n + e < p.N) storeElem(p.out, at + e, v[e], p.out_dtype);
        }
    }
}

static long long directTiles(const IgemmArgs &a) { return (long long)((a.M + 31) / 32) * ((a.N + 31) / 32); }

// What the kernel assumes of its operands, their addresses' alignment included (the ring kernel stores at any).
static bool directTakes(const IgemmArgs &a) {
    const bool window = a.loader == kLoaderWindow;
    if (!a.A || !a.Bp || !a.bias || !a.scale || !a.out || a.M <= 0 || a.N <= 0 || a.K <= 0 || (!window && a.loader != kLoaderDense)) return false;
    if (a.K % 16 != 0 || a.Kp < (a.K + 31) / 32 * 32 || a.Np < (a.N + 31) / 32 * 32 || a.Kp % 16 != 0) return false;
    if ((((uintptr_t)a.Bp | (uintptr_t)a.bias | (uintptr_t)a.scale) & 15) || (((uintptr_t)a.A & 15) && a.row_bytes == 0)) return false;
    if (a.out_dtype < kDtypeI8 || a.out_dtype > kDtypeI32 || ((uintptr_t)a.out & 3) || (a.skip && (((uintptr_t)a.skip & 3) || a.N % 4 != 0 || a.out_dtype != kDtypeI8))) return false;
    if (window) {
        if (a.C < 16 || a.C % 16 != 0 || a.KH <= 0 || a.KW <= 0 || a.H <= 0 || a.W <= 0 || a.OH <= 0 || a.OW <= 0 || a.SH <= 0 || a.SW <= 0 || a.PT < 0 || a.PL < 0) return false;
        if (a.M % (a.OH * a.OW) != 0 || (long long)a.K != (long long)a.KH * a.KW * a.C) return false;
        if (a.a_bytes != (long long)(a.M / (a.OH * a.OW)) * a.H * a.W * (a.row_bytes ? a.row_bytes : a.C) || a.a_bytes >= (1LL << 32)) return false;
    }
    if (a.row_bytes != 0) {
        // a row's last chunk reaches into the next one; behind the last row its load begins earlier
        if (a.row_bytes < 0 || (a.row_bytes + 15) / 16 * 16 != a.C || a.a_bytes < 20 || a.a_bytes >= (1LL << 31)) return false;
        if (!window && (a.K != a.C || a.a_bytes != (long long)a.M * a.row_bytes)) return false;
    }
    return true;
}

// Against the ring kernel's own tile, us (tiles; ring / direct):
//   dense   49 x 960 -> 160 (10) 4.2 / 3.4, 1429 x 1344 -> 48 (90) 5.0 / 4.1, 400 x 512 -> 512 (208) 3.7 / 3.6, 450 x 80 -> 752 (360)
//           2.9 / 3.2, 28 x 5536 -> 144 (5) 12.4 / 8.6, 40 x 8192 -> 2048 (128) 17.6 / 18.1
//   window  3x3 7x7x304 -> 64, batch 4 (14) 11.4 / 5.5, stride 2 64x64x256 -> 8, batch 8 (256) 11.3 / 6.9, stride 2 142x142x144 -> 8,
//           batch 3 (473) 8.3 / 6.0, 5x5 32x32x32 -> 64, batch 15 (960) 6.8 / 6.1, 14x14x512 -> 512, batch 8 (784) 18.0 / 33.4
// so: up to a workgroup per CU, or, where the ring has to address a window, up to the 50 MB that its tiles' operands may be together.
bool igemmDirectBetter(const IgemmArgs &a) {
    if (!directTakes(a)) return false;
    const long long tiles = directTiles(a), bytes = tiles * 64 * a.K;
    return a.loader == kLoaderWindow ? tiles <= 1024 && bytes <= 50000000 : tiles <= 256 && bytes <= 25000000;
}

template <bool WINDOW, int NW, int RAGGED>
static hipError_t launchDirect(const IgemmArgs &a, const LaunchCtx &ctx) {
    const long long tiles = directTiles(a);
    THIP_ENQUEUE(ctx, (RAGGED ? kernelLabel("igemm_direct_i8", {(int)WINDOW, NW, RAGGED}) : kernelLabel("igemm_direct_i8", {(int)WINDOW, NW})), (igemm_direct_i8<WINDOW, NW, RAGGED>), dim3((unsigned)tiles), dim3(NW * 64), 0, a,
                 makeFastDiv((uint32_t)(WINDOW ? a.C : 1)), makeFastDiv((uint32_t)(WINDOW ? a.KW : 1)), makeFastDiv((uint32_t)(WINDOW ? a.OH * a.OW : 1)),
                 makeFastDiv((uint32_t)(WINDOW ? a.OW : 1)));
    return hipGetLastError();
}

hipError_t launchIgemmDirect(const IgemmArgs &a, const LaunchCtx &ctx) {
    const bool window = a.loader == kLoaderWindow;
    if (!directTakes(a)) return hipErrorInvalidValue;
    // eight waves while that leaves a CU two workgroups (3x3 56x56x64 -> 64: 3.4 us against 3.8 with four), four beyond (142x142x144
    // -> 8, batch 3: 6.0 against 6.8)
    const bool few = directTiles(a) <= 400;
    if (a.row_bytes % 4 != 0) {
        if (window) return few ? launchDirect<true, 8, 2>(a, ctx) : launchDirect<true, 4, 2>(a, ctx);
        return few ? launchDirect<false, 8, 2>(a, ctx) : launchDirect<false, 4, 2>(a, ctx);
    }
    if (a.row_bytes != 0) {
        if (window) return few ? launchDirect<true, 8, 1>(a, ctx) : launchDirect<true, 4, 1>(a, ctx);
        return few ? launchDirect<false, 8, 1>(a, ctx) : launchDirect<false, 4, 1>(a, ctx);
    }
    if (window) return few ? launchDirect<true, 8, 0>(a, ctx) : launchDirect<true, 4, 0>(a, ctx);
    return few ? launchDirect<false, 8, 0>(a, ctx) : launchDirect<false, 4, 0>(a, ctx);
}

}  // namespace thip
