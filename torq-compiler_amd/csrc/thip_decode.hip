// gfx950 kernels of decode-shaped bf16 programs (a decoder's step: at most 32 input rows per linear, so every
// matrix is read once and the weights are the traffic): dec_linear, the grouped linear on block-quantized int8
// weights (torq_hl.expand_weights folded into torq_hl.matmul, the add behind it folded into the epilogue), and
// dec_matmul, the batched small matmul against a run-time operand held [N][K] (the attention's two products).
//
// Both use v_mfma_f32_16x16x32_bf16 with the weights as the row operand: a lane (c = lane & 15, g = lane >> 4) feeds
// weight column c and input row c, each with the 8 consecutive k of group g, and receives
// D[n = 4 g + e][m = c] in register e: four neighbouring output columns of one input row.  fp32 products of bf16
// values are exact; only the order of the additions differs from a sum in k order.
#include "thip_kernels_common.h"

namespace thip {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kDecWaves = 8;      // waves of a dec_matmul workgroup = ways K is split inside it
constexpr int kDecMaxWaves = 16;  // dec_linear: between 8 and 16, one k-block each where K allows (DecLinearArgs::nwaves)

__device__ __forceinline__ unsigned ldsOffset(const void *p) {
    return (unsigned)(uintptr_t)(__attribute__((address_space(3))) const int8_t *)p;
}

// 64 lanes x 4 bytes, global -> LDS (see dmaLoad16).
__device__ __forceinline__ void dmaLoad4(const void *gptr, unsigned ldsAddr) {
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dword %1, off" : : "s"(ldsAddr), "v"(gptr) : "memory", "m0");
}

// s_waitcnt vmcnt(n) for a wave-uniform run-time n (the instruction takes an immediate).
__device__ __forceinline__ void waitVmcntDyn(int n) {
#define THIP_VMCNT_CASE(k) \
    case k: waitVmcnt<k>(); break;
    switch (n) {
        THIP_VMCNT_CASE(0) THIP_VMCNT_CASE(1) THIP_VMCNT_CASE(2) THIP_VMCNT_CASE(3) THIP_VMCNT_CASE(4) THIP_VMCNT_CASE(5) THIP_VMCNT_CASE(6) THIP_VMCNT_CASE(7)
        THIP_VMCNT_CASE(8) THIP_VMCNT_CASE(9) THIP_VMCNT_CASE(10) THIP_VMCNT_CASE(11) THIP_VMCNT_CASE(12) THIP_VMCNT_CASE(13) THIP_VMCNT_CASE(14) THIP_VMCNT_CASE(15)
        THIP_VMCNT_CASE(16) THIP_VMCNT_CASE(17) THIP_VMCNT_CASE(18) THIP_VMCNT_CASE(19) THIP_VMCNT_CASE(20) THIP_VMCNT_CASE(21) THIP_VMCNT_CASE(22) THIP_VMCNT_CASE(23)
        THIP_VMCNT_CASE(24) THIP_VMCNT_CASE(25) THIP_VMCNT_CASE(26) THIP_VMCNT_CASE(27) THIP_VMCNT_CASE(28) THIP_VMCNT_CASE(29) THIP_VMCNT_CASE(30) THIP_VMCNT_CASE(31)
        THIP_VMCNT_CASE(32) THIP_VMCNT_CASE(33) THIP_VMCNT_CASE(34) THIP_VMCNT_CASE(35) THIP_VMCNT_CASE(36) THIP_VMCNT_CASE(37) THIP_VMCNT_CASE(38) THIP_VMCNT_CASE(39)
        THIP_VMCNT_CASE(40) THIP_VMCNT_CASE(41) THIP_VMCNT_CASE(42) THIP_VMCNT_CASE(43) THIP_VMCNT_CASE(44) THIP_VMCNT_CASE(45) THIP_VMCNT_CASE(46) THIP_VMCNT_CASE(47)
    default: break;  // 48 or more may stay in flight: more than a wave of these kernels ever has
    }
#undef THIP_VMCNT_CASE
}

// Where element (row, n) of a result of `rows` rows and N columns lies, in elements.
__device__ __forceinline__ size_t decResultAt(bool blocked, int rows, int row, int n, int N) {
    return blocked ? (size_t)(n >> 5) * (size_t)(rows * 32) + (size_t)(row * 32 + (n & 31)) : (size_t)row * N + n;
}

constexpr int kDecLdsSlot = 2048 + 128;  // a k-block's weights, scales and (room for) biases in LDS

// MR: groups of 16 input rows (1 or 2).  XLDS: the input rows come through LDS as well (at most four rows): then every
// global load of a wave is an LDS-DMA load issued up front and each k-block is computed as soon as it has landed.
// Otherwise the rows come through registers, CH k-blocks at a time, two such chunks in flight, or (ONE) the one that a wave has at most.  QB: the slots carry block biases.
// QC: the expansion clamps.
// S (XLDS only): the 16-column tile is shared out over S workgroups of CW = 16 / S columns, each an MFMA's row operand made of S
// k-blocks of its columns: operand row c holds column c % CW of k-block c / CW and input column c holds input row c % CW of k-block
// c / CW, so of the 16 x 16 products the S blocks on the diagonal are wanted; their sum is the result.  The lanes, loads and expansions of
// a workgroup are as full as with one k-block, of which it has S times fewer.
template <int MR, int CH, bool XLDS, bool QB, bool QC, int S, bool ONE>
__global__ __launch_bounds__(kDecMaxWaves * 64) void dec_linear(DecLinearArgs p) {
    extern __shared__ __attribute__((aligned(16))) int8_t smem[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int NW = p.nwaves;  // waves of this workgroup: k-blocks wave, wave + NW, ... are this wave's
    const int c = lane & 15, g = lane >> 4;
    // the input rows of this workgroup: grid.y workgroups share a column tile, rows_per_group rows each
    const int row0 = (int)blockIdx.y * p.rows_per_group;
    const int M = p.M - row0 < p.rows_per_group ? p.M - row0 : p.rows_per_group;
    const uint16_t *x = p.x + (size_t)row0 * p.K;
    static_assert(S == 1 || (XLDS && MR == 1), "");
    constexpr int CW = 16 / S;
    const int cj = c / CW;  // of the S k-blocks at a time, the one this lane's column (and input row) belongs to
    // the tile of this workgroup: (matrix, 16 columns of it); a pair owns the same columns of both matrices
    int tile = (int)blockIdx.x / S, seg = 0;
    const int col0 = ((int)blockIdx.x % S) * CW;  // its first column of the tile
    if (!p.pair) {
        if (p.nseg > 1 && tile >= p.N[0] / 16) {
            tile -= p.N[0] / 16;
            seg = 1;
            if (p.nseg > 2 && tile >= p.N[1] / 16) {
                tile -= p.N[1] / 16;
                seg = 2;
            }
        }
    }
    const int nmat = p.pair ? 2 : 1;
    const int kblocks = p.K >> 7;  // K % 128 == 0
    const int units = (kblocks + S - 1) / S;  // S k-blocks each
    const int nkb = wave >= units ? 0 : ONE ? 1 : (units - wave + NW - 1) / NW;
    const int maxkb = ONE ? 1 : (units + NW - 1) / NW;
    const int slotBytes = kDecSlotBytes + (QB ? 64 : 0);
    const int xRowBytes = XLDS ? M * S * 256 : 0;  // a unit of the input rows in LDS
    const unsigned regionBytes = (unsigned)maxkb * (unsigned)(xRowBytes + nmat * kDecLdsSlot);
    int8_t *region = smem + (size_t)wave * regionBytes;
    int8_t *slots = region + (size_t)maxkb * xRowBytes;
    const unsigned regionLds = ldsOffset(smem) + (unsigned)wave * regionBytes;
    const unsigned slotsLds = regionLds + (unsigned)(maxkb * xRowBytes);
    const int8_t *wsrc[2];
    {
        const int s0 = p.pair ? 0 : seg, s1 = p.pair ? 1 : seg;
        wsrc[0] = s0 == 0 ? p.w[0] : s0 == 1 ? p.w[1] : p.w[2];
        wsrc[1] = s1 == 0 ? p.w[0] : s1 == 1 ? p.w[1] : p.w[2];
    }
    if (XLDS) {
        // lane l brings 16 bytes of row l >> 4: a k-block of one row is 16 lanes x 16 bytes
        for (int i = 0; i < nkb; i++) {
            const int kb = wave + NW * i;
            if constexpr (S == 1) {
                if (lane < 16 * M) dmaLoad16(x + (size_t)(lane >> 4) * p.K + kb * 128 + (lane & 15) * 8, regionLds + (unsigned)(i * xRowBytes));
            } else {
                // piece = (row, k-block of the unit); a k-block past the last one is read as the last (its weights expand to zero)
                for (int q = 0; q < M * S; q += 4) {
                    const int piece = q + (lane >> 4), row = piece / S, b = kb * S + piece % S;
                    if (piece < M * S) dmaLoad16(x + (size_t)row * p.K + (b < kblocks ? b : kblocks - 1) * 128 + (lane & 15) * 8, regionLds + (unsigned)(i * xRowBytes + q * 256));
                }
            }
        }
    }
    // the wave's whole share of the weights, one burst: per k-block and matrix 2 KiB and the scales, straight into LDS
    for (int i = 0; i < ((p.ablate & 1) ? 0 : nkb); i++) {
        const int kb = wave + NW * i;
        for (int m = 0; m < nmat; m++) {
            const unsigned dst = slotsLds + (unsigned)(i * nmat + m) * kDecLdsSlot;
            if constexpr (S == 1) {
                const int8_t *src = wsrc[m] + ((size_t)tile * kblocks + kb) * slotBytes;
                dmaLoad16(src + (size_t)lane * 16, dst);
                dmaLoad16(src + 1024 + (size_t)lane * 16, dst + 1024u);
                if (lane < (QB ? 32 : 16)) dmaLoad4(src + 2048 + (size_t)lane * 4, dst + 2048u);
            } else {
                const int b = kb * S + cj, column = col0 + c % CW;
                const int8_t *src = wsrc[m] + ((size_t)tile * kblocks + (b < kblocks ? b : kblocks - 1)) * slotBytes;
                dmaLoad16(src + (size_t)(g * 16 + column) * 16, dst);
                dmaLoad16(src + 1024 + (size_t)(g * 16 + column) * 16, dst + 1024u);
                if (lane < (QB ? 32 : 16)) dmaLoad4(src + 2048 + (size_t)(g * 16 + column) * 4, dst + 2048u);
            }
        }
    }
    v4f acc[2][MR];
#pragma unroll
    for (int m = 0; m < 2; m++) {
#pragma unroll
        for (int mr = 0; mr < MR; mr++) acc[m][mr] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    }
    // one k-block of one matrix: 32 weights of the lane expanded, four MFMAs per row group
    auto kblock = [&](int i, int m, const v4i (&xp)[4][MR]) {
        const int8_t *slot = slots + (size_t)(i * nmat + m) * kDecLdsSlot;
        const v4i p0 = *(const v4i *)(slot + lane * 16), p1 = *(const v4i *)(slot + 1024 + lane * 16);
        float sc = *(const float *)(slot + 2048 + c * 4);
        float bi = QB ? *(const float *)(slot + 2048 + 64 + c * 4) : 0.0f;
        bool beyond = false;
        if constexpr (S > 1) {
            beyond = (wave + NW * i) * S + cj >= kblocks;
            if (beyond) sc = bi = 0.0f;
        }
        const int dw[8] = {p0[0], p0[1], p0[2], p0[3], p1[0], p1[1], p1[2], p1[3]};
#pragma unroll
        for (int j = 0; j < 4; j++) {
            int o[4];
            expandQ8<QC>(dw[2 * j], sc, bi, p.qlo, p.qhi, &o[0], &o[1]);
            expandQ8<QC>(dw[2 * j + 1], sc, bi, p.qlo, p.qhi, &o[2], &o[3]);
            if constexpr (QC && S > 1) {  // zero may lie outside the expansion's clamp
#pragma unroll
                for (int e = 0; e < 4; e++) o[e] = beyond ? 0 : o[e];
            }
            const v8bf wfrag = __builtin_bit_cast(v8bf, v4i{o[0], o[1], o[2], o[3]});
#pragma unroll
            for (int mr = 0; mr < MR; mr++) {
                acc[m][mr] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wfrag, __builtin_bit_cast(v8bf, xp[j][mr]), acc[m][mr], 0, 0, 0);
            }
        }
    };
    if constexpr (XLDS) {
        // lanes of rows the input does not have read row 0 (never stored)
        const int xrow = ((c % CW < M ? c % CW : 0) * S + cj) * 256 + g * 16;
        for (int i = 0; i < ((p.ablate & 2) ? 0 : nkb); i++) {
            waitVmcntDyn((p.ablate & 1) ? 0 : (nkb - 1 - i) * 3 * nmat);  // everything up to this k-block has landed
            v4i xp[4][MR];
#pragma unroll
            for (int j = 0; j < 4; j++) xp[j][0] = *(const v4i *)(region + (size_t)i * xRowBytes + xrow + j * 64);
            if constexpr (S > 1) {
                if ((wave + NW * i) * S + cj >= kblocks) {
#pragma unroll
                    for (int j = 0; j < 4; j++) xp[j][0] = v4i{0, 0, 0, 0};
                }
            }
            kblock(i, 0, xp);
            if (nmat > 1) kblock(i, 1, xp);
        }
    } else {
        constexpr int UN = ONE ? 1 : CH;
        struct XBuf {
            v4i x[UN][4][MR];
        };
        // A load brings 64 bytes of each of 16 rows: half a line each where rows lie one behind the other, and a wave's second half only hits
        // while the first is in its CU's 32 KB cache, among the loads of 15 other waves.  Block by block it is 1 KB of whole lines.
        const bool xBlocked = (p.blocked & kDecBlockedX) != 0;
        const uint32_t xRow = xBlocked ? 32u : (uint32_t)p.K, xStep = xBlocked ? 32u * (uint32_t)p.M : 32u;
        const int8_t *xFirst = (const int8_t *)(p.x + (size_t)((uint32_t)row0 * xRow));
        uint32_t xLane[MR];  // bytes; the rest of an address is the same for the wave
#pragma unroll
        for (int mr = 0; mr < MR; mr++) xLane[mr] = ((uint32_t)(c + 16 * mr) * xRow + 8u * (uint32_t)g) * 2u;
        // Loads only; a k-block the wave does not have and a row beyond M read nothing and feed zeros.
        auto loadChunk = [&](int ch, XBuf &b) {
#pragma unroll
            for (int u = 0; u < UN; u++) {
                const int i = ch * UN + u;
                const int kb = wave + NW * i;
#pragma unroll
                for (int mr = 0; mr < MR; mr++) {
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        b.x[u][j][mr] = (i < nkb && c + 16 * mr < M) ? *(const v4i *)(xFirst + (size_t)(2u * (uint32_t)(4 * kb + j) * xStep) + xLane[mr]) : v4i{0, 0, 0, 0};
                    }
                }
            }
        };
        auto computeChunk = [&](int ch, const XBuf &b) {
#pragma unroll
            for (int u = 0; u < UN; u++) {
                const int i = ch * UN + u;
                if (i >= nkb) break;
                kblock(i, 0, b.x[u]);
                if (nmat > 1) kblock(i, 1, b.x[u]);
            }
        };
        const int nchunks = (nkb + UN - 1) / UN;
        XBuf b0;
        loadChunk(0, b0);
        if constexpr (ONE) {
            waitVmcnt<0>();
            computeChunk(0, b0);
        } else {
            XBuf b1;
            if (nchunks > 1) loadChunk(1, b1);
            waitVmcnt<0>();  // the DMA burst (and the rows of two chunks) has landed; the compiler counts only its own loads
            for (int ch = 0; ch < nchunks; ch += 2) {
                computeChunk(ch, b0);
                if (ch + 2 < nchunks) loadChunk(ch + 2, b0);
                if (ch + 1 < nchunks) {
                    computeChunk(ch + 1, b1);
                    if (ch + 3 < nchunks) loadChunk(ch + 3, b1);
                }
            }
        }
    }
    // the waves' partial sums meet in LDS: each leaves its own in its own region (its weights are used up)
    asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
#pragma unroll
    for (int m = 0; m < 2; m++) {
#pragma unroll
        for (int mr = 0; mr < MR; mr++) {
            if (m < nmat) ((v4f *)region)[(m * MR + mr) * 64 + lane] = acc[m][mr];
        }
    }
    __syncthreads();
    if (wave >= MR) return;
    const int mr = wave;  // this wave finishes row group `wave`
    const bool mine = c + 16 * mr < M && 4 * g < CW;
    if (S == 1 && !mine) return;  // S > 1: every lane's sums are wanted below
    const int row = row0 + c + 16 * mr;  // as the whole launch counts them
    const int s0 = p.pair ? 0 : seg;
    const int Nseg = s0 == 0 ? p.N[0] : s0 == 1 ? p.N[1] : p.N[2];
    const int n = tile * 16 + col0 + 4 * g;
    // what the epilogue reads from memory, issued before the sums are collected
    v4f bias4[2];
#pragma unroll
    for (int m = 0; m < 2; m++) {
        const int sm = p.pair ? m : seg;
        const float *bias = sm == 0 ? p.bias[0] : sm == 1 ? p.bias[1] : p.bias[2];
        bias4[m] = m < nmat && mine ? *(const v4f *)(bias + n) : v4f{0.0f, 0.0f, 0.0f, 0.0f};
    }
    v2i rv = v2i{0, 0};
    if (p.add_mode == 1 && mine) rv = *(const v2i *)(p.res + decResultAt(p.blocked & kDecBlockedRes, p.M, row, n, Nseg));
    uint16_t y[2][4];
#pragma unroll
    for (int m = 0; m < 2; m++) {
        if (m >= nmat) break;
        v4f s = v4f{0.0f, 0.0f, 0.0f, 0.0f};
        // ONE: a wave's sum and that of the eighth behind it first: 9 to 16 sums added in turn are further from the 64-bit sum than eight waves' of up to two
        // k-blocks each (a model of both orders on the CPU, K = 2048: 4.01e-6 against 3.70e-6 rms; so paired 3.50e-6, and less than the eight's at every K from 1152 on).  The
        // pairs cost a step of four layers at hidden 2048, 20 rows, 145.9 -> 148.5 us (eight waves 153.0), at 1152, 32 rows, 137.2 -> 137.9 (142.0).
        for (int w = 0; w < (ONE ? kDecWaves : NW); w++) {
            v4f t = ((const v4f *)(smem + (size_t)w * regionBytes))[(m * MR + mr) * 64 + lane];
            if (ONE && w + kDecWaves < NW) t += ((const v4f *)(smem + (size_t)(w + kDecWaves) * regionBytes))[(m * MR + mr) * 64 + lane];
            s += t;
        }
        if constexpr (S > 1) {
            // block j of the diagonal lies in the lanes 5 CW further on: input columns CW j .., weight rows CW j .. in lane groups CW / 4 j ..
            v4f d = s;
#pragma unroll
            for (int j = 1; j < S; j++) {
#pragma unroll
                for (int e = 0; e < 4; e++) d[e] += __shfl(s[e], lane + 5 * CW * j);
            }
            s = d;
        }
        const int sm = p.pair ? m : seg;
        uint16_t *out = sm == 0 ? p.out[0] : sm == 1 ? p.out[1] : p.out[2];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float t0 = s[e] + bias4[m][e];
            y[m][e] = bf16Bits(t0 < p.lo ? p.lo : (t0 > p.hi ? p.hi : t0));
        }
        if (out && mine) {
            *(v2i *)(out + decResultAt(p.blocked & (kDecBlockedOut << sm), p.M, row, n, Nseg)) = v2i{(int)((uint32_t)y[m][0] | ((uint32_t)y[m][1] << 16)), (int)((uint32_t)y[m][2] | ((uint32_t)y[m][3] << 16))};
        }
    }
    if (p.add_mode == 0 || !mine) return;
    uint16_t z[4];
    if (p.add_mode == 1) {
        const uint16_t r[4] = {(uint16_t)rv[0], (uint16_t)((uint32_t)rv[0] >> 16), (uint16_t)rv[1], (uint16_t)((uint32_t)rv[1] >> 16)};
#pragma unroll
        for (int e = 0; e < 4; e++) {
            z[e] = p.res_first ? addBf16One(r[e], y[0][e], p.aw0, p.aw1, p.abias, p.alo, p.ahi) : addBf16One(y[0][e], r[e], p.aw0, p.aw1, p.abias, p.alo, p.ahi);
        }
    } else {
#pragma unroll
        for (int e = 0; e < 4; e++) z[e] = addBf16One(y[0][e], y[1][e], p.aw0, p.aw1, p.abias, p.alo, p.ahi);
    }
    *(v2i *)(p.add_out + decResultAt(p.blocked & kDecBlockedAdd, p.M, row, n, Nseg)) = v2i{(int)((uint32_t)z[0] | ((uint32_t)z[1] << 16)), (int)((uint32_t)z[2] | ((uint32_t)z[3] << 16))};
}

template <int MR, int CH, bool XLDS, bool QB, bool QC, int S = 1, bool ONE = false>
static hipError_t launchDecLinearT(const DecLinearArgs &a, int tiles, size_t lds, const LaunchCtx &ctx) {
    auto kernel = dec_linear<MR, CH, XLDS, QB, QC, S, ONE>;
    static std::once_flag once;
    static hipError_t configured = hipSuccess;
    std::call_once(once, [&] { configured = hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024); });
    if (configured != hipSuccess) return configured;
    const int groups = (a.M + a.rows_per_group - 1) / a.rows_per_group;
    THIP_ENQUEUE(ctx, (ONE ? kernelLabel("dec_linear", {MR, CH, (int)XLDS, (int)QB, (int)QC, a.pair ? 2 : a.nseg, a.add_mode, S, 1}) : kernelLabel("dec_linear", {MR, CH, (int)XLDS, (int)QB, (int)QC, a.pair ? 2 : a.nseg, a.add_mode, S})),
                 kernel, dim3((unsigned)tiles * S, (unsigned)groups),
                 dim3((unsigned)a.nwaves * 64), lds, a);
    return hipGetLastError();
}

// LDS a launch needs: every wave's share of the weights, and of the input rows when they come through LDS (the
// partial sums reuse it).
static size_t decLinearLds(int K, int nmat, int xRows, int nwaves) {
    const int kblocks = K / 128, maxkb = (kblocks + nwaves - 1) / nwaves;
    return (size_t)nwaves * maxkb * (size_t)(xRows * 256 + nmat * kDecLdsSlot);
}
// Waves per workgroup: one k-block each where K has between 8 and 16 of them, 16 for a longer K (a wave's
// arithmetic is the launch's critical path: 128 x 16 weights expanded per k-block and matrix).
int decLinearWaves(int K) {
    const int kblocks = K / 128;
    return kblocks < kDecWaves ? kDecWaves : (kblocks > kDecMaxWaves ? kDecMaxWaves : kblocks);
}
constexpr size_t kDecMaxLds = 152 * 1024;

// Workgroups per column tile.  A workgroup streams its rows of the input next to its 16 columns of the weights: with few
// column tiles and many rows (32 rows of K = 6912 are 442 KB per workgroup against 110 KB of weights, on 72 of 256 CUs)
// the rows are the traffic, and sharing them out over several workgroups, each re-reading the weights, spreads it over
// the chip.  As many groups as keep the launch within one workgroup per CU, at least eight rows each.
static int decLinearRowGroups(int M, int tiles, const Tuning *tuning) {
    if (M <= kDecLdsRows) return 1;
    int groups = (tuning && tuning->decTargetGroups > 0 ? tuning->decTargetGroups : 256) / tiles;
    const int most = (M + 7) / 8;
    groups = groups < 1 ? 1 : (groups > most ? most : groups);
    return groups;
}

// Workgroups that share a 16-column tile, eight columns each (see dec_linear's S).  A K of more k-blocks than a workgroup has
// waves is walked in rounds, on as many CUs as there are tiles: two workgroups per tile halve the rounds where that still is one per
// CU (one row, 6912 -> 1152: 7.6 us with 72 workgroups of 16 waves, 6.35 with 144 of 14, 7.0 with 288, four columns each; 1152 ->
// 1536 and 1024 -> 1152, one round either way, 4.2 and 4.6 us against 4.3 and 4.5; 1152 -> 2 x 6912, whose 432 tiles fill the chip,
// 7.8 against 9.2).
static int decLinearSplit(int K, int tiles, const Tuning *tuning) {
    if (tuning && tuning->decSplit > 0) return tuning->decSplit;
    return K / 128 > kDecMaxWaves && tiles * 2 <= 256 ? 2 : 1;
}

template <bool QB, bool QC>
static hipError_t launchDecLinearQ(const DecLinearArgs &in, int tiles, const LaunchCtx &ctx) {
    DecLinearArgs a = in;
    const int nmat = a.pair ? 2 : 1;
    a.rows_per_group = a.M;
    if (a.M <= kDecLdsRows) {
        // the input rows through LDS as well, with the most waves whose regions still fit
        for (int nw = a.nwaves; nw >= kDecWaves; nw--) {
            if (decLinearLds(a.K, nmat, a.M, nw) > kDecMaxLds) continue;
            const int split = decLinearSplit(a.K, tiles, ctx.tuning);
            if (split > 1) {  // less LDS than one workgroup per tile, which fits
                const int units = (a.K / 128 + split - 1) / split, rounds = (units + kDecMaxWaves - 1) / kDecMaxWaves;
                a.nwaves = (units + rounds - 1) / rounds;
                const size_t lds = (size_t)a.nwaves * rounds * (size_t)(a.M * split * 256 + nmat * kDecLdsSlot);
                return launchDecLinearT<1, 1, true, QB, QC, 2>(a, tiles, lds, ctx);
            }
            a.nwaves = nw;
            return launchDecLinearT<1, 1, true, QB, QC>(a, tiles, decLinearLds(a.K, nmat, a.M, nw), ctx);
        }
    }
    const int groups = decLinearRowGroups(a.M, tiles, ctx.tuning);
    a.rows_per_group = (a.M + groups - 1) / groups;
    // A wave of one k-block holds the rows of that one only (64 registers at most): two workgroups of 16 such waves share a CU.  Where K has more k-blocks
    // than waves and the launch more workgroups than CUs, eight waves each, so that two of them (at four waves per SIMD) share one and the launch is
    // one round of workgroups rather than two.  Steps of four layers, us, always eight / this (sums added in turn; in pairs, as now, 0.4 to 1.8 % more): hidden 1152 at 32 rows 165.6 / 160.7, at 8 129.1 / 123.8;
    // 1536 at 16 rows 134.1 / 130.0, at 32 155.4 / 148.7; 2048 at 20 rows 167.2 / 160.0 (with more than 12 such waves left at eight 164.7), at 12 157.2 / 147.5; 768 at 24 rows
    // 107.6 / 103.8 (the registers alone).
    const bool few = a.rows_per_group <= 16;
    if ((long long)tiles * groups > 256 && a.nwaves < a.K / 128) a.nwaves = kDecWaves;
    const size_t lds = decLinearLds(a.K, nmat, 0, a.nwaves);
    if (a.nwaves >= a.K / 128) return few ? launchDecLinearT<1, 2, false, QB, QC, 1, true>(a, tiles, lds, ctx) : launchDecLinearT<2, 1, false, QB, QC, 1, true>(a, tiles, lds, ctx);
    if (few) return launchDecLinearT<1, 2, false, QB, QC>(a, tiles, lds, ctx);
    return launchDecLinearT<2, 1, false, QB, QC>(a, tiles, lds, ctx);
}

hipError_t launchDecLinear(const DecLinearArgs &in, const LaunchCtx &ctx) {
    DecLinearArgs a = in;
    a.nwaves = a.K > 0 ? decLinearWaves(a.K) : kDecWaves;
    if (!a.x || a.M <= 0 || a.M > kDecMaxRows || a.K <= 0 || a.K % 128 != 0 || a.qblock <= 0 || a.qblock % 128 != 0 || a.K % a.qblock != 0) return hipErrorInvalidValue;
    if (a.nseg < 1 || a.nseg > kDecMaxSegments || (a.pair && a.nseg != 2) || (((uintptr_t)a.x) & 15)) return hipErrorInvalidValue;
    if (a.add_mode < 0 || a.add_mode > 2 || (a.add_mode == 1 && (a.nseg != 1 || !a.res)) || (a.add_mode == 2 && !a.pair) || (a.pair && a.add_mode != 2)) return hipErrorInvalidValue;
    if (a.blocked && a.M <= kDecLdsRows) return hipErrorInvalidValue;
    if (a.add_mode != 0 && (!a.add_out || (((uintptr_t)a.add_out) & 7) || (a.res && (((uintptr_t)a.res) & 7)))) return hipErrorInvalidValue;
    long long tiles = 0;
    for (int s = 0; s < a.nseg; s++) {
        if (!a.w[s] || !a.bias[s] || a.N[s] <= 0 || a.N[s] % 16 != 0) return hipErrorInvalidValue;
        if ((((uintptr_t)a.w[s]) & 15) || (((uintptr_t)a.bias[s]) & 15) || (((uintptr_t)a.out[s]) & 7)) return hipErrorInvalidValue;
        if (!a.out[s] && a.add_mode == 0) return hipErrorInvalidValue;  // a result nobody receives
        if (a.N[s] % 32 != 0 && (a.blocked & (kDecBlockedRes | kDecBlockedAdd | kDecBlockedOut << s))) return hipErrorInvalidValue;
        tiles += a.N[s] / 16;
    }
    if (a.pair) {
        if (a.N[0] != a.N[1]) return hipErrorInvalidValue;
        tiles = a.N[0] / 16;
    }
    if (tiles <= 0 || tiles > 65535 || decLinearLds(a.K, a.pair ? 2 : 1, 0, a.nwaves) > kDecMaxLds) return hipErrorInvalidValue;
    const bool clamp = !(a.qlo == -INFINITY && a.qhi == INFINITY);
    const int t = (int)tiles;
    if (ctx.tuning->decAblate) {
        DecLinearArgs b = a;
        b.ablate = ctx.tuning->decAblate;
        return launchDecLinearQ<false, false>(b, t, ctx);
    }
    if (clamp) return a.has_qbias ? launchDecLinearQ<true, true>(a, t, ctx) : launchDecLinearQ<false, true>(a, t, ctx);
    return a.has_qbias ? launchDecLinearQ<true, false>(a, t, ctx) : launchDecLinearQ<false, false>(a, t, ctx);
}

// dec_matmul: a workgroup owns 16 columns (rows of w) of one batch element; its eight waves split K in steps of 32
// (wave, wave + 8, ...), each lane loading 16 bytes of its weight row and of its input row per step; the partial
// sums meet in LDS.  A wave's loads of up to ST steps are all issued before the first MFMA.
template <int MR, int ST>
__global__ __launch_bounds__(kDecWaves * 64) void dec_matmul(DecMatmulArgs p) {
    __shared__ v4f red[kDecWaves][MR][64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int c = lane & 15, g = lane >> 4;
    const int n0 = (int)blockIdx.x * 16, b = (int)blockIdx.y;
    const uint16_t *a = p.a + (size_t)b * p.a_stride, *w = p.w + (size_t)b * p.w_stride;
    const int steps = (p.K + 31) >> 5;
    const int nrow = n0 + c < p.N ? n0 + c : p.N - 1;  // clamped columns are never stored
    v4f acc[MR];
#pragma unroll
    for (int mr = 0; mr < MR; mr++) acc[mr] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    for (int s0 = wave; s0 < steps; s0 += kDecWaves * ST) {
        v4i wv[ST], xv[ST][MR];
#pragma unroll
        for (int u = 0; u < ST; u++) {
            const int k = (s0 + kDecWaves * u) * 32 + 8 * g;
            const bool in = k < p.K;  // K % 8 == 0: a piece lies inside K or outside
            wv[u] = in ? *(const v4i *)(w + (size_t)nrow * p.K + k) : v4i{0, 0, 0, 0};
#pragma unroll
            for (int mr = 0; mr < MR; mr++) {
                const int row = c + 16 * mr;
                xv[u][mr] = (in && row < p.M) ? *(const v4i *)(a + (size_t)row * p.K + k) : v4i{0, 0, 0, 0};
            }
        }
#pragma unroll
        for (int u = 0; u < ST; u++) {
#pragma unroll
            for (int mr = 0; mr < MR; mr++) {
                acc[mr] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, wv[u]), __builtin_bit_cast(v8bf, xv[u][mr]), acc[mr], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int mr = 0; mr < MR; mr++) red[wave][mr][lane] = acc[mr];
    __syncthreads();
    if (wave >= MR) return;
    const int mr = wave, row = c + 16 * mr;
    if (row >= p.M) return;
    v4f s = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    for (int wv = 0; wv < kDecWaves; wv++) s += red[wv][mr][lane];
    const int n = n0 + 4 * g;
    uint16_t *out = p.out + (size_t)b * p.out_stride + (size_t)row * p.N;
    if (p.blocked) out = p.out + decResultAt(true, p.B, b, row * p.N + n, 0) - n;  // its four columns lie in one block
    uint16_t y[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const float t0 = s[e] + p.bias;
        y[e] = bf16Bits(t0 < p.lo ? p.lo : (t0 > p.hi ? p.hi : t0));
    }
    if ((p.N & 3) == 0 && n + 3 < p.N) {
        *(v2i *)(out + n) = v2i{(int)((uint32_t)y[0] | ((uint32_t)y[1] << 16)), (int)((uint32_t)y[2] | ((uint32_t)y[3] << 16))};
    } else {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            if (n + e < p.N) out[n + e] = y[e];
        }
    }
}

hipError_t launchDecMatmul(const DecMatmulArgs &a, const LaunchCtx &ctx) {
    if (!a.a || !a.w || !a.out || a.B <= 0 || a.B > 65535 || a.M <= 0 || a.M > kDecMaxRows || a.K <= 0 || a.K % 8 != 0 || a.N <= 0) return hipErrorInvalidValue;
    if (a.a_stride < 0 || a.w_stride < 0 || a.out_stride < 0 || a.a_stride % 8 != 0 || a.w_stride % 8 != 0) return hipErrorInvalidValue;
    if (((((uintptr_t)a.a) | ((uintptr_t)a.w)) & 15) || (((uintptr_t)a.out) & (a.N % 4 == 0 ? 7 : 1)) || (a.N % 4 == 0 && a.out_stride % 4 != 0)) return hipErrorInvalidValue;
    if (a.blocked && (a.blocked != kDecBlockedOut || a.N % 4 != 0 || a.out_stride != (int64_t)a.M * a.N || a.out_stride % 32 != 0 || a.B * a.out_stride >= (1LL << 31))) return hipErrorInvalidValue;
    const long long tiles = ((long long)a.N + 15) / 16;
    if (tiles > 0x7fffffffLL) return hipErrorInvalidValue;
    const dim3 grid((unsigned)tiles, (unsigned)a.B);
    // steps of 32 per wave: up to four are one round of loads
    const int perWave = ((a.K + 31) / 32 + kDecWaves - 1) / kDecWaves;
    if (a.M <= 16) {
        if (perWave <= 1) THIP_ENQUEUE(ctx, "dec_matmul<1,1>", (dec_matmul<1, 1>), grid, dim3(kDecWaves * 64), 0, a);
        else if (perWave <= 2) THIP_ENQUEUE(ctx, "dec_matmul<1,2>", (dec_matmul<1, 2>), grid, dim3(kDecWaves * 64), 0, a);
        else THIP_ENQUEUE(ctx, "dec_matmul<1,4>", (dec_matmul<1, 4>), grid, dim3(kDecWaves * 64), 0, a);
    } else {
        if (perWave <= 1) THIP_ENQUEUE(ctx, "dec_matmul<2,1>", (dec_matmul<2, 1>), grid, dim3(kDecWaves * 64), 0, a);
        else if (perWave <= 2) THIP_ENQUEUE(ctx, "dec_matmul<2,2>", (dec_matmul<2, 2>), grid, dim3(kDecWaves * 64), 0, a);
        else THIP_ENQUEUE(ctx, "dec_matmul<2,4>", (dec_matmul<2, 4>), grid, dim3(kDecWaves * 64), 0, a);
    }
    return hipGetLastError();
}

}  // namespace thip
