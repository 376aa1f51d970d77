// gfx950 kernel of the bf16 linears with many input rows (a prompt, an image's pixels): the tile form of
// fc_bf16, on v_mfma_f32_32x32x16_bf16 with both operands staged through an LDS ring by the DMA path.
#include "thip_kernels_common.h"

namespace thip {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));

// What a lane beyond K reads instead of its chunk: both factors of such a product must be zero or finite, and the
// activations next to it need not be.
__device__ __constant__ static const v4i kZeroChunk = {0, 0, 0, 0};

// Two floats as bf16, the first in the low half (nearest, ties to even; NaN stays NaN).
__device__ __forceinline__ uint32_t packBf16(float lo, float hi) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v2f{lo, hi}, v2bf));
}

// ---------------------------------------------------------------------------
// fc_bf16, tile form: out[m][n] = bf16(clamp(sum_k x[m][k] * w[n][k] + bias[n])), fp32 accumulation.
//
// The streaming form (thip_bf16.hip) reads the weights once per 32 rows of the input, which is what few rows want; with many rows every weight and
// every activation then passes L2 -> registers once per 32 x 32 outputs (2048 x 1152 -> 6912: 13 824 blocks move 2 GB,
// 155 us = 210 TFLOP/s).  Here a workgroup owns BM x BN outputs and a byte that reaches LDS is used BN (BM) times.
//
// The ring is that of igemm_dense_i8 with 128-byte k-tiles: a k-tile is 64 elements = 128 bytes of every row, moved by
// global_load_lds_dwordx4 (inline asm, waited on with hand-counted vmcnt, every wave issues the same number per k-tile),
// slot p of activation row r holds 16-byte chunk p ^ ((r >> 1) & 7) so that the rows of a ds_read_b128 phase fall into
// distinct banks.  MFMA step c of a k-tile takes chunk 4 h + c of both operands (h = lane half), which is the order the
// packed weights have in memory: FRAG weights go to LDS as they are, 4 KiB of 32 columns x 64 k at a time, and a
// fragment read is 1 KiB in lane order.  Row-major weights (a run-time operand) are staged like the activations.
//
// The weights are the MFMA's row operand: register 4 q + e of lane (r, h) is out[m = r][n = 8 q + 4 h + e].  Two
// v_permlane32_swap give a lane 8 neighbouring columns of a row: one 16-byte store, at any alignment.  RUNS: the results go through LDS instead, each
// wave's by itself, so that a store covers whole runs of a row: columns that are no whole eight, whose rows begin anywhere, cost
// what others do (2048 x 1152 -> 6911 67.7 us in single elements, 43.3 in unaligned 16-byte pieces of a lane's own row, 35.0 in runs; 1649 x
// 288 -> 4747 28.6, 13.5, 12.0; 2608 x 1024 -> 2530 33.7, 20.1, 19.9).  Where a wave's columns are 32 that way round costs more than it brings (654 x
// 1736 -> 208 9.0, 9.3), and for aligned rows the 128 x 128 tiles lose by it (1267 x 384 -> 5584 10.6, 11.3; 2042 x 176 -> 5760 11.8, 12.9; 1993 x
// 768 -> 5808 24.8, 26.1) while 256 x 256 ones do not (2048 x 1152 -> 6912 34.3, 34.0; 14 others alike): launchTile.
//
// KG groups of waves share a workgroup's outputs and take every KG-th k-tile each, with a ring of their own; their sums
// meet in LDS (few tiles under a long K: more loads in flight per CU).
//
// Bound by the ring's data path (64 KiB per k-tile of a 256 x 256 tile in 1.1 us, 58 KB/us per CU where LDS-DMA loads alone, of lines in
// the XCD's L2, reach 138; 0.86 us of MFMA work), with the launch, the ring fill and 28 MB of output at the end next to it: 2048 x 1152 -> 6912 takes 34.0 us (960 TFLOP/s).  Eight waves
// on the 256 x 256 tile rather than four: 35.7 -> 34.4 us, and the epilogue of a short K 13.0 -> 9.1.
// ---------------------------------------------------------------------------
template <int BM, int BN, int WAVES_M, int WAVES_N, int STAGES, int BLOCKS_PER_CU, int KG, bool FRAG, bool RUNS>
__global__ __launch_bounds__(WAVES_M *WAVES_N *KG * 64, BLOCKS_PER_CU) void fc_bf16(FcBf16Args p) {
    constexpr int NW = WAVES_M * WAVES_N;
    constexpr int WTM = BM / WAVES_M, WTN = BN / WAVES_N;
    constexpr int TM = WTM / 32, TN = WTN / 32, NF = TM + TN;
    constexpr int LA = BM / 8 / NW, LB = BN / 8 / NW, LPT = LA + LB;  // DMA instructions (1 KiB = 8 rows) per wave per k-tile
    constexpr int A_STAGE = BM * 128, STAGE = (BM + BN) * 128;
    static_assert(BM % (8 * NW) == 0 && BN % (8 * NW) == 0 && NW % 2 == 0, "unbalanced DMA loads");
    static_assert(WTM % 32 == 0 && WTN % 32 == 0, "wave tile must be a multiple of the MFMA tile");
    static_assert(LPT * (STAGES - 1) < 64, "vmcnt is a 6-bit counter");
    extern __shared__ __attribute__((aligned(16))) int8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int blockWave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave = blockWave % NW, kg = blockWave / NW;  // the wave's place in its group, the group
    int8_t *ring = smem + kg * (STAGES * STAGE);
    const unsigned ldsBase = (unsigned)(uintptr_t)(__attribute__((address_space(3))) int8_t *)smem + (unsigned)kg * (STAGES * STAGE);
    const int wm = wave / WAVES_N, wn = wave % WAVES_N;

    // each XCD gets a contiguous range of tiles, walked in groups of 8 tile rows (see igemm_dense_i8)
    const int tilesM = (p.M + BM - 1) / BM, tilesN = (p.N + BN - 1) / BN;
    int lin;
    {
        const int nb = (int)gridDim.x, pid = (int)blockIdx.x;
        const int per = nb / 8, rem = nb % 8, xcd = pid % 8, idx = pid / 8;
        lin = xcd * per + (xcd < rem ? xcd : rem) + idx;
    }
    constexpr int GROUP = 8;
    const int width = GROUP * tilesN, group = lin / width, firstM = group * GROUP;
    const int gsize = (tilesM - firstM) < GROUP ? (tilesM - firstM) : GROUP;
    const int m0 = (firstM + (lin % width) % gsize) * BM, n0 = ((lin % width) / gsize) * BN;

    const int allKT = (p.K + 63) / 64, KT = (allKT - kg + KG - 1) / KG;  // k-tiles of the product, of this group (kg, kg + KG, ...)
    // DMA sources.  Rows and column blocks past the end are clamped to the last one: their results are never stored.
    const int lrow = lane >> 3, lchunk = (lane & 7) ^ ((((wave & 1) << 2) + (lrow >> 1)) & 7);
    const int8_t *aTile = (const int8_t *)(p.x + (size_t)m0 * p.K);
    const int8_t *bTile = FRAG ? (const int8_t *)p.w : (const int8_t *)(p.w + (size_t)n0 * p.K);
    uint32_t aOff[LA], bOff[LB];
#pragma unroll
    for (int i = 0; i < LA; i++) {
        int r = 8 * (wave + NW * i) + lrow;
        r = m0 + r < p.M ? r : p.M - 1 - m0;
        aOff[i] = (uint32_t)r * (uint32_t)p.K * 2u + (uint32_t)lchunk * 16u;
    }
    size_t bBlock[LB];  // FRAG: byte offset of the 1 KiB pieces this wave moves, per k-tile 4 KiB apart
#pragma unroll
    for (int i = 0; i < LB; i++) {
        const int wl = wave + NW * i;
        if (FRAG) {
            const int blocks = (p.N + 31) / 32, nb = n0 / 32 + (wl >> 2);
            bBlock[i] = (size_t)(nb < blocks ? nb : blocks - 1) * allKT * 4096 + (size_t)(wl & 3) * 1024;
            bOff[i] = (uint32_t)lane * 16u;
        } else {
            int r = 8 * wl + lrow;
            r = n0 + r < p.N ? r : p.N - 1 - n0;
            bOff[i] = (uint32_t)r * (uint32_t)p.K * 2u + (uint32_t)lchunk * 16u;
            bBlock[i] = 0;
        }
    }
    // issues this wave's loads number [part * LPT / parts, (part + 1) * LPT / parts) of the group's k-tile `own`; `whole`: it lies below K
    auto issueTile = [&](int own, int part, int parts, auto wholeTag) {
        constexpr bool kWhole = decltype(wholeTag)::value;
        const unsigned stage = ldsBase + (unsigned)(own % STAGES) * STAGE;
        const int kt = own * KG + kg;
        const int8_t *aBase = aTile + (size_t)kt * 128;
        const bool beyond = !kWhole && kt * 64 + lchunk * 8 >= p.K;
#pragma unroll
        for (int x = 0; x < LPT; x++) {
            if (x * parts / LPT != part) continue;
            if (x < LA) {
                const unsigned dst = stage + (unsigned)(wave + NW * x) * 1024u;
                if (kWhole) dmaLoad16(aBase, aOff[x], dst);
                else dmaLoad16(beyond ? (const void *)&kZeroChunk : (const void *)(aBase + aOff[x]), dst);
            } else {
                const int i = x - LA;
                const unsigned dst = stage + A_STAGE + (unsigned)(wave + NW * i) * 1024u;
                if (FRAG) {
                    dmaLoad16(bTile + bBlock[i] + (size_t)kt * 4096, bOff[i], dst);
                } else {
                    const int8_t *bBase = bTile + (size_t)kt * 128;
                    if (kWhole) dmaLoad16(bBase, bOff[i], dst);
                    else dmaLoad16(beyond ? (const void *)&kZeroChunk : (const void *)(bBase + bOff[i]), dst);
                }
            }
        }
    };
    const int fr = lane & 31, half = lane >> 5, swz = (fr >> 1) & 7;
    const int off0 = ((4 * half) ^ swz) * 16;  // MFMA step 0; step c is off0 ^ (16 c)
    const int aFrag = (wm * WTM + fr) * 128 + off0;
    const int bFrag = FRAG ? A_STAGE + wn * TN * 4096 + lane * 16 : A_STAGE + (wn * WTN + fr) * 128 + off0;
    auto readFrag = [&](const int8_t *st, int c, int x, v4i(&af)[TM], v4i(&bf)[TN]) {
        if (x < TM) af[x] = *(const v4i *)(st + ((aFrag + x * 4096) ^ (c * 16)));
        else if (FRAG) bf[x - TM] = *(const v4i *)(st + bFrag + (x - TM) * 4096 + c * 1024);
        else bf[x - TM] = *(const v4i *)(st + ((bFrag + (x - TM) * 4096) ^ (c * 16)));
    };
    v16f acc[TN][TM];
#pragma unroll
    for (int j = 0; j < TN; j++) {
#pragma unroll
        for (int i = 0; i < TM; i++) {
#pragma unroll
            for (int r = 0; r < 16; r++) acc[j][i][r] = 0.0f;
        }
    }
    float myBias = 0.0f;  // parked in LDS for the epilogue
    if (tid < BN) myBias = p.bias[n0 + tid < p.N ? n0 + tid : p.N - 1];
#pragma unroll
    for (int t = 0; t < STAGES; t++) {
        if (t < KT) issueTile(t, 0, 1, std::false_type{});
    }
    if (KT >= STAGES) waitVmcnt<LPT *(STAGES - 1)>();
    else waitVmcnt<0>();
    blockBarrier();
    v4i af0[TM], bf0[TN], af1[TM], bf1[TN];
#pragma unroll
    for (int x = 0; x < NF; x++) readFrag(ring, 0, x, af0, bf0);
    // One k-tile, four MFMA steps; the reads of a step go out behind the first weight row of the one before.  In front of
    // the last the wave waits for the next k-tile, meets the block, and then refills the stage everybody has finished with.
    auto step = [&](int kt, auto steady) {
        constexpr bool kSteady = decltype(steady)::value;
        const int8_t *st = ring + (kt % STAGES) * STAGE;
        const int8_t *stNext = ring + ((kt + 1) % STAGES) * STAGE;
        auto mfmaStep = [&](v4i(&afC)[TM], v4i(&bfC)[TN], v4i(&afN)[TM], v4i(&bfN)[TN], int cNext) {
#pragma unroll
            for (int j = 0; j < TN; j++) {
#pragma unroll
                for (int i = 0; i < TM; i++) {
                    acc[j][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, bfC[j]), __builtin_bit_cast(v8bf, afC[i]), acc[j][i], 0, 0, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
                if (j == 0) {
#pragma unroll
                    for (int x = 0; x < NF; x++) readFrag(st, cNext, x, afN, bfN);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        };
        const bool have = KG == 1 || kSteady || kt < KT;  // a group may have one k-tile less than the others
        if (have) {
            mfmaStep(af0, bf0, af1, bf1, 1);
            mfmaStep(af1, bf1, af0, bf0, 2);
            mfmaStep(af0, bf0, af1, bf1, 3);
        }
        const bool more = kSteady || kt + 1 < KT;
        if (kSteady) {
            waitVmcnt<LPT *(STAGES - 2)>();
        } else if (more) {
            const int inFlight = (KT - 2 - kt) < (STAGES - 2) ? (KT - 2 - kt) : (STAGES - 2);
            if (inFlight >= 2) waitVmcnt<(LPT * 2 < 64 ? LPT * 2 : 0)>();
            else if (inFlight == 1) waitVmcnt<LPT>();
            else waitVmcnt<0>();
        }
        asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");  // this wave's reads of k-tile kt are complete
        blockBarrier();
        const bool refill = kSteady || kt + STAGES < KT;
#pragma unroll
        for (int j = 0; j < TN; j++) {
            if (refill) issueTile(kt + STAGES, j, TN, steady);
            if (!have) continue;
#pragma unroll
            for (int i = 0; i < TM; i++) {
                acc[j][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, bf1[j]), __builtin_bit_cast(v8bf, af1[i]), acc[j][i], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (j == 0 && more) {
#pragma unroll
                for (int x = 0; x < NF; x++) readFrag(stNext, 0, x, af0, bf0);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    static_assert(STAGES <= 4, "step() counts at most two k-tiles in flight behind the next one");
    int kt = 0;
    for (; kt + STAGES < allKT / KG - 1; kt++) step(kt, std::true_type{});  // every group has these
    for (; kt < (allKT + KG - 1) / KG; kt++) step(kt, std::false_type{});
    if constexpr (KG > 1) {
        // the groups' sums meet in LDS, where their rings were, and the first group adds them in group order
        blockBarrier();
        constexpr int GROUP_ACC = TN * TM * NW * 64 * 64;
        if (kg > 0) {
#pragma unroll
            for (int j = 0; j < TN; j++) {
#pragma unroll
                for (int i = 0; i < TM; i++) {
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        *(float4 *)(smem + (kg - 1) * GROUP_ACC + ((((j * TM + i) * 4 + q) * NW + wave) * 64 + lane) * 16) =
                            float4{acc[j][i][4 * q], acc[j][i][4 * q + 1], acc[j][i][4 * q + 2], acc[j][i][4 * q + 3]};
                    }
                }
            }
        }
        __syncthreads();
        if (kg == 0) {
            for (int o = 0; o < KG - 1; o++) {
#pragma unroll
                for (int j = 0; j < TN; j++) {
#pragma unroll
                    for (int i = 0; i < TM; i++) {
#pragma unroll
                        for (int q = 0; q < 4; q++) {
                            const float4 v = *(const float4 *)(smem + o * GROUP_ACC + ((((j * TM + i) * 4 + q) * NW + wave) * 64 + lane) * 16);
                            acc[j][i][4 * q] += v.x; acc[j][i][4 * q + 1] += v.y; acc[j][i][4 * q + 2] += v.z; acc[j][i][4 * q + 3] += v.w;
                        }
                    }
                }
            }
        }
        static_assert((KG - 1) * GROUP_ACC <= KG * STAGES * STAGE, "the groups' sums fit where the rings were");
    }

    blockBarrier();  // the ring is free: the bias goes where it was
    float *ldsBias = (float *)smem;
    if (tid < BN) ldsBias[tid] = myBias;
    __syncthreads();
    if (KG > 1 && kg > 0) return;
    // Eight results of row m from column n on, at any alignment.
    auto store = [&](int m, int n, v4i v) {
        if (m >= p.M || n >= p.N) return;
        uint16_t *out = p.out + (size_t)m * p.N + n;
        if (n + 8 <= p.N) {
            ((UnalignedV4 *)out)->v = v;
        } else {
#pragma unroll
            for (int e = 0; e < 7; e++) {
                if (n + e < p.N) out[e] = (uint16_t)((uint32_t)v[e >> 1] >> (16 * (e & 1)));
            }
        }
    };
    // Bias, clamp, v_cvt_pk_bf16_f32 and the stores; a copy without the clamp's compares, which are half the instructions
    // of an epilogue that every CU runs at the same time (a linear layer has none).  RUNS: 32 rows of a wave's results pass through LDS.
    constexpr int CHUNKS = WTN / 8;  // of eight results in a row of a wave
    int8_t *mine = smem + BN * 4 + wave * (WTM * WTN * 2);
    const int sc = lane % CHUNKS, sr = lane / CHUNKS;
    auto finish = [&](auto clampTag) {
        constexpr bool kClamp = decltype(clampTag)::value;
#pragma unroll
        for (int i = 0; i < TM; i++) {
            int8_t *rows = mine + i * (32 * WTN * 2);
#pragma unroll
            for (int j = 0; j < TN; j++) {
                uint32_t d[8];  // d[2 q + (e >> 1)]: columns 8 q + 4 half + e, + 1
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const float4 b4 = *(const float4 *)(ldsBias + wn * WTN + j * 32 + 8 * q + 4 * half);
                    const float b[4] = {b4.x, b4.y, b4.z, b4.w};
                    float v[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        v[e] = acc[j][i][4 * q + e] + b[e];
                        if (kClamp) v[e] = v[e] < p.lo ? p.lo : (v[e] > p.hi ? p.hi : v[e]);
                    }
                    d[2 * q] = packBf16(v[0], v[1]);
                    d[2 * q + 1] = packBf16(v[2], v[3]);
                    if (RUNS) *(v2i *)(rows + fr * (WTN * 2) + (((4 * j + q) ^ fr) % CHUNKS) * 16 + 8 * half) = v2i{(int)d[2 * q], (int)d[2 * q + 1]};
                }
                if (RUNS) continue;
#pragma unroll
                for (int q2 = 0; q2 < 2; q2++) {  // the lower half of the wave ends up with the first 8 of 16 columns, the upper with the others
                    const auto s0 = __builtin_amdgcn_permlane32_swap(d[4 * q2], d[4 * q2 + 2], false, false);
                    const auto s1 = __builtin_amdgcn_permlane32_swap(d[4 * q2 + 1], d[4 * q2 + 3], false, false);
                    store(m0 + wm * WTM + i * 32 + fr, n0 + wn * WTN + j * 32 + 16 * q2 + 8 * half, v4i{(int)s0[0], (int)s1[0], (int)s0[1], (int)s1[1]});
                }
            }
            if (!RUNS) continue;
            asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
#pragma unroll
            for (int t = 0; t < CHUNKS / 2; t++) {
                const int r = t * (64 / CHUNKS) + sr;
                store(m0 + wm * WTM + i * 32 + r, n0 + wn * WTN + sc * 8, *(const v4i *)(rows + r * (WTN * 2) + ((sc ^ r) % CHUNKS) * 16));
            }
        }
    };
    if (p.lo == -INFINITY && p.hi == INFINITY) finish(std::false_type{});
    else finish(std::true_type{});
}

template <int BM, int BN, int WAVES_M, int WAVES_N, int STAGES, int BLOCKS_PER_CU, int KG, bool FRAG, bool RUNS>
static hipError_t launchTileRuns(const FcBf16Args &a, const LaunchCtx &ctx) {
    auto kernel = fc_bf16<BM, BN, WAVES_M, WAVES_N, STAGES, BLOCKS_PER_CU, KG, FRAG, RUNS>;
    constexpr size_t ring = (size_t)KG * STAGES * (BM + BN) * 128, results = (size_t)BN * 4 + (size_t)BM * BN * 2, lds = RUNS && results > ring ? results : ring;
    static std::once_flag once;
    static hipError_t configured = hipSuccess;
    std::call_once(once, [&] { configured = hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds); });
    if (configured != hipSuccess) return configured;
    const long long tiles = (long long)((a.M + BM - 1) / BM) * ((a.N + BN - 1) / BN);
    if (tiles > 0x7fffffffLL) return hipErrorInvalidValue;
    THIP_ENQUEUE(ctx, kernelLabel("fc_bf16", {BM, BN, WAVES_M, WAVES_N, STAGES, BLOCKS_PER_CU, KG, (int)FRAG + 2 * (int)RUNS}), kernel, dim3((unsigned)tiles), dim3(WAVES_M * WAVES_N * KG * 64), lds, a);
    return hipGetLastError();
}
template <int BM, int BN, int WAVES_M, int WAVES_N, int STAGES, int BLOCKS_PER_CU, int KG, bool FRAG>
static hipError_t launchTile(const FcBf16Args &a, const LaunchCtx &ctx) {
    if constexpr (BN / WAVES_N > 32) {
        if (BM == 256 || a.N % 8 != 0 || ((uintptr_t)a.out & 15)) return launchTileRuns<BM, BN, WAVES_M, WAVES_N, STAGES, BLOCKS_PER_CU, KG, FRAG, true>(a, ctx);
    }
    if constexpr (BM < 256) return launchTileRuns<BM, BN, WAVES_M, WAVES_N, STAGES, BLOCKS_PER_CU, KG, FRAG, false>(a, ctx);
    return hipErrorInvalidValue;
}

// The tiles, by number (THIP_FC_TILE forces one).
enum : int { kTile64 = 1, kTile64TwoGroups = 2, kTile128 = 3, kTile128Deep = 4, kTile256 = 5 };

template <bool FRAG>
static hipError_t launchTileChoice(const FcBf16Args &a, int choice, const LaunchCtx &ctx) {
    switch (choice) {
    case kTile64: return launchTile<64, 64, 2, 2, 4, 2, 1, FRAG>(a, ctx);
    case kTile64TwoGroups: return launchTile<64, 64, 2, 2, 4, 1, 2, FRAG>(a, ctx);
    case kTile128: return launchTile<128, 128, 2, 2, 2, 2, 1, FRAG>(a, ctx);
    case kTile128Deep: return launchTile<128, 128, 2, 2, 4, 1, 1, FRAG>(a, ctx);
    case kTile256: return launchTile<256, 256, 2, 4, 2, 1, 1, FRAG>(a, ctx);
    default: return hipErrorInvalidValue;
    }
}

// Which tile, or 0 for the streaming kernel: the smallest estimate, in us, of a fixed part (launch, ring fill, epilogue)
// plus rounds of 256 workgroups times k-tiles times what a CU takes per k-tile: 0.2, 0.47 and 1.2 us for 16, 32 and 64 KB.
// Fitted to 80 shapes (33 .. 4096 rows, K 72 .. 6912, 128 .. 8192 columns), all of which take a tile within a fifth of their best; some
// of them, us on the streaming kernel / 64 / 64 two groups / 128 / 128 deep / 256:
//   2048 x 1152 -> 6912  154.8 /  53 /  54 / 39.9 / 49.1 / 34.4      1024 x 1152 -> 6912  80.8 / 28.9 / 30 / 21.4 / 24.3 / 28.6
//    512 x 6912 -> 1152   58.7 / 25.3 / 21.9 / 62.8 / 44.6 / 123      128 x 4096 -> 128    7.2 / 16.0 / 13.1 / 27.0 / 27.5 / 72
//     64 x 256 -> 640      6.0 /  3.7 /  3.9 /  5.5 /  5.5 / 9       4096 x 256 -> 256     9.6 /  4.0 /  4.2 / 5.6 / 5.9 / 11.3
int fcBf16TileChoice(const FcBf16Args &a, const LaunchCtx &ctx) {
    if ((long long)a.K * 2 * 256 >= (1LL << 32)) return 0;  // 32-bit offsets inside a tile
    if (ctx.tuning->fcTile >= 0) return ctx.tuning->fcTile;
    if (a.M <= 32) return 0;  // one row block: the weights are streamed once as it is
    const double kt = (a.K + 63) / 64;
    auto tiles = [&](int bm, int bn) { return (double)((a.M + bm - 1) / bm) * ((a.N + bn - 1) / bn); };
    auto rounds = [](double t) { return (double)(long long)((t + 255) / 256); };
    const double t64 = tiles(64, 64), t128 = tiles(128, 128), r256 = rounds(tiles(256, 256));
    const double cost[] = {
        5.5 + 0.08 * kt / a.ksplit + (a.ksplit > 1 ? 1.0 : 0.0) + tiles(32, 32) * kt * 8192 / 11e6,
        3.0 + rounds(t64) * kt * 0.2,
        t64 <= 256 ? 3.5 + kt * 0.17 : 1e30,
        5.0 + rounds(t128) * kt * 0.47,
        t128 <= 256 ? 5.3 + kt * 0.38 : 1e30,
        r256 * (kt * 1.2 + 9.0),
    };
    return (int)(std::min_element(cost, cost + 6) - cost);
}

hipError_t launchFcBf16Tile(const FcBf16Args &a, int choice, const LaunchCtx &ctx) {
    return a.w_fragments == 1 ? launchTileChoice<true>(a, choice, ctx) : launchTileChoice<false>(a, choice, ctx);
}

}  // namespace thip
