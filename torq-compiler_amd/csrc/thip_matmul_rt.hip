// gfx950 kernel of torq_hl.matmul on int8 with a second operand that is produced at run time: igemm_rt_i8, a batch of
// products in one launch, input2 read as it lies in memory.
#include <mutex>

#include "thip_kernels_common.h"

namespace thip {

// Bytes of LDS from one row of B to the next.
constexpr int rtRowB(int BM) { return BM > 64 ? 160 : 128; }

// ds_read_b64_tr_b8: of 16 lanes' 8 bytes each, as 8 rows of 16, a lane gets a column.
__device__ __forceinline__ v2i readTransposed(const int8_t *p) {
    return __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) v2i *)p);
}

// ---------------------------------------------------------------------------
// igemm_rt_i8: out[b][m][n] = R1(sum_k A[b][m][k] * B[b][k][n]) with ONE (bias, scale) pair, int8 / int16 / int32 results.
//
// The MFMA wants 16 consecutive k of one column, and B has its columns side by side.  The records say so with a transpose
// per batch into [N][Kp] and a GEMM per batch behind it: two launches per batch element, 5 us each whatever their size
// (4 x 1024x128x1024 -> int16: eight launches, 47 us for 9.4 MB of operands).  Here a workgroup copies the B tile into LDS as it
// lies, 16 bytes of a row at a time, and ds_read_b64_tr_b8 turns it on the way into the MFMA's registers.  Batches are part of the grid.
//
// LDS rows of A are 128 bytes of K, chunk c of row r at slot c ^ ((r >> 1) & 7); those of B are 128 columns, chunk c of row r at slot
// c ^ (r & 7), or (tiles of 128 rows) at slot c of rows 160 bytes apart: the 8 rows of 32 columns that 32 lanes read fall into distinct
// banks.  Two buffers, or two groups of waves (KG) with one each, which make every other k-tile and add up at the end; the loads of a
// k-tile are in flight during the MFMAs of the one before.  What lies beyond K is zero in B only; bytes beyond the tensors are never read.
//
// Bound by a wave's issue (about one instruction in 5 cycles while it is alone on its SIMD: turning B with v_perm_b32 behind dword loads, 100 more
// instructions a k-tile, took 0.8 us a k-tile where this takes 0.4; more k-tiles in flight change nothing) and then by the stores.  With v_perm_b32
// and one group / now, us: 1 x 1024x1024x1024 10.0 / 5.7, 1 x 1x1024x1024 9.8 / 5.4, 16 x 32x512x64 6.4 / 4.2, 8 x 512x256x512 5.3 / 4.5,
// 4 x 1024x128x1024 -> int16 5.77 / 5.40, 2 x 2048x1024x2048 -> int32 20.0 / 19.8.  Rows of B without a gap leave room for three workgroups of 64 rows
// and two buffers a CU, 160 bytes apart for two: 8 x 1472x1024x512 (736 tiles of 64 rows) 16.3 / 13.2, 2 x 2304x256x1024 (576) 8.1 / 6.7.  Of 128 rows there
// are two either way, and the slots' addresses cost 2 % (2 x 2048x1024x2048 -> int32 19.5 / 19.9).
// MFMA operands, accumulator layout and requant tails are those of igemm_dense_i8.
// ---------------------------------------------------------------------------
// FEW: B has fewer bytes than a chunk, and so one k-tile; all of them are read one by one, as a chunk from the tensor's start.  A test in the
// other kernels cost 4 x 1024x128x1024 -> int16 0.8 %.
template <int BM, int WAVES_M, int WAVES_N, int OUT, int KG, bool FEW>
__global__ __launch_bounds__(256 * KG, 2) void igemm_rt_i8(MatmulRtArgs p, FastDiv divTiles, FastDiv divTilesM) {
    constexpr int BN = 128, LA = BM / 32, BUFS = KG == 1 ? 2 : 1;
    constexpr int WTM = BM / WAVES_M, WTN = BN / WAVES_N, TM = WTM / 32, TN = WTN / 32;
    constexpr int A_BYTES = BM * 128, ROWB = rtRowB(BM), TURN = ROWB == 128 ? 7 : 0, BUF = A_BYTES + 128 * ROWB;
    static_assert(WAVES_M * WAVES_N == 4, "four waves");
    extern __shared__ __attribute__((aligned(16))) int8_t smem[];
    const int tid = threadIdx.x & 255, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // in the group
    const int group = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8);
    const int wm = wave / WAVES_N, wn = wave % WAVES_N;
    // each XCD gets a contiguous range of (batch, column tile, row tile)
    int lin;
    {
        const int nb = (int)gridDim.x, pid = (int)blockIdx.x;
        const int per = nb / 8, rem = nb % 8, xcd = pid % 8, idx = pid / 8;
        lin = xcd * per + (xcd < rem ? xcd : rem) + idx;
    }
    const int batch = (int)fastDiv((uint32_t)lin, divTiles), tile = lin - batch * (int)divTiles.d;
    const int tileN = (int)fastDiv((uint32_t)tile, divTilesM), n0 = tileN * BN, m0 = (tile - tileN * (int)divTilesM.d) * BM;
    // Offsets are from the start of the tensors, which end below 2^31, and of 32 bits (matmulRtFits); the last ones at which a
    // whole chunk still lies inside:
    const int aLast = (int)p.a_bytes - 16;
    const uint32_t bLast = FEW ? 0 : (uint32_t)p.b_bytes - 16;
    const int KT = (p.K + 128 * KG - 1) / (128 * KG);  // k-tiles of a group: group, group + KG, ...

    // chunk `chunk` of every 32nd row of both tiles is this thread's; offsets of those of k-tile 0
    const int chunk = tid & 7, row0 = tid >> 3;
    int aOff[LA];
#pragma unroll
    for (int i = 0; i < LA; i++) {
        const int row = m0 + row0 + 32 * i;
        aOff[i] = (int)(batch * p.a_stride) + (row < p.M ? row : p.M - 1) * p.K + chunk * 16;
    }
    const uint32_t bOff = (uint32_t)(batch * p.b_stride) + (uint32_t)(n0 + chunk * 16) + (uint32_t)row0 * (uint32_t)p.N;
    v4i ra[LA], rb[4];
    // Loads only, no branch and no use of what is loaded: a load that would pass the end of its tensor starts as much
    // earlier, and store() moves its bytes to where they belong.
    auto load = [&](int kt) {
#pragma unroll
        for (int i = 0; i < LA; i++) {
            const int off = aOff[i] + kt * 128;
            ra[i] = ((const UnalignedV4 *)(p.A + (uint32_t)(off < aLast ? off : aLast)))->v;
        }
        if constexpr (FEW) {
            uint32_t few[4] = {0, 0, 0, 0};
#pragma unroll
            for (int e = 0; e < 15; e++) few[e / 4] |= e < (int)p.b_bytes ? (uint32_t)(uint8_t)p.B[e] << (8 * (e % 4)) : 0u;
            rb[0] = v4i{(int)few[0], (int)few[1], (int)few[2], (int)few[3]};
            rb[1] = rb[2] = rb[3] = v4i{0, 0, 0, 0};  // K < 16
            return;
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int k = kt * 128 + 32 * i;
            const uint32_t off = bOff + (uint32_t)(k < p.K ? k : p.K) * (uint32_t)p.N;
            rb[i] = ((const UnalignedV4 *)(p.B + (off < bLast ? off : bLast)))->v;
        }
    };
    auto store = [&](int kt, int8_t *buf) {
        if (kt * 128 + 144 > p.K) {  // K's end, and where N < 16 the rows whose chunk passes the end of the tensor, lie no further away
            auto moved = [](v4i v, int past) {
                if (past <= 0 || past >= 16) return v;
                unsigned __int128 bytes;
                __builtin_memcpy(&bytes, &v, 16);
                bytes >>= 8 * past;
                __builtin_memcpy(&v, &bytes, 16);
                return v;
            };
#pragma unroll
            for (int i = 0; i < LA; i++) ra[i] = moved(ra[i], aOff[i] + kt * 128 - aLast);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int k = kt * 128 + 32 * i;
                rb[i] = k + row0 < p.K ? moved(rb[i], (int)(bOff + (uint32_t)k * (uint32_t)p.N - bLast)) : v4i{0, 0, 0, 0};
            }
        }
#pragma unroll
        for (int i = 0; i < LA; i++) {
            const int row = row0 + 32 * i;
            *(v4i *)(buf + row * 128 + ((chunk ^ ((row >> 1) & 7)) << 4)) = ra[i];
        }
#pragma unroll
        for (int i = 0; i < 4; i++) *(v4i *)(buf + A_BYTES + (row0 + 32 * i) * ROWB + ((chunk ^ (row0 & TURN)) << 4)) = rb[i];
    };
    v16i acc[TN][TM];
#pragma unroll
    for (int j = 0; j < TN; j++) {
#pragma unroll
        for (int i = 0; i < TM; i++) {
#pragma unroll
            for (int r = 0; r < 16; r++) acc[j][i][r] = 0;
        }
    }
    const int fr = lane & 31, half = lane >> 5;
    int8_t *const own = smem + group * (BUFS * BUF);
    // of an operand's 16 columns and 8 rows a lane reads 8 bytes of row (lane & 15) / 2 and gets its column's
    int turned[TN];
#pragma unroll
    for (int j = 0; j < TN; j++) turned[j] = A_BYTES + (16 * half + ((lane & 15) >> 1)) * ROWB + 8 * (lane & 1) + 16 * ((2 * (wn * TN + j) + (lane >> 4 & 1)) ^ (lane >> 1 & TURN));
    auto multiply = [&](int steps, const int8_t *buf) {
#pragma unroll
        for (int s = 0; s < 4; s++) {
            if (s >= steps) continue;
            v4i af[TM], bf[TN];
#pragma unroll
            for (int i = 0; i < TM; i++) {
                const int row = wm * WTM + i * 32 + fr;
                af[i] = *(const v4i *)(buf + row * 128 + (((2 * s + half) ^ ((row >> 1) & 7)) << 4));
            }
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const int8_t *at = buf + turned[j] + 32 * s * ROWB;
                const v2i low = readTransposed(at), high = readTransposed(at + 8 * ROWB);
                bf[j] = v4i{low[0], low[1], high[0], high[1]};
            }
#pragma unroll
            for (int j = 0; j < TN; j++) {
#pragma unroll
                for (int i = 0; i < TM; i++) acc[j][i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(bf[j], af[i], acc[j][i], 0, 0, 0);
            }
        }
    };
    load(group);
    store(group, own);
    const int8_t *last = own;
    if (KT > 1) {
        load(KG + group);
        __syncthreads();
        for (int it = 1; it < KT; it++) {
            multiply(4, last);  // whole k-tiles, all but a group's last one
            if (BUFS == 1) __syncthreads();
            // two buffers: the readers of the other one met the barrier a k-tile ago
            int8_t *next = own + (BUFS == 2 ? (it & 1) * BUF : 0);
            store(it * KG + group, next);
            load((it + 1) * KG + group);  // past the last one nobody uses it: behind a branch the compiler waits for it at once
            last = next;
            __syncthreads();
        }
    } else {
        __syncthreads();
    }
    const int rest = p.K - ((KT - 1) * KG + group) * 128;
    multiply(rest < 128 ? (rest + 31) / 32 : 4, last);  // none for a group whose k-tiles have ended
    if constexpr (KG > 1) {
        // the second group's sums through LDS, 16 bytes a lane; the first one adds them to its own and goes on
        static_assert(KG == 2, "one group besides the first");
        v4i *const sums = (v4i *)smem;
        __syncthreads();
        if (group > 0) {
#pragma unroll
            for (int j = 0; j < TN; j++) {
#pragma unroll
                for (int i = 0; i < TM; i++) {
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        sums[(j * TM + i) * 1024 + q * 256 + tid] = v4i{acc[j][i][4 * q], acc[j][i][4 * q + 1], acc[j][i][4 * q + 2], acc[j][i][4 * q + 3]};
                    }
                }
            }
        }
        __syncthreads();
        if (group > 0) return;
#pragma unroll
        for (int j = 0; j < TN; j++) {
#pragma unroll
            for (int i = 0; i < TM; i++) {
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const v4i v = sums[(j * TM + i) * 1024 + q * 256 + tid];
#pragma unroll
                    for (int e = 0; e < 4; e++) acc[j][i][4 * q + e] = (int)((uint32_t)acc[j][i][4 * q + e] + (uint32_t)v[e]);
                }
            }
        }
    }

    // Register 4 q + e of lane (fr, half) is out[m = fr][n = 8 q + 4 half + e] of a 32 x 32 tile.  Results narrower than 32 bits
    // change places between the wave halves so that a lane stores 16 consecutive bytes.
    constexpr int ELEM = OUT == kDtypeI8 ? 1 : OUT == kDtypeI16 ? 2 : 4;
    int8_t *out = (int8_t *)p.out + (size_t)batch * p.out_stride * ELEM;
    const long long rnd = roundTerm(p.rq.shift);
    const WideRequant wrq = wideRequant(p.rq);
    // clamp(t + zp, min, max) = clamp(t, min - zp, max - zp) + zp for a product that is neither scaled nor shifted
    const long long lo64 = (long long)p.rq.out_min - p.rq.out_zp, hi64 = (long long)p.rq.out_max - p.rq.out_zp;
    const int32_t lo = (int32_t)(lo64 < INT32_MIN ? INT32_MIN : lo64), hi = (int32_t)(hi64 > INT32_MAX ? INT32_MAX : hi64);
    auto finish = [&](auto requantOne) {
#pragma unroll
        for (int j = 0; j < TN; j++) {
            const int nt = n0 + wn * WTN + j * 32;
#pragma unroll
            for (int i = 0; i < TM; i++) {
                const int m = m0 + wm * WTM + i * 32 + fr;
                int32_t v[16];
#pragma unroll
                for (int r = 0; r < 16; r++) v[r] = requantOne((int32_t)((uint32_t)acc[j][i][r] + (uint32_t)p.bias));
                constexpr int STORES = ELEM, PER = 16 / ELEM;  // 16-byte stores of a lane, elements in each
                v4i w[STORES];
                int nOf[STORES];  // first column of each, within the tile
                if constexpr (OUT == kDtypeI8) {
                    uint32_t d[4];
#pragma unroll
                    for (int q = 0; q < 4; q++) d[q] = packBytes(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
                    const auto s02 = __builtin_amdgcn_permlane32_swap(d[0], d[2], false, false);
                    const auto s13 = __builtin_amdgcn_permlane32_swap(d[1], d[3], false, false);
                    w[0] = v4i{(int)s02[0], (int)s02[1], (int)s13[0], (int)s13[1]};
                    nOf[0] = 16 * half;
                } else if constexpr (OUT == kDtypeI16) {
                    uint32_t d[8];
#pragma unroll
                    for (int t = 0; t < 8; t++) d[t] = __builtin_amdgcn_perm((uint32_t)v[2 * t + 1], (uint32_t)v[2 * t], 0x05040100u);
#pragma unroll
                    for (int h = 0; h < 2; h++) {
                        const auto s0 = __builtin_amdgcn_permlane32_swap(d[4 * h], d[4 * h + 2], false, false);
                        const auto s1 = __builtin_amdgcn_permlane32_swap(d[4 * h + 1], d[4 * h + 3], false, false);
                        w[h] = v4i{(int)s0[0], (int)s1[0], (int)s0[1], (int)s1[1]};
                        nOf[h] = 16 * h + 8 * half;
                    }
                } else {
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        w[q] = v4i{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
                        nOf[q] = 8 * q + 4 * half;
                    }
                }
                if (m >= p.M) continue;
#pragma unroll
                for (int s = 0; s < STORES; s++) {
                    const int n = nt + nOf[s];
                    if (n >= p.N) continue;
                    int8_t *dst = out + ((size_t)m * p.N + n) * ELEM;
                    if (n + PER <= p.N) {
                        ((UnalignedV4 *)dst)->v = w[s];
                    } else {
#pragma unroll
                        for (int e = 0; e < PER; e++) {
                            const uint32_t word = (uint32_t)w[s][e * ELEM / 4] >> (8 * (e * ELEM % 4));
                            if (n + e < p.N) {
                                if constexpr (OUT == kDtypeI8) dst[e] = (int8_t)word;
                                else if constexpr (OUT == kDtypeI16) ((int16_t *)dst)[e] = (int16_t)word;
                                else ((int32_t *)dst)[e] = (int32_t)word;
                            }
                        }
                    }
                }
            }
        }
    };
    if (p.scale == 1 && p.rq.shift == 0) {
        finish([&](int32_t t) { return (int32_t)((uint32_t)med3(t, lo, hi) + (uint32_t)p.rq.out_zp); });
    } else {
        withRequantMode(wrq, [&](auto tag) { finish([&](int32_t t) { return requantT0<decltype(tag)::value>(t, p.scale, rnd, p.rq, wrq); }); });
    }
}

template <int BM, int WAVES_M, int WAVES_N, int OUT, int KG, bool FEW = false>
static hipError_t launchRt(const MatmulRtArgs &a, const LaunchCtx &ctx) {
    auto kernel = igemm_rt_i8<BM, WAVES_M, WAVES_N, OUT, KG, FEW>;
    constexpr size_t buffer = BM * 128 + 128 * rtRowB(BM);
    if constexpr (2 * buffer > 64 * 1024) {
        static std::once_flag once;
        static hipError_t configured = hipSuccess;
        std::call_once(once, [&] { configured = hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)(2 * buffer)); });
        if (configured != hipSuccess) return configured;
    }
    const size_t lds = (KG > 1 || a.K > 128 ? 2 : 1) * buffer;
    const long long tilesM = (a.M + BM - 1) / BM, tiles = tilesM * ((a.N + 127) / 128);
    if (tiles * a.batches > 0x7fffffffLL) return hipErrorInvalidValue;
    THIP_ENQUEUE(ctx, kernelLabel("igemm_rt_i8", {BM, WAVES_M, WAVES_N, OUT, KG, (int)FEW}), kernel, dim3((unsigned)(tiles * a.batches)), dim3(256 * KG), lds, a,
                 makeFastDiv((uint32_t)tiles), makeFastDiv((uint32_t)tilesM));
    return hipGetLastError();
}

// Rows of a tile, us.  Up to one workgroup per CU the smallest tile is ahead (1 x 1024x1024x1024: 6.7 on 32 rows, 7.6 on 64, 9.6 on 128), and a second
// group of waves where there is a second k-tile for it (5.7; four groups 5.7, and behind two on 2 x 300x700x300: 5.1, 5.6); beyond that 64 rows
// (3 x 777x333x555 -> int16: 7.6, 6.6, 8.9; 8 x 512x256x512 4.7, 4.5, 5.5; 4 x 1024x128x1024 -> int16 5.6, 5.4, 6.1) as long as all of them run at once: three a CU
// hold two buffers of 24 KB each.  64 / 128 rows at 544 tiles of 64 rows 8 x 4352x256x128 6.8 / 7.0, at 664 2 x 10621x512x256 -> int32 12.3 / 14.0, at 736
// 4 x 2941x1024x512 -> int32 16.9 / 17.5, at 816 4 x 3264x256x512 8.8 / 7.0, at 1024 8 x 1024x1024x1024 17.7 / 15.0.  Of 84 drawn products of 257 .. 768 tiles two are
// faster on 128 rows by more than 1 %, of 40 of more tiles eleven on 64 (short K, or 2 x 8512x512x512 -> int32, 1064 tiles, 18.1 / 20.8).
template <int OUT>
static hipError_t launchRtOut(const MatmulRtArgs &a, const LaunchCtx &ctx) {
    auto tiles = [&](int bm) { return (long long)a.batches * ((a.M + bm - 1) / bm) * ((a.N + 127) / 128); };
    if (a.b_bytes < 16) return launchRt<32, 1, 4, OUT, 1, true>(a, ctx);
    if (a.M <= 32 || tiles(32) <= 256) return a.K <= 128 ? launchRt<32, 1, 4, OUT, 1>(a, ctx) : launchRt<32, 1, 4, OUT, 2>(a, ctx);
    if (tiles(64) <= 768) return launchRt<64, 2, 2, OUT, 1>(a, ctx);
    return launchRt<128, 2, 2, OUT, 1>(a, ctx);
}

hipError_t launchMatmulRt(const MatmulRtArgs &a, const LaunchCtx &ctx) {
    if (!a.A || !a.B || !a.out || a.batches <= 0 || a.M <= 0 || a.N <= 0 || a.K <= 0) return hipErrorInvalidValue;
    if (a.a_stride < 0 || a.b_stride < 0 || a.out_stride < 0) return hipErrorInvalidValue;
    // every byte a tile may read lies in the tensors the record was checked against, at an offset of 31 bits
    if (a.a_bytes < (int64_t)(a.batches - 1) * a.a_stride + (int64_t)a.M * a.K || a.b_bytes < (int64_t)(a.batches - 1) * a.b_stride + (int64_t)a.K * a.N) return hipErrorInvalidValue;
    if (!matmulRtFits(a.a_bytes, a.b_bytes, a.M, a.N, a.K)) return hipErrorInvalidValue;
    switch (a.out_dtype) {
    case kDtypeI8: return launchRtOut<kDtypeI8>(a, ctx);
    case kDtypeI16: return launchRtOut<kDtypeI16>(a, ctx);
    case kDtypeI32: return launchRtOut<kDtypeI32>(a, ctx);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace thip
