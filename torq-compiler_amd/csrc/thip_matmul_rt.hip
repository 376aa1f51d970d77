// gfx950 kernel of torq_hl.matmul on int8 with a second operand that is produced at run time: igemm_rt_i8, a batch of
// products in one launch, input2 read as it lies in memory.
#include "thip_kernels_common.h"

namespace thip {

// ---------------------------------------------------------------------------
// igemm_rt_i8: out[b][m][n] = R1(sum_k A[b][m][k] * B[b][k][n]) with ONE (bias, scale) pair, int8 / int16 / int32 results.
//
// The MFMA wants 16 consecutive k of one column, and B has its columns side by side.  The records say so with a transpose
// per batch into [N][Kp] and a GEMM per batch behind it: two launches per batch element, 5 us each whatever their size
// (4 x 1024x128x1024 -> int16: eight launches, 47 us for 9.4 MB of operands).  Here a workgroup transposes the B tile on its
// way into LDS: a thread loads the dwords of 16 rows of four columns (a wave: two runs of 128 bytes per row) and turns them with
// 32 v_perm_b32 into the 16-byte chunks of four LDS rows, 1/BM of an instruction per product.  Batches are part of the grid.
//
// LDS rows are 128 bytes of K; chunk c of row r sits at slot c ^ swizzle(r): (r >> 1) & 7 for A, whose rows are written 8
// lanes at a time; for B, whose writes go to every fourth row, also bit 4 of the row, so that the eight lanes of a write phase
// and the 16 rows of a read phase both fall into distinct banks.  Two buffers; the loads of a k-tile are in flight during the
// MFMAs of the one before.  What lies beyond K is zero in B only; bytes beyond the tensors are never read.
//
// Bound by latency (one k-tile for K <= 128: load, MFMA, store, nothing to overlap but other workgroups) and then by
// the stores: 4 x 1024x128x1024 -> int16 5.9 us.  MFMA operands, accumulator layout and requant tails are those of igemm_dense_i8.
// ---------------------------------------------------------------------------
template <int BM, int WAVES_M, int WAVES_N, int OUT>
__global__ __launch_bounds__(256, 2) void igemm_rt_i8(MatmulRtArgs p) {
    constexpr int BN = 128, LA = BM / 32;
    constexpr int WTM = BM / WAVES_M, WTN = BN / WAVES_N, TM = WTM / 32, TN = WTN / 32;
    constexpr int A_BYTES = BM * 128, BUF = (BM + BN) * 128;
    static_assert(WAVES_M * WAVES_N == 4, "four waves");
    extern __shared__ __attribute__((aligned(16))) int8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WAVES_N, wn = wave % WAVES_N;
    // each XCD gets a contiguous range of (batch, column tile, row tile)
    const int tilesM = (p.M + BM - 1) / BM, tilesN = (p.N + BN - 1) / BN;
    int lin;
    {
        const int nb = (int)gridDim.x, pid = (int)blockIdx.x;
        const int per = nb / 8, rem = nb % 8, xcd = pid % 8, idx = pid / 8;
        lin = xcd * per + (xcd < rem ? xcd : rem) + idx;
    }
    const int batch = lin / (tilesM * tilesN), tile = lin - batch * (tilesM * tilesN);
    const int n0 = (tile / tilesM) * BN, m0 = (tile % tilesM) * BM;
    // Offsets are from the start of the tensors, below 2^31 (matmulRtFits); the last ones at which a whole chunk / word still
    // lies inside:
    const int aLast = (int)p.a_bytes - 16, bLast = (int)p.b_bytes - 4;
    const int KT = (p.K + 127) / 128;

    const int bg = tid & 31, bc = tid >> 5;  // this thread's four columns and 16-row chunk of the B tile
    const int bn = n0 + 4 * bg;
    int aOff[LA];  // of this thread's chunks in k-tile 0
#pragma unroll
    for (int i = 0; i < LA; i++) {
        const int id = tid + 256 * i, row = m0 + (id >> 3) < p.M ? m0 + (id >> 3) : p.M - 1;
        aOff[i] = (int)(batch * p.a_stride) + row * p.K + (id & 7) * 16;
    }
    const int bBase = (int)(batch * p.b_stride) + bn;
    v4i ra[LA];
    uint32_t rb[16];
    // Loads only, no branch and no use of what is loaded: a load that would pass the end of its tensor starts as much
    // earlier, and store() moves its bytes to where they belong.
    auto load = [&](int kt) {
#pragma unroll
        for (int i = 0; i < LA; i++) {
            const int off = aOff[i] + kt * 128;
            ra[i] = ((const UnalignedV4 *)(p.A + (uint32_t)(off < aLast ? off : aLast)))->v;
        }
        const int k0 = kt * 128 + bc * 16;
        int off = bBase + (k0 < p.K ? k0 : p.K) * p.N;
#pragma unroll
        for (int r = 0; r < 16; r++) {
            rb[r] = ((const UnalignedU32 *)(p.B + (uint32_t)(off < bLast ? off : bLast)))->v;
            off = off < bLast ? off + p.N : off;
        }
    };
    auto store = [&](int kt, int8_t *buf) {
#pragma unroll
        for (int i = 0; i < LA; i++) {
            const int id = tid + 256 * i, row = id >> 3, past = aOff[i] + kt * 128 - aLast;
            if (past > 0 && past < 16) {  // the tensor's last bytes, and only where K is no multiple of 16
                uint32_t w[8] = {(uint32_t)ra[i][0], (uint32_t)ra[i][1], (uint32_t)ra[i][2], (uint32_t)ra[i][3], 0, 0, 0, 0};
                for (int e = 0; e < past; e++) {
#pragma unroll
                    for (int d = 0; d < 4; d++) w[d] = (w[d] >> 8) | (w[d + 1] << 24);
                }
                ra[i] = v4i{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
            }
            *(v4i *)(buf + row * 128 + (((id & 7) ^ ((row >> 1) & 7)) << 4)) = ra[i];
        }
        // rows beyond K are zero, and among the last ones (several where N < 4) a word may have started early
        const int k0 = kt * 128 + bc * 16;
        if (kt * 128 + 132 > p.K) {
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int past = bBase + (k0 < p.K ? k0 + r : 0) * p.N - bLast;
                if (past > 0) rb[r] >>= 8 * (past & 3);  // 1 .. 3 where the word holds a column at all
                rb[r] = k0 + r < p.K ? rb[r] : 0;
            }
        }
        uint32_t o[4][4];
#pragma unroll
        for (int a = 0; a < 4; a++) transpose4x4(rb[4 * a], rb[4 * a + 1], rb[4 * a + 2], rb[4 * a + 3], o[a]);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int row = 4 * bg + j, swz = ((row >> 1) & 7) ^ ((row >> 4) & 1);
            *(v4i *)(buf + A_BYTES + row * 128 + ((bc ^ swz) << 4)) = v4i{(int)o[0][j], (int)o[1][j], (int)o[2][j], (int)o[3][j]};
        }
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
    load(0);
    store(0, smem);
    __syncthreads();
    for (int kt = 0; kt < KT; kt++) {
        if (kt + 1 < KT) load(kt + 1);
        const int8_t *buf = smem + (kt & 1) * BUF;
        const int steps = p.K - kt * 128 < 128 ? (p.K - kt * 128 + 31) / 32 : 4;
#pragma unroll
        for (int s = 0; s < 4; s++) {
            if (s >= steps) break;
            v4i af[TM], bf[TN];
#pragma unroll
            for (int i = 0; i < TM; i++) {
                const int row = wm * WTM + i * 32 + fr;
                af[i] = *(const v4i *)(buf + row * 128 + (((2 * s + half) ^ ((row >> 1) & 7)) << 4));
            }
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const int row = wn * WTN + j * 32 + fr, swz = ((row >> 1) & 7) ^ ((row >> 4) & 1);
                bf[j] = *(const v4i *)(buf + A_BYTES + row * 128 + (((2 * s + half) ^ swz) << 4));
            }
#pragma unroll
            for (int j = 0; j < TN; j++) {
#pragma unroll
                for (int i = 0; i < TM; i++) acc[j][i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(bf[j], af[i], acc[j][i], 0, 0, 0);
            }
        }
        if (kt + 1 < KT) store(kt + 1, smem + ((kt + 1) & 1) * BUF);  // the other buffer: its readers met the barrier a k-tile ago
        __syncthreads();
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

template <int BM, int WAVES_M, int WAVES_N, int OUT>
static hipError_t launchRt(const MatmulRtArgs &a, const LaunchCtx &ctx) {
    auto kernel = igemm_rt_i8<BM, WAVES_M, WAVES_N, OUT>;
    constexpr size_t lds = 2 * (size_t)(BM + 128) * 128;
    const long long tiles = (long long)a.batches * ((a.M + BM - 1) / BM) * ((a.N + 127) / 128);
    if (tiles > 0x7fffffffLL) return hipErrorInvalidValue;
    THIP_ENQUEUE(ctx, kernelLabel("igemm_rt_i8", {BM, WAVES_M, WAVES_N, OUT}), kernel, dim3((unsigned)tiles), dim3(256), lds, a);
    return hipGetLastError();
}

// Rows of a tile.  A k-tile takes a workgroup about 1.3 us whatever its rows (the loads' latency), so up to one workgroup per
// CU the smallest tile is ahead (1 x 1024x128x1024: 3.9 us on 32 rows, 4.5 on 64, 5.3 on 128); beyond that 64 rows (4 x
// 1024x128x1024: 6.9, 5.9, 6.2), and from three workgroups of these per CU the operands' traffic counts (2 x 2000x1024x2000,
// int32: 35.2, 27.9, 21.9).
template <int OUT>
static hipError_t launchRtOut(const MatmulRtArgs &a, const LaunchCtx &ctx) {
    auto tiles = [&](int bm) { return (long long)a.batches * ((a.M + bm - 1) / bm) * ((a.N + 127) / 128); };
    if (a.M <= 32 || tiles(32) <= 256) return launchRt<32, 1, 4, OUT>(a, ctx);
    if (tiles(64) <= 768) return launchRt<64, 2, 2, OUT>(a, ctx);
    return launchRt<128, 2, 2, OUT>(a, ctx);
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
