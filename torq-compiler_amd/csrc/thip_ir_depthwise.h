// The 3 x 3 depthwise convolution as a product of matrix instructions, of 32 channels in LDS: what ir_expand_dw_i8 and ir_block_i8 share.
#pragma once

#include "thip_kernels_common.h"

namespace thip {

// A cell holds 16 bytes of a pixel in each of two planes, channel 8 a + 4 j + e at byte 4 a + e of plane j.  Of a plane, 16 channels x 16 pixels are one
// v_mfma_i32_16x16x64_i8 per window row: its K are the 16 channels at the window's three columns (and 16 zeros), the lanes of a group have a column's cells, and
// the weights are diagonals of 16 x 16 blocks.  slot, group: lane & 15, lane >> 4.  A lane's results are the channels 8 group + 4 j + e of pixel `slot`.

// Where a lane's dword of taps (byte kw: tap kw) lies among those of a chunk's plane, dwords.  `whole`: the chunk has all 32 channels; of half a chunk the other
// lanes take the first one's.
__device__ __forceinline__ uint32_t depthwiseTapAt(bool whole, int slot) { return whole || slot < 8 ? 8 * (slot >> 2) + (slot & 3) : 0; }

__device__ __forceinline__ void depthwiseWeights(const uint32_t (&taps)[2][3], int slot, int group, v4i (&w)[2][3]) {
#pragma unroll
    for (int j = 0; j < 2; j++) {
#pragma unroll
        for (int kh = 0; kh < 3; kh++) {
            const uint32_t tap = group < 3 ? (taps[j][kh] >> (8 * group) & 0xffu) << (8 * (slot & 3)) : 0u;
#pragma unroll
            for (int d = 0; d < 4; d++) w[j][kh][d] = d == (slot >> 2) ? (int)tap : 0;
        }
    }
}

// A row of cells under the lane's column of the window; src goes on to the next one.
__device__ __forceinline__ void depthwiseRow(const int8_t *&src, int planeBytes, int rowBytes, v4i (&cells)[2]) {
#pragma unroll
    for (int j = 0; j < 2; j++) cells[j] = *(const v4i *)(src + j * planeBytes);
    src += rowBytes;
}

// The requantised results of a window of three rows.
template <int MODE>
__device__ __forceinline__ v2i depthwiseResults(const v4i (&w)[2][3], const v4i (&r0)[2], const v4i (&r1)[2], const v4i (&r2)[2], const v4i (&bias)[2], const v4i (&scale)[2], const Requant &rq,
                                                const WideRequant &wide) {
    v2i o;
#pragma unroll
    for (int j = 0; j < 2; j++) {
        v4i acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[j][0], r0[j], bias[j], 0, 0, 0);
        acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[j][1], r1[j], acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[j][2], r2[j], acc, 0, 0, 0);
        o[j] = (int)requantPack4<MODE>(acc, scale[j], 0, rq, wide);
    }
    return o;
}

}  // namespace thip
