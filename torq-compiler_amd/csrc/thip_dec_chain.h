// A run of decode-shaped records (grouped linears and batched small matmuls, each reading what one before it wrote) as one launch:
// the table that the kernel walks and the index arithmetic of its weights, shared by the planner (host only) and the kernel.
#pragma once

#include "thip_kernels.h"

namespace thip {

constexpr int kChainWaves = 9;         // waves of a workgroup that multiply
constexpr int kChainPollers = 2;       // waves that bring the input rows; one more adds up and stores
constexpr int kChainRing = 4;          // units of weights that a wave holds in registers ahead of their use
constexpr int kChainResults = 4;       // matrix tiles that a workgroup makes between two collections of partial sums
constexpr int kChainMaxRows = 4;       // input rows of a linear
constexpr int kChainMaxHeads = 16;     // and of a matmul
constexpr int kChainMaxPhases = 256;
constexpr int kChainMinPhases = 2;
constexpr int kChainWorkgroups = 256;  // of a launch, as it is planned: one per CU
constexpr int kChainLds = 156 * 1024;  // table, input rows and partial sums of a workgroup

// An operand: an address, or a binding of the dispatch (its index + 1 in the top byte) and the bytes from its start.
typedef uint64_t ChainRef;

// One record.  A job is a tile of at most 16 output columns (of every matrix of a pair); jobs are dealt to the workgroups one
// after the other, a phase going on where the one before it ended: who has few jobs of one phase has time to fetch its weights of the next.
// Its K is walked in `units`: 128 rows of one matrix (linear; two times 128 where two jobs share a tile), or 64 (matmul).
// What a phase makes for another one goes through an exchange: a dword per element, the value and, in the upper half, a
// number of the launch, so that a reader sees by the value itself that it is there.  *Tag: where an operand lies in the exchange, in
// dwords, or -1: it is no result of the chain (x, res), or none of its phases reads it (out, addOut).
struct ChainPhase {
    ChainRef x, w[3], bias[3], out[3], res, addOut;
    int32_t xTag, resTag, outTag[3], addTag;
    int32_t M, K;
    int32_t start;              // the workgroup that has job 0
    int32_t jobs, units, split; // split: jobs per 16-column tile (1 or 2; linear only)
    int32_t perPass;            // jobs of a workgroup between two collections of partial sums
    int32_t nmat, nseg;         // linear: matrices per job (2: a pair), matrices in all
    int32_t N[3];
    int32_t slotBytes;          // linear on block-quantized int8 weights: kDecSlotBytes, or with block biases 64 more; 0: batched matmul against a bf16 operand held [N][K]
    int32_t tiles;              // matmul: 16-column tiles of a batch element
    int32_t aStride, wStride, outStride;  // matmul: elements from one batch element to the next
    uint32_t wBytes;            // matmul: of the operand held [N][K], all batch elements
    float bias0, lo, hi;        // matmul: its one bias; both: the clamp
    int32_t addMode;            // 0: no add; 1: of the result and res; 2: of a pair's two results; 3: of res and the result
    float aw0, aw1, abias, alo, ahi;
    uint32_t unitsMul, unitsShift, tilesMul, tilesShift, itemsMul, itemsShift;  // division by `units`, `tiles` and the elements of a job
};
static_assert(sizeof(ChainPhase) == 256, "a dword for each lane of a wave");

struct DecChainArgs {
    const ChainPhase *phases;
    uint32_t *sync;      // word 0 launches done, word 32 set by a workgroup that gave up, word 64 workgroups done, words kChainTell and the next one the
                         // address of a word of host memory that is set where a workgroup gave up, from word kChainSyncHead on the exchange
    int32_t count, xRoom, redRoom;  // phases; bytes of LDS for input rows and for partial sums
    uint32_t byGridMul, byGridShift;  // division by the workgroups of the launch
    uint64_t waitTicks;  // of the 100 MHz clock: how long a workgroup waits for the others before it gives up
    uint8_t *bindings[64];
};
constexpr uint64_t kChainSyncHead = 96, kChainTell = 66;

// Index arithmetic of the weights, shared by the kernel and a check on the host.

// A job of a linear makes the same tile of a pair's matrices, or a tile of one of up to three.
struct ChainTile {
    int seg, tile;
};
__host__ __device__ inline ChainTile chainTile(int tile, int nmat, int nseg, int tiles0, int tiles1) {
    if (nmat > 1 || nseg < 2 || tile < tiles0) return ChainTile{0, tile};
    if (nseg < 3 || tile < tiles0 + tiles1) return ChainTile{1, tile - tiles0};
    return ChainTile{2, tile - tiles0 - tiles1};
}

// The units of a result, one behind the other: where the first one starts in the operand, how many bytes may be read from there on (a load
// of what lies beyond returns zero and touches no memory), and a unit's bytes; then, from the start of a unit, its scales, from its
// weights the second half of them, and from a scale its bias.
struct ChainUnits {
    uint64_t first;
    uint32_t bytes, unitBytes, scales, half, bias;
};
// A linear's end with their tile: where two jobs share one of an odd number of k-blocks, the second half of the last unit is not there, and
// behind it lies another tile, or what follows the matrix, which may be nothing.
// odd: of a shared tile's two jobs the one with columns 8 .. 15.
__host__ __device__ inline ChainUnits chainLinearUnits(int K, int slotBytes, int split, int tile, int odd) {
    ChainUnits u;
    u.first = (uint64_t)((uint32_t)tile * (uint32_t)(K >> 7)) * (uint32_t)slotBytes + (uint32_t)(odd * 128);
    u.bytes = (uint32_t)(K >> 7) * (uint32_t)slotBytes - (uint32_t)(odd * 128);
    u.unitBytes = (uint32_t)(split * slotBytes);
    u.scales = 2048u - (uint32_t)(odd * 96);
    u.half = 1024;
    u.bias = slotBytes > kDecSlotBytes ? 64 : 0;
    return u;
}
// A matmul's end with the operand.  wBytes: of it; wStride: elements from one batch element to the next.
__host__ __device__ inline ChainUnits chainMatmulUnits(int K, uint32_t wBytes, int wStride, int batch, int tile) {
    ChainUnits u;
    const uint32_t at = ((uint32_t)batch * (uint32_t)wStride + (uint32_t)(tile * 16 * K)) * 2u;
    u.first = at;
    u.bytes = wBytes - at;
    u.unitBytes = 128;
    u.scales = 0;
    u.half = 64;
    u.bias = 0;
    return u;
}
// Where lane (c = lane & 15, g = lane >> 4) finds its weights and its scale in a unit (a lane of a matmul has none).
struct ChainLane {
    uint32_t weights, scales;
};
__host__ __device__ inline ChainLane chainLinearLane(int c, int g, int slotBytes, int split) {
    const int column = split == 1 ? c : c & 7, second = split == 1 ? 0 : c >> 3;
    return ChainLane{(uint32_t)(second * slotBytes + (g * 16 + column) * 16), (uint32_t)(second * slotBytes + column * 4)};
}
__host__ __device__ inline ChainLane chainMatmulLane(int c, int g, int K) { return ChainLane{(uint32_t)((c * K + 8 * g) * 2), 0}; }

}  // namespace thip
