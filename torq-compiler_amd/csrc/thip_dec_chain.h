// A run of decode-shaped records (grouped linears and batched small matmuls, each reading what one before it wrote) as one launch:
// the table that the kernel walks, shared by the planner (host only) and the kernel.
#pragma once

#include <stdint.h>

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
    uint32_t *sync;      // word 0 launches done, word 32 set by a workgroup that gave up, word 64 workgroups done, from word 96 on the exchange
    int32_t count, xRoom, redRoom;  // phases; bytes of LDS for input rows and for partial sums
    uint32_t byGridMul, byGridShift;  // division by the workgroups of the launch
    uint64_t waitTicks;  // of the 100 MHz clock: how long a workgroup waits for the others before it gives up
    uint8_t *bindings[64];
};
constexpr uint64_t kChainSyncHead = 96;  // words in front of the exchange

}  // namespace thip
