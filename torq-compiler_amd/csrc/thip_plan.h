// From the records of a descriptor to the launches of a dispatch: runs of records that one kernel does as a whole.
// Host-only (no HIP calls).
#pragma once

#include <vector>

#include "thip_validate.h"

namespace thip {

enum StepKind {
    kStepRecord,    // one record, by its own launcher
    kStepExpandDw,  // a pointwise convolution and the depthwise one behind it (ir_expand_dw_i8)
    kStepPadded,    // a GEMM-shaped record whose channels fill no 16-byte chunks: its input padded, then a dense kernel
    kStepMatmulRt,  // a batch of int8 matmuls with a run-time input2: its transposes and its GEMMs (igemm_rt_i8)
};

struct Step {
    StepKind kind;
    uint32_t first, count;  // the records it stands for
    // kStepMatmulRt: the matrices of batch element 0, elements from one batch element to the next (0: shared), and the one
    // (bias, scale) pair
    DescRef a, b, out;
    int32_t batches;
    int64_t a_stride, b_stride, out_stride;
    int32_t bias, scale;
    // kStepPadded: rows of `from` bytes padded to `to`, and the record that reads them.  Its operands of space kSpacePlan are the
    // step's own: index 0 the padded rows, index 1 `constants` (on the device).
    int64_t rows;
    int32_t from, to;
    DescOp op;
    std::vector<uint8_t> constants;
};
constexpr uint32_t kSpacePlan = 16;

// The launches of a dispatch in order.  Every record belongs to exactly one step; a step that stands for several leaves
// the intermediates between them unwritten, so it is only formed where no other record reads them.
// `plain`: one step per record.
std::vector<Step> planSteps(const DescriptorView &view, bool plain);

}  // namespace thip
