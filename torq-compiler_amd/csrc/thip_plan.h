// From the records of a descriptor to the launches of a dispatch: runs of records that one kernel does as a whole.
// Host-only (no HIP calls).
#pragma once

#include <string.h>

#include <functional>
#include <vector>

#include "thip_dec_chain.h"
#include "thip_kernels.h"
#include "thip_validate.h"

namespace thip {

enum StepKind {
    kStepRecord,    // one record, by its own launcher
    kStepExpandDw,  // a pointwise convolution and the depthwise one behind it (ir_expand_dw_i8); three records: and the pointwise one behind that (ir_block_i8)
    kStepPadded,    // a GEMM-shaped record whose channels fill no 16-byte chunks: its input padded, then a dense kernel; or its weights padded only
    kStepMatmulRt,  // a batch of int8 matmuls with a run-time input2: its transposes and its GEMMs (igemm_rt_i8)
    kStepDecChain,  // grouped linears and small matmuls of a decoder's step, each behind the one before it (dec_chain)
};

// The kernel that a GEMM-shaped record of a dispatch runs by.
enum IgemmRoute {
    kIgemmOwnTile,  // the record's
    kIgemmDirect,   // igemm_direct_i8
    kIgemmPatch,    // conv_patch_i8
    kIgemmWide,     // the record's tile in k-tiles of 128 bytes
};

struct Step {
    StepKind kind;
    uint32_t first, count;  // the records it stands for
    IgemmRoute route;       // of the record, of `op` (kStepPadded), or of the third record where it is launched by itself (kStepExpandDw)
    int32_t images, stripRows;  // kStepExpandDw: of a workgroup of ir_expand_dw_i8 (irExpandDwTime)
    // kStepMatmulRt: the matrices of batch element 0, elements from one batch element to the next (0: shared), and the one
    // (bias, scale) pair
    DescRef a, b, out;
    int32_t batches;
    int64_t a_stride, b_stride, out_stride;
    int32_t bias, scale;
    // kStepPadded: rows of `from` bytes padded to `to`, and the record that reads them; or (asIs) a record that reads them as they are, its
    // weights alone padded (igemm_direct_i8), and that reads them padded only where its result lies on them (copies).  Its operands of space
    // kSpacePlan are the step's own: index 0 the padded rows, index 1 `constants` (on the device).
    int64_t rows;
    int32_t from, to;
    bool asIs, copies;
    DescOp op;
    std::vector<uint8_t> constants;
    // kStepRecord, grouped linears and small matmuls: DecBlocked, the intermediates that lie in blocks of columns
    int32_t blocked;
    // kStepDecChain: bytes of LDS for input rows and for partial sums; set when its table is laid out
    int32_t xRoom, redRoom;
};
constexpr uint32_t kSpacePlan = 16;

// The arguments of a GEMM-shaped record, its operands where `at` (const DescRef & -> uint8_t *) says.
template <typename At>
IgemmArgs igemmArgs(const DescriptorView &v, const DescOp &op, At &&at) {
    IgemmArgs a;
    memset(&a, 0, sizeof(a));
    a.A = (const int8_t *)at(op.in0);
    a.Bp = (const int8_t *)at(op.weights);
    a.bias = (const int32_t *)at(op.bias);
    a.scale = (const int32_t *)at(op.scale);
    a.ktab = (const uint32_t *)at(op.table);
    a.out = at(op.out);
    a.M = op.M; a.N = op.Nn; a.K = op.K; a.Kp = op.Kp; a.Np = op.Np;
    a.H = op.H; a.W = op.W; a.C = op.C; a.OH = op.OH; a.OW = op.OW;
    a.SH = op.SH; a.SW = op.SW; a.PT = op.PT; a.PL = op.PL;
    a.KH = op.KH; a.KW = op.KW;
    a.input_zp = op.input_zp;
    a.out_dtype = op.out_dtype;
    a.a_bytes = (int64_t)op.N * op.H * op.W * op.C;
    a.loader = op.loader;
    a.gran = op.gran;
    a.rq = Requant{op.shift, op.output_zp, op.output_min, op.output_max, op.pre_shift, op.t0_clamp};
    if (op.in1.space != kSpaceNone) {
        ResidualAddParams ap;
        memcpy(&ap, v.blob + v.header.data_offset + v.consts[op.table.index].offset + op.table.offset, sizeof(ap));
        a.skip = (const int8_t *)at(op.in1);
        a.add_skip_first = ap.other_first;
        a.add_w0 = ap.w0; a.add_w1 = ap.w1; a.add_bias = ap.bias; a.add_scale = ap.scale;
        a.arq = Requant{ap.shift, ap.output_zp, ap.output_min, ap.output_max, 0, 0};
    }
    return a;
}

// The same for igemm_direct_i8 on a record whose input's pixels are of `channels` bytes, no whole 16-byte chunks.  Its weights have zeros
// from there to the next whole chunk: those that a step has spread, and any of a window of one pixel.
template <typename At>
IgemmArgs raggedArgs(const DescriptorView &v, const DescOp &op, int32_t channels, At &&at) {
    IgemmArgs a = igemmArgs(v, op, at);
    const bool pointwise = op.KH == 1 && op.KW == 1 && op.SH == 1 && op.SW == 1 && op.PT == 0 && op.PL == 0 && op.OH == op.H && op.OW == op.W;
    a.loader = pointwise ? kLoaderDense : kLoaderWindow;
    a.row_bytes = channels;
    a.C = (channels + 15) / 16 * 16;
    a.K = op.KH * op.KW * a.C;
    a.a_bytes = (int64_t)op.N * op.H * op.W * channels;
    return a;
}

// The arguments of a step of three records that widen, convolve depthwise and narrow, its operands where `at` says.
template <typename At>
IrBlockArgs irBlockArgs(const DescriptorView &v, const Step &s, At &&at) {
    const DescOp &e = v.ops[s.first], &d = v.ops[s.first + 1], &g = v.ops[s.first + 2];
    const IgemmArgs last = igemmArgs(v, g, at);
    IrBlockArgs a;
    memset(&a, 0, sizeof(a));
    a.x = (const int8_t *)at(e.in0);
    a.wexp = (const int8_t *)at(e.weights);
    a.bias1 = (const int32_t *)at(e.bias);
    a.scale1 = (const int32_t *)at(e.scale);
    a.wdw = (const int32_t *)at(d.weights);
    a.bias2 = (const int32_t *)at(d.bias);
    a.scale2 = (const int32_t *)at(d.scale);
    a.wproj = last.Bp;
    a.bias3 = last.bias;
    a.scale3 = last.scale;
    a.skip = last.skip;
    a.out = (int8_t *)last.out;
    a.N = d.N; a.H = d.H; a.W = d.W; a.K = e.K; a.Kp = e.Kp; a.Np = e.Np; a.C = d.C;
    a.OH = d.OH; a.OW = d.OW; a.S = d.SW; a.PT = d.PT; a.PL = d.PL; a.O = g.Nn; a.Kp3 = g.Kp; a.zp = d.input_zp;
    a.rq1 = Requant{e.shift, e.output_zp, e.output_min, e.output_max, e.pre_shift, e.t0_clamp};
    a.rq2 = Requant{d.shift, d.output_zp, d.output_min, d.output_max, d.pre_shift, d.t0_clamp};
    a.rq3 = last.rq;
    a.arq = last.arq;
    a.addSkipFirst = last.add_skip_first;
    a.addW0 = last.add_w0; a.addW1 = last.add_w1; a.addBias = last.add_bias; a.addScale = last.add_scale;
    if (e.loader == kLoaderRuns) {
        a.CKH = e.KH; a.CS = e.SH; a.CPT = e.PT; a.CPL = e.PL; a.IH = e.H; a.IW = e.W; a.IC = e.C;
        a.runBytes = e.KW * e.C; a.czp = e.input_zp;
        a.xBytes = (int64_t)e.N * e.H * e.W * e.C;
    }
    return a;
}

// The records from `first` on that one launch of dec_chain takes, at most `most`, its operands where `at` says.
struct Chain {
    std::vector<ChainPhase> phases;
    uint64_t exchangeWords = 0;
    int32_t xRoom = 0, redRoom = 0;  // LDS of a workgroup for input rows and for partial sums
};
Chain layoutChain(const DescriptorView &v, uint32_t first, uint32_t most, int workgroups, const std::function<ChainRef(const DescRef &)> &at);

// The launches of a dispatch in order.  Every record belongs to exactly one step; a step that stands for several leaves
// the intermediates between them unwritten, so it is only formed where no other record reads them.
// tuning.plainRecords: one step per record, by the record's own kernel.  Routes are settled here, on all that their launchers ask: a dispatch's
// buffers start at 16-byte boundaries, so the offsets say how its operands are aligned.
std::vector<Step> planSteps(const DescriptorView &view, const Tuning &tuning);

// Whether the step's last record writes a binding whose bytes, where the dispatch has them (`bp`: a pointer per binding), are another
// binding's that the step reads.
bool writesWhatItReads(const DescriptorView &v, const Step &s, uint8_t *const *bp);

// Whether a dispatch of so many launches is worth a graph; `constantBytes`: what all of them read of weights.
bool replayPays(size_t launches, uint64_t constantBytes);

}  // namespace thip
