// Run side: device, executable and dispatch.
//
// The shape of this file follows the reference's HAL driver for this path:
//   thip_executable_create  <- iree_hal_torq_native_executable_create
//                              (runtime/driver/native_executable.cc:41-108): copy the
//                              program blob and the executable constants, build the
//                              executor object, initialise it (version / target gate,
//                              runtime/driver/TorqExecutable.cc:655-752).
//   thip_executable_run     <- iree_hal_torq_native_executable_run (:180-192) ->
//                              TorqExecutable::executeDispatch
//                              (runtime/driver/TorqExecutable.cc:1025-1125): lock,
//                              write inputs, walk the action list, read outputs.
// Instead of NSS programs on an NPU the action list is a list of kernel
// records, each launched on the executable's HIP stream.
#include <hip/hip_runtime.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <errno.h>
#include <sys/stat.h>

#include <algorithm>
#include <chrono>
#include <mutex>
#include <new>
#include <string>
#include <thread>
#include <vector>

#include "thip_chain_turn.h"
#include "thip_descriptor.h"
#include "thip_host_copy.h"
#include "thip_kernels.h"
#include "thip_plan.h"
#include "thip_status.h"
#include "thip_validate.h"

using namespace thip;

struct thip_device_t {
    int ordinal = 0;
    std::string arch;
    std::mutex logMutex;
    FILE *eventLog = nullptr;
    std::chrono::steady_clock::time_point t0 = std::chrono::steady_clock::now();
    int computeUnits = 0;
    uint8_t *staticScratch = nullptr;    // this GPU's copy of the library's scratch array (kStaticScratchBytes)
    // dump directories (empty: off): bindings of every blocking dispatch / every buffer a kernel record wrote
    std::string dumpIoDir, dumpBuffersDir;
    CopyCrew crew;                       // helps dispatches on host bindings to copy
};

struct thip_executable_t {
    thip_device_t *device = nullptr;
    std::vector<uint8_t> blob;           // private copy of the descriptor
    std::vector<uint32_t> constants;     // executable-level constants (copied)
    DescHeader header;
    const DescOp *ops = nullptr;
    const DescBinding *bindings = nullptr;
    const DescTemp *temps = nullptr;
    const DescConst *consts = nullptr;
    uint8_t *constData = nullptr;        // device copy of the constant segment
    std::vector<uint8_t *> tempPtrs;     // device intermediates
    std::vector<uint8_t *> staging;      // device staging of host bindings
    // Pinned memory between host bindings and their staging, allocated by the first dispatch that has some: for what is read two halves used in
    // turn (see stageIn), for what is written one place each; null: there is no memory for it and the runtime copies.
    struct {
        bool tried = false;
        uint8_t *in = nullptr, *out = nullptr;
        size_t half = 0;                 // bytes of one
        hipEvent_t done[2] = {nullptr, nullptr};  // behind the last copy out of it
    } pinned;
    hipStream_t stream = nullptr;
    hipEvent_t evStart = nullptr, evStop = nullptr, evDone = nullptr;
    // A wait for the GPU gives up after this long (the reference turns a wait that exceeds its timeout into
    // IREE_STATUS_INTERNAL, runtime/torq_hw/src/TorqHw.cpp:172-186).  <= 0: no limit.
    int64_t waitTimeoutMs = 120000;
    bool abandoned = false;              // a wait timed out: work may still be running, the executable is unusable
    std::mutex mutex;                    // one dispatch at a time
    // Multi-kernel programs on device bindings are replayed as HIP graphs, one per set of binding pointers (kGraphsKept
    // of them): the first dispatch on a set runs eagerly, the second is captured, later ones are one graph launch.
    struct Replay {
        std::vector<uint8_t *> ptrs;     // the binding pointers
        hipGraph_t graph = nullptr;
        hipGraphExec_t exec = nullptr;   // null: the set has been dispatched, eagerly
        uint64_t lastUse = 0;            // the invocation
    };
    std::vector<Replay> replays;
    // Graphs that made room for others, until the event behind their last replay says that they are done.
    struct Retired {
        hipGraph_t graph;
        hipGraphExec_t exec;
        hipEvent_t done;
    };
    std::vector<Retired> retired;
    bool graphsDisabled = false;
    uint64_t invocation = 0;             // dispatches so far (the event log's invocation_id)
    Tuning tuning;                       // the environment's switches as they were when the executable was created
    std::vector<std::string> kernelNames;  // per record: the kernel its launcher resolved at creation
    // thip_executable_enqueue_noalloc: where each record's scratch (a K-split workspace) sits in the static array,
    // and the program's total
    std::vector<Step> steps;             // the launches of a dispatch, in order
    std::vector<std::string> launchNames;  // their kernels
    std::vector<uint8_t *> stepBuffers;  // two per step: operands of space kSpacePlan; or the table and the counters of a chain (null: none)
    bool chained = false;                // a step's workgroups wait for one another (kStepDecChain)
    ChainMember chain;                   // then: among the device's executables that have such a step
    std::vector<uint64_t> scratchOffset;
    uint64_t scratchBytes = 0;
};

static thip_status_t hipFail(hipError_t e, const char *what) {
    const thip_status_t code = e == hipErrorOutOfMemory ? THIP_RESOURCE_EXHAUSTED : THIP_INTERNAL;
    return fail(code, "%s: %s", what, hipGetErrorString(e));
}

#define THIP_HIP(call, what)                          \
    do {                                              \
        hipError_t e_ = (call);                       \
        if (e_ != hipSuccess) return hipFail(e_, what); \
    } while (0)

// The kernel family of a record (error messages before the launcher has named the instantiation).
static const char *opKernelName(const DescOp &op) {
    switch (op.kind) {
    case kKindTranspose: return "transpose_i8";
    case kKindIgemm: return igemmTile(op.variant).name;
    case kKindFcSkinny: return "fc_skinny";
    case kKindDepthwise: return op.variant == kDepthwiseDot4Rows ? "depthwise3x3_dot4_i8" : "depthwise_i8";
    case kKindMaxPool: return "maxpool_i8";
    case kKindAvgPool: return "avgpool_i8";
    case kKindAdd: return "add_i8";
    case kKindFcBf16: return "fc_bf16";
    case kKindAddBf16: return "add_bf16";
    case kKindIm2colBf16: return "im2col_bf16";
    case kKindDepthwiseBf16: return "depthwise_bf16";
    case kKindAvgPoolBf16: return "avgpool_bf16";
    case kKindExpandWeights: return "expand_weights_bf16";
    case kKindEltwise: return "eltwise_int";
    case kKindDecLinear: return "dec_linear";
    case kKindDecMatmul: return "dec_matmul";
    default: return "unknown";
    }
}

// One row of the event log, in the reference's runtime CSV columns (doc/user-manual/profiling.md:53-63, written by
// runtime/torq_hw/src/TorqEventLog.cpp:48,97-101): dispatch_name, invocation_id, action_id, timestamp_us, event
// (an EventType name + _BEGIN / _END), plus one column of this backend's own: the kernel of a launch row.
static void logEvent(const thip_executable_t *e, uint64_t invocation, int32_t action, const char *event, const char *phase, const char *kernel) {
    thip_device_t *d = e->device;
    if (!d->eventLog) return;
    std::lock_guard<std::mutex> lock(d->logMutex);
    const auto us = std::chrono::duration_cast<std::chrono::microseconds>(std::chrono::steady_clock::now() - d->t0).count();
    fprintf(d->eventLog, "%s,%llu,%d,%lld,%s_%s,%s\n", e->header.name, (unsigned long long)invocation, action, (long long)us, event, phase, kernel);
}

static DescriptorView viewOf(const thip_executable_t *e) { return DescriptorView{e->blob.data(), e->header, e->ops, e->bindings, e->temps, e->consts}; }

// Resolves an operand reference against the buffers of this dispatch.
static uint8_t *resolve(const thip_executable_t *e, const DescRef &r, uint8_t *const *bindingPtrs) {
    switch (r.space) {
    case kSpaceBinding: return bindingPtrs[r.index] + r.offset;
    case kSpaceTemp: return e->tempPtrs[r.index] + r.offset;
    case kSpaceConst: return e->constData + e->consts[r.index].offset + r.offset;
    default: return nullptr;
    }
}

// Launches `op`, which is record i or stands in for it, or (ctx.name set) only asks its launcher which kernel it takes for these
// operands.  `scratch` (or null): the static scratch array, which then stands in for the record's workspace intermediate.
// `step` (or null): the buffers of space kSpacePlan.  `route`: the kernel of a GEMM-shaped record.
// `blocked`: DecBlocked, the intermediates of a decoder's record that lie in blocks of columns.  `planned`: a step's launch, not the record's own kernel.
static thip_status_t launchOp(thip_executable_t *e, uint32_t i, const DescOp &op, uint8_t *const *bp, const LaunchCtx &ctx, uint8_t *scratch = nullptr,
                              uint8_t *const *step = nullptr, IgemmRoute route = kIgemmOwnTile, int32_t blocked = 0, bool planned = false) {
    auto resolve = [step](const thip_executable_t *exe, const DescRef &r, uint8_t *const *bindings) {
        return r.space == kSpacePlan ? step[r.index] + r.offset : ::resolve(exe, r, bindings);
    };
    const Requant rq{op.shift, op.output_zp, op.output_min, op.output_max, op.pre_shift, op.t0_clamp};
    hipError_t err = hipSuccess;
    switch (op.kind) {
    case kKindTranspose: {
        TransposeArgs a{(const int8_t *)resolve(e, op.in0, bp), (int8_t *)resolve(e, op.out, bp), op.TB, op.TR, op.TS, op.gran == 2 ? 2 : 1, op.TP ? op.TP : op.TR};
        err = launchTranspose(a, ctx);
        break;
    }
    case kKindIgemm: {
        auto at = [&](const DescRef &r) { return resolve(e, r, bp); };
        const bool asIs = route == kIgemmDirect && e->ops[i].loader == kLoaderGather && op.in0.space != kSpacePlan;
        const IgemmArgs a = asIs ? raggedArgs(viewOf(e), op, e->ops[i].C, at) : igemmArgs(viewOf(e), op, at);
        LaunchCtx own = ctx;
        own.any_rows = planned && !e->tuning.plainRecords;
        if (route == kIgemmDirect) err = launchIgemmDirect(a, ctx);
        else if (route == kIgemmPatch) err = launchConvPatch(a, ctx);
        else err = launchIgemm(a, op.variant, own, route == kIgemmWide);
        break;
    }
    case kKindFcSkinny: {
        FcSkinnyArgs a{(const int8_t *)resolve(e, op.in0, bp), (const int8_t *)resolve(e, op.weights, bp),
                       (const int32_t *)resolve(e, op.bias, bp), (const int32_t *)resolve(e, op.scale, bp),
                       resolve(e, op.out, bp), op.M, op.Nn, op.K, op.out_dtype, rq};
        err = launchFcSkinny(a, ctx);
        break;
    }
    case kKindDepthwise: {
        DepthwiseArgs a{(const int8_t *)resolve(e, op.in0, bp), (const int8_t *)resolve(e, op.weights, bp),
                        (const int32_t *)resolve(e, op.bias, bp), (const int32_t *)resolve(e, op.scale, bp),
                        (int8_t *)resolve(e, op.out, bp), op.N, op.H, op.W, op.C, op.OH, op.OW, op.KH, op.KW,
                        op.SH, op.SW, op.PT, op.PL, op.input_zp, op.variant, rq};
        err = launchDepthwise(a, ctx);
        break;
    }
    case kKindMaxPool: {
        MaxPoolArgs a{(const int8_t *)resolve(e, op.in0, bp), (int8_t *)resolve(e, op.out, bp), op.N, op.H, op.W, op.C,
                      op.OH, op.OW, op.KH, op.KW, op.SH, op.SW, op.PT, op.PL, op.input_zp, op.output_min, op.output_max};
        err = launchMaxPool(a, ctx);
        break;
    }
    case kKindAvgPool: {
        AvgPoolArgs a{(const int8_t *)resolve(e, op.in0, bp), (int8_t *)resolve(e, op.out, bp), op.N, op.H * op.W, op.C,
                      op.w0, op.bias0, op.scale0, rq};
        err = launchAvgPool(a, ctx);
        break;
    }
    case kKindAdd: {
        AddArgs a{(const int8_t *)resolve(e, op.in0, bp), (const int8_t *)resolve(e, op.in1, bp),
                  (int8_t *)resolve(e, op.out, bp), (int64_t)op.C, op.w0, op.w1, op.bias0, op.scale0, rq};
        err = launchAdd(a, ctx);
        break;
    }
    case kKindIm2colBf16: {
        Im2colBf16Args a{(const uint16_t *)resolve(e, op.in0, bp), (uint16_t *)resolve(e, op.out, bp), op.N, op.H, op.W, op.C,
                         op.OH, op.OW, op.KH, op.KW, op.SH, op.SW, op.PT, op.PL, op.Kp};
        err = launchIm2colBf16(a, ctx);
        break;
    }
    case kKindDepthwiseBf16: {
        float lo, hi;
        memcpy(&lo, &op.output_min, 4);
        memcpy(&hi, &op.output_max, 4);
        DepthwiseBf16Args a{(const uint16_t *)resolve(e, op.in0, bp), (const uint16_t *)resolve(e, op.weights, bp),
                            (const float *)resolve(e, op.bias, bp), (uint16_t *)resolve(e, op.out, bp), op.N, op.H, op.W, op.C,
                            op.OH, op.OW, op.KH, op.KW, op.SH, op.SW, op.PT, op.PL, lo, hi};
        err = launchDepthwiseBf16(a, ctx);
        break;
    }
    case kKindAddBf16: {
        auto asFloat = [](int32_t bits) {
            float f;
            memcpy(&f, &bits, 4);
            return f;
        };
        AddBf16Args a{(const uint16_t *)resolve(e, op.in0, bp), (const uint16_t *)resolve(e, op.in1, bp),
                      (uint16_t *)resolve(e, op.out, bp), (int64_t)op.C, asFloat(op.w0 << 16), asFloat(op.w1 << 16),
                      asFloat(op.bias0), asFloat(op.output_min), asFloat(op.output_max)};
        err = launchAddBf16(a, ctx);
        break;
    }
    case kKindFcBf16: {
        float lo, hi;
        memcpy(&lo, &op.output_min, 4);
        memcpy(&hi, &op.output_max, 4);
        FcBf16Args a{(const uint16_t *)resolve(e, op.in0, bp), (const uint16_t *)resolve(e, op.weights, bp),
                     (const float *)resolve(e, op.bias, bp), (uint16_t *)resolve(e, op.out, bp), op.M, op.K, op.Nn, lo, hi,
                     op.w0 > 1 ? op.w0 : 1, op.w0 > 1 ? (void *)(scratch ? scratch + e->scratchOffset[i] : resolve(e, op.in1, bp)) : nullptr, (int32_t)op.loader,
                     nullptr, nullptr, 0, 0, 0.0f, 0.0f};
        if (op.loader == 2) {
            a.qscale = (const uint16_t *)resolve(e, op.scale, bp);
            a.qbias = (const float *)resolve(e, op.table, bp);
            a.qblock = (int32_t)op.gran;
            a.qcols = op.Np;
            memcpy(&a.qlo, &op.bias0, 4);
            memcpy(&a.qhi, &op.scale0, 4);
        }
        err = launchFcBf16(a, ctx);
        break;
    }
    case kKindAvgPoolBf16: {
        AvgPoolBf16Args a{(const uint16_t *)resolve(e, op.in0, bp), (uint16_t *)resolve(e, op.out, bp), op.N, op.H * op.W, op.C,
                          0.0f, 0.0f, 0.0f, 0.0f};
        const uint32_t wbits = (uint32_t)op.w0 << 16;
        memcpy(&a.weight, &wbits, 4);
        memcpy(&a.bias, &op.bias0, 4);
        memcpy(&a.lo, &op.output_min, 4);
        memcpy(&a.hi, &op.output_max, 4);
        err = launchAvgPoolBf16(a, ctx);
        break;
    }
    case kKindEltwise: {
        EltwiseArgs a{resolve(e, op.in0, bp), eltwiseTwoInputs((int32_t)op.variant) ? resolve(e, op.in1, bp) : nullptr, resolve(e, op.out, bp), (int64_t)op.C,
                      (int32_t)op.variant, (int32_t)op.gran, op.out_dtype == THIP_DTYPE_I8 ? 1 : op.out_dtype == THIP_DTYPE_I16 ? 2 : 4, op.w1,
                      op.w0, op.bias0, op.scale0, op.output_min, op.output_max, rq};
        err = launchEltwise(a, ctx);
        break;
    }
    case kKindExpandWeights: {
        ExpandWeightsArgs a{(const int8_t *)resolve(e, op.in0, bp), (const uint16_t *)resolve(e, op.scale, bp),
                            (const float *)resolve(e, op.bias, bp), (uint16_t *)resolve(e, op.out, bp), op.K, op.Nn,
                            (int32_t)op.gran, op.Np, 0.0f, 0.0f};
        memcpy(&a.lo, &op.output_min, 4);
        memcpy(&a.hi, &op.output_max, 4);
        err = launchExpandWeights(a, ctx);
        break;
    }
    case kKindDecLinear: {
        DecLinearExt x;
        memcpy(&x, e->blob.data() + e->header.data_offset + e->consts[op.table.index].offset + op.table.offset, sizeof(x));  // the host copy
        DecLinearArgs a;
        memset(&a, 0, sizeof(a));
        a.x = (const uint16_t *)resolve(e, op.in0, bp);
        a.M = op.M; a.K = op.K; a.qblock = (int32_t)op.gran;
        a.nseg = op.w0;
        a.pair = (op.w1 & kDecPair) ? 1 : 0;
        a.has_qbias = x.has_qbias;
        for (int m = 0; m < op.w0 && m < kDecMaxSegments; m++) {
            a.w[m] = (const int8_t *)resolve(e, x.weights[m], bp);
            a.bias[m] = (const float *)resolve(e, x.bias[m], bp);
            a.out[m] = (uint16_t *)resolve(e, x.out[m], bp);
            a.N[m] = x.N[m];
        }
        memcpy(&a.lo, &op.output_min, 4);
        memcpy(&a.hi, &op.output_max, 4);
        memcpy(&a.qlo, &op.bias0, 4);
        memcpy(&a.qhi, &op.scale0, 4);
        a.add_mode = (op.w1 & kDecAddResidual) ? 1 : (op.w1 & kDecAddPair) ? 2 : 0;
        a.res_first = (op.w1 & kDecResFirst) ? 1 : 0;
        if (a.add_mode) {
            a.res = (const uint16_t *)resolve(e, x.res, bp);
            a.add_out = (uint16_t *)resolve(e, x.add_out, bp);
            const uint32_t w0 = (uint32_t)x.aw0 << 16, w1 = (uint32_t)x.aw1 << 16;
            memcpy(&a.aw0, &w0, 4);
            memcpy(&a.aw1, &w1, 4);
            memcpy(&a.abias, &x.abias, 4);
            memcpy(&a.alo, &x.alo, 4);
            memcpy(&a.ahi, &x.ahi, 4);
        }
        a.blocked = blocked;
        err = launchDecLinear(a, ctx);
        break;
    }
    case kKindDecMatmul: {
        DecMatmulArgs a{(const uint16_t *)resolve(e, op.in0, bp), (const uint16_t *)resolve(e, op.weights, bp), (uint16_t *)resolve(e, op.out, bp),
                        op.TB, op.M, op.K, op.Nn, op.w0 ? 0 : (int64_t)op.M * op.K, op.w1 ? 0 : (int64_t)op.Nn * op.K, (int64_t)op.M * op.Nn, 0.0f, 0.0f, 0.0f, blocked};
        memcpy(&a.bias, &op.bias0, 4);
        memcpy(&a.lo, &op.output_min, 4);
        memcpy(&a.hi, &op.output_max, 4);
        err = launchDecMatmul(a, ctx);
        break;
    }
    default: return fail(THIP_INTERNAL, "op %u has unknown kind %u", i, op.kind);
    }
    if (err != hipSuccess) {
        return fail(THIP_INTERNAL, "op %u (%s): launch failed: %s", i, ctx.name ? opKernelName(op) : e->kernelNames[i].c_str(), hipGetErrorString(err));
    }
    return THIP_OK;
}

// Validates the dispatch state against the binding table.  Mirrors the checks of
// iree_hal_torq_command_buffer_dispatch (runtime/driver/torq_command_buffer.c:453-494).
static thip_status_t checkState(const thip_executable_t *e, const thip_dispatch_state_t *st, bool deviceOnly) {
    if (!st) return fail(THIP_INVALID_ARGUMENT, "dispatch state is NULL");
    if (st->constant_count > 0 && !st->constants) return fail(THIP_FAILED_PRECONDITION, "constants pointer is NULL");
    if (st->binding_count < e->header.binding_count) {
        return fail(THIP_INVALID_ARGUMENT, "dispatch carries %u bindings, the executable uses %u", st->binding_count, e->header.binding_count);
    }
    if (e->header.binding_count > 0 && (!st->binding_ptrs || !st->binding_lengths)) {
        return fail(THIP_FAILED_PRECONDITION, "binding tables are NULL");
    }
    for (uint32_t i = 0; i < e->header.binding_count; i++) {
        if (e->bindings[i].flags == 0) continue;  // declared but unused
        if (!st->binding_ptrs[i]) {
            return fail(THIP_FAILED_PRECONDITION, "required binding %u is NULL; all bindings must have a valid pointer", i);
        }
        if (st->binding_lengths[i] < e->bindings[i].size) {
            return fail(THIP_OUT_OF_RANGE, "binding %u is %zu bytes, the executable touches %llu", i, st->binding_lengths[i],
                        (unsigned long long)e->bindings[i].size);
        }
        const bool isDevice = st->binding_flags && (st->binding_flags[i] & THIP_BINDING_DEVICE);
        if (deviceOnly && !isDevice) return fail(THIP_FAILED_PRECONDITION, "binding %u is a host pointer; this entry point takes device bindings only", i);
        if (isDevice && ((uintptr_t)st->binding_ptrs[i] & 15) != 0) {
            return fail(THIP_FAILED_PRECONDITION, "device binding %u is not 16-byte aligned", i);
        }
    }
    return THIP_OK;
}

// Waits for everything enqueued on the executable's stream, at most waitTimeoutMs.  On expiry the executable is
// marked abandoned (kernels may still be running on its buffers: later calls are refused and destruction does not
// free them) and THIP_INTERNAL comes back; the process goes on and can report the failure.
static thip_status_t waitBounded(thip_executable_t *e, hipEvent_t event, const char *what) {
    if (e->waitTimeoutMs <= 0) {
        THIP_HIP(hipEventSynchronize(event), what);
        return THIP_OK;
    }
    const auto start = std::chrono::steady_clock::now();
    const auto deadline = start + std::chrono::milliseconds(e->waitTimeoutMs);
    for (;;) {
        const hipError_t q = hipEventQuery(event);
        if (q == hipSuccess) return THIP_OK;
        if (q != hipErrorNotReady) return hipFail(q, what);
        (void)hipGetLastError();  // not-ready is no error
        const auto now = std::chrono::steady_clock::now();
        if (now >= deadline) {
            e->abandoned = true;
            e->chain.abandoned = true;
            return fail(THIP_INTERNAL, "%s: the GPU did not finish within %lld ms; the executable is abandoned", what, (long long)e->waitTimeoutMs);
        }
        // poll hard at first (dispatches are microseconds to a few milliseconds long, and a sleep of any length costs
        // some 100 us before the thread runs again), then back off
        if (now - start > std::chrono::microseconds(3000)) std::this_thread::sleep_for(std::chrono::microseconds(50));
    }
}
static thip_status_t waitBounded(thip_executable_t *e, const char *what) {
    e->chain.waiting();
    if (e->waitTimeoutMs <= 0) {
        THIP_HIP(hipStreamSynchronize(e->stream), what);
    } else {
        THIP_HIP(hipEventRecord(e->evDone, e->stream), "hipEventRecord");
        if (thip_status_t s = waitBounded(e, e->evDone, what)) return s;
    }
    e->chain.finished();
    return THIP_OK;
}

static bool makeDirs(const std::string &path) {
    for (size_t i = 1; i <= path.size(); i++) {
        if (i == path.size() || path[i] == '/') {
            const std::string part = path.substr(0, i);
            if (mkdir(part.c_str(), 0777) != 0 && errno != EEXIST) return false;
        }
    }
    return true;
}

// Raw bytes of a binding, named as the reference names them (runtime/driver/TorqDump.cc:329-339):
// <dir>/<executable>/npu.{in,out}.host_binding.<i>.torq_binding.<i>.bin
static void dumpBinding(const thip_executable_t *e, uint32_t binding, const void *host, size_t size, bool isInput) {
    const thip_device_t *d = e->device;
    if (d->dumpIoDir.empty()) return;
    const std::string dir = d->dumpIoDir + "/" + e->header.name;
    if (!makeDirs(dir)) return;
    const std::string n = std::to_string(binding);
    const std::string path = dir + "/npu" + (isInput ? ".in" : ".out") + ".host_binding." + n + ".torq_binding." + n + ".bin";
    if (FILE *f = fopen(path.c_str(), "wb")) {
        fwrite(host, 1, size, f);
        fclose(f);
    }
}

// What record i wrote, as a NumPy array file <dir>/<executable>/action<i>/buffer<id>.npy (the reference writes one
// .npy per live buffer per action, runtime/driver/TorqDump.cc:341-428), id = "binding<k>" or "temp<k>", plus one
// line of <dir>/<executable>/buffers.csv in the reference's columns.  The record's kernels must have finished.
static thip_status_t dumpOpOutput(thip_executable_t *e, uint32_t i, uint8_t *const *bp) {
    const thip_device_t *d = e->device;
    const DescOp &op = e->ops[i];
    std::vector<int64_t> shape;
    const char *descr = "|i1", *typeName = "i8";
    size_t elem = 1;
    auto outType = [&]() {
        if (op.out_dtype == THIP_DTYPE_I32) { descr = "<i4"; typeName = "i32"; elem = 4; }
        else if (op.out_dtype == THIP_DTYPE_I16) { descr = "<i2"; typeName = "i16"; elem = 2; }
    };
    auto bf16 = [&]() { descr = "<u2"; typeName = "bf16"; elem = 2; };  // bf16 bit patterns, as uint16
    switch (op.kind) {
    case kKindTranspose: shape = {op.TB, op.TS, op.TP ? op.TP : op.TR}; if (op.gran == 2) bf16(); break;
    case kKindIgemm: case kKindFcSkinny: shape = {op.M, op.Nn}; outType(); break;
    case kKindDepthwise: case kKindMaxPool: shape = {op.N, op.OH, op.OW, op.C}; break;
    case kKindAvgPool: shape = {op.N, op.C}; break;
    case kKindAdd: shape = {op.C}; break;
    case kKindEltwise: shape = {op.C}; outType(); break;
    case kKindFcBf16: case kKindDecLinear: shape = {op.M, op.Nn}; bf16(); break;
    case kKindDecMatmul: shape = {op.TB, op.M, op.Nn}; bf16(); break;
    case kKindAddBf16: shape = {op.C}; bf16(); break;
    case kKindIm2colBf16: shape = {op.N, op.OH, op.OW, op.Kp}; bf16(); break;
    case kKindDepthwiseBf16: shape = {op.N, op.OH, op.OW, op.C}; bf16(); break;
    case kKindAvgPoolBf16: shape = {op.N, op.C}; bf16(); break;
    case kKindExpandWeights: shape = {op.K, op.Nn}; bf16(); break;
    default: return THIP_OK;
    }
    size_t count = 1;
    for (int64_t v : shape) count *= (size_t)v;
    if (count == 0 || op.out.space == kSpaceNone) return THIP_OK;  // e.g. a convolution whose result only feeds its fused add
    std::vector<uint8_t> host(count * elem);
    THIP_HIP(hipMemcpy(host.data(), resolve(e, op.out, bp), host.size(), hipMemcpyDeviceToHost), "reading a buffer back for the dump");
    const std::string base = d->dumpBuffersDir + "/" + e->header.name, dir = base + "/action" + std::to_string(i);
    if (!makeDirs(dir)) return fail(THIP_INVALID_ARGUMENT, "cannot create dump directory %s", dir.c_str());
    const std::string id = (op.out.space == kSpaceBinding ? "binding" : "temp") + std::to_string(op.out.index);
    std::string dims, dimsX;
    for (size_t k = 0; k < shape.size(); k++) {
        dims += std::to_string(shape[k]) + ",";
        dimsX += std::to_string(shape[k]) + "x";
    }
    std::string header = std::string("{'descr': '") + descr + "', 'fortran_order': False, 'shape': (" + dims + "), }";
    while ((10 + header.size() + 1) % 64 != 0) header += ' ';
    header += '\n';
    FILE *f = fopen((dir + "/buffer" + id + ".npy").c_str(), "wb");
    if (!f) return fail(THIP_INVALID_ARGUMENT, "cannot write into dump directory %s", dir.c_str());
    const uint8_t magic[10] = {0x93, 'N', 'U', 'M', 'P', 'Y', 1, 0, (uint8_t)(header.size() & 0xff), (uint8_t)(header.size() >> 8)};
    fwrite(magic, 1, sizeof(magic), f);
    fwrite(header.data(), 1, header.size(), f);
    fwrite(host.data(), 1, host.size(), f);
    fclose(f);
    // index of the buffers, one line per record output; started afresh by the first record of every dispatch
    if (FILE *csv = fopen((base + "/buffers.csv").c_str(), i == 0 ? "w" : "a")) {
        if (i == 0) {
            fprintf(csv, "id;type;shape;strides;address;size;allocation_action;last_use_action;deallocation_action;"
                         "allocation_location;last_use_location;deallocation_location\n");
        }
        fprintf(csv, "%s;%s;%s%s;;%llu;%zu;%u;%u;%u;%s;;\n", id.c_str(), op.out.space == kSpaceBinding ? "BINDING" : "INTERMEDIATE", dimsX.c_str(),
                typeName, (unsigned long long)op.out.offset, host.size(), i, i, e->header.op_count - 1, e->kernelNames[i].c_str());
        fclose(csv);
    }
    return THIP_OK;
}

// Whether a binding that the program writes shares bytes with another one.  A chain fetches its inputs ahead, so it does not take these.
static bool chainAliased(const thip_executable_t *e, uint8_t *const *bp) {
    for (uint32_t i = 0; i < e->header.binding_count; i++) {
        if (!(e->bindings[i].flags & kBindingWritten)) continue;
        for (uint32_t j = 0; j < e->header.binding_count; j++) {
            if (j != i && e->bindings[j].flags != 0 && bp[i] < bp[j] + e->bindings[j].size && bp[j] < bp[i] + e->bindings[i].size) return true;
        }
    }
    return false;
}

// Launches one step: a record by its own launcher, a run of records by the kernel that does them as a whole.  `apart`: a chain record by record.
// A run whose result lies where it still reads (a block in place) is launched in parts that read nothing that another workgroup of theirs writes.
static thip_status_t launchStep(thip_executable_t *e, const Step &s, uint8_t *const *bp, const LaunchCtx &ctx, uint8_t *scratch = nullptr, bool apart = false) {
    hipError_t err = hipSuccess;
    // asked for its kernel, a step asks for those that it launches on shared memory too
    char others[96];
    LaunchCtx behind = ctx;
    behind.name = others;
    behind.name_capacity = sizeof(others);
    auto recordByRecord = [&]() -> thip_status_t {
        for (uint32_t i = s.first; i < s.first + s.count; i++) {
            if (thip_status_t st = launchOp(e, i, e->ops[i], bp, ctx, scratch)) return st;
        }
        return THIP_OK;
    };
    switch (s.kind) {
    case kStepExpandDw: {
        const bool shared = !ctx.name && writesWhatItReads(viewOf(e), s, bp), block = s.count == 3 && !shared;
        if (s.count == 2 && shared) return recordByRecord();
        if (block) err = launchIrBlock(irBlockArgs(viewOf(e), s, [&](const DescRef &r) { return r.space == kSpaceNone ? nullptr : (uint8_t *)resolve(e, r, bp); }), ctx);
        if (block && (err != hipSuccess || !ctx.name)) break;
        const LaunchCtx &parts = block ? behind : ctx;
        const DescOp &x = e->ops[s.first], &d = e->ops[s.first + 1];
        IrExpandDwArgs a;
        memset(&a, 0, sizeof(a));
        a.x = (const int8_t *)resolve(e, x.in0, bp);
        a.wexp = (const int8_t *)resolve(e, x.weights, bp);
        a.bias1 = (const int32_t *)resolve(e, x.bias, bp);
        a.scale1 = (const int32_t *)resolve(e, x.scale, bp);
        a.wdw = (const int32_t *)resolve(e, d.weights, bp);
        a.bias2 = (const int32_t *)resolve(e, d.bias, bp);
        a.scale2 = (const int32_t *)resolve(e, d.scale, bp);
        a.out = (int8_t *)resolve(e, d.out, bp);
        a.N = d.N; a.H = d.H; a.W = d.W; a.K = x.K; a.Kp = x.Kp; a.Np = x.Np; a.C = d.C;
        a.OH = d.OH; a.OW = d.OW; a.S = d.SW; a.PT = d.PT; a.PL = d.PL; a.zp = d.input_zp;
        a.rq1 = Requant{x.shift, x.output_zp, x.output_min, x.output_max, x.pre_shift, x.t0_clamp};
        a.rq2 = Requant{d.shift, d.output_zp, d.output_min, d.output_max, d.pre_shift, d.t0_clamp};
        if (x.loader == kLoaderRuns) {
            a.CKH = x.KH; a.CS = x.SH; a.CPT = x.PT; a.CPL = x.PL; a.IH = x.H; a.IW = x.W; a.IC = x.C;
            a.runBytes = x.KW * x.C; a.czp = x.input_zp;
            a.xBytes = (int64_t)x.N * x.H * x.W * x.C;
        }
        a.images = s.images; a.stripRows = s.stripRows;
        err = launchIrExpandDw(a, parts);
        if (err == hipSuccess && s.count == 3) return launchOp(e, s.first + 2, e->ops[s.first + 2], bp, parts, scratch, nullptr, s.route, 0, true);
        break;
    }
    case kStepMatmulRt: {
        if (!ctx.name && writesWhatItReads(viewOf(e), s, bp)) return recordByRecord();
        const DescOp &g = e->ops[s.first + s.count - 1];
        MatmulRtArgs a;
        memset(&a, 0, sizeof(a));
        a.A = (const int8_t *)resolve(e, s.a, bp);
        a.B = (const int8_t *)resolve(e, s.b, bp);
        a.out = resolve(e, s.out, bp);
        a.M = g.M; a.N = g.Nn; a.K = g.K; a.batches = s.batches;
        a.a_stride = s.a_stride; a.b_stride = s.b_stride; a.out_stride = s.out_stride;
        a.a_bytes = (int64_t)(s.a_stride ? s.batches : 1) * g.M * g.K;
        a.b_bytes = (int64_t)(s.b_stride ? s.batches : 1) * g.K * g.Nn;
        a.bias = s.bias; a.scale = s.scale; a.out_dtype = g.out_dtype;
        a.rq = Requant{g.shift, g.output_zp, g.output_min, g.output_max, g.pre_shift, g.t0_clamp};
        err = launchMatmulRt(a, ctx);
        break;
    }
    case kStepPadded: {
        uint8_t *const *buffers = &e->stepBuffers[2 * (size_t)(&s - e->steps.data())];
        const bool shared = s.asIs && !ctx.name && writesWhatItReads(viewOf(e), s, bp);
        if (shared && !buffers[0]) return recordByRecord();  // no memory for the copy
        if (s.asIs && !shared) {
            const thip_status_t st = launchOp(e, s.first, s.op, bp, ctx, scratch, buffers, s.route, 0, true);
            if (st != THIP_OK || !ctx.name || !buffers[0]) return st;
        }
        const LaunchCtx &copied = s.asIs && ctx.name ? behind : ctx;
        err = launchPadRows((const int8_t *)resolve(e, e->ops[s.first].in0, bp), (int8_t *)buffers[0], s.rows, s.from, s.to, copied);
        if (err != hipSuccess) break;
        DescOp op = s.op;
        op.in0 = DescRef{kSpacePlan, 0, 0};
        return launchOp(e, s.first, op, bp, copied, scratch, buffers, s.route, 0, true);
    }
    case kStepDecChain: {
        if (!ctx.name && apart) return recordByRecord();
        uint8_t *const *buffers = &e->stepBuffers[2 * (size_t)(&s - e->steps.data())];
        DecChainArgs a;
        memset(&a, 0, sizeof(a));
        a.phases = (const ChainPhase *)buffers[0];
        a.sync = (uint32_t *)buffers[1];
        a.count = (int32_t)s.count;
        a.xRoom = s.xRoom;
        a.redRoom = s.redRoom;
        a.waitTicks = (uint64_t)e->tuning.decChainWait;
        for (uint32_t i = 0; i < e->header.binding_count && i < 64; i++) a.bindings[i] = bp[i];
        err = launchDecChain(a, e->device->computeUnits, ctx);
        break;
    }
    default: {
        const bool shared = s.route == kIgemmDirect && !ctx.name && writesWhatItReads(viewOf(e), s, bp);
        return launchOp(e, s.first, e->ops[s.first], bp, ctx, scratch, nullptr, shared ? kIgemmOwnTile : s.route, s.blocked, !shared);
    }
    }
    if (err != hipSuccess) return fail(THIP_INTERNAL, "ops %u .. %u: launch failed: %s", s.first, s.first + s.count - 1, hipGetErrorString(err));
    return THIP_OK;
}

// A log or a dump is told of every record.
static bool tellsRecords(const thip_executable_t *e) { return e->device->eventLog || !e->device->dumpBuffersDir.empty(); }

// Enqueues every kernel of the program.  `bp` holds one device pointer per binding.
static thip_status_t enqueueOps(thip_executable_t *e, uint8_t *const *bp, bool apart = false) {
    if (!tellsRecords(e)) {
        const LaunchCtx ctx{e->stream, &e->tuning, nullptr, 0, e->device->ordinal};
        for (const Step &s : e->steps) {
            if (thip_status_t st = launchStep(e, s, bp, ctx, nullptr, apart)) return st;
        }
        return THIP_OK;
    }
    for (uint32_t i = 0; i < e->header.op_count; i++) {
        // a kernel launch is what starting an NSS task is on the reference's hardware
        logEvent(e, e->invocation, (int32_t)i, "NSS_START", "BEGIN", e->kernelNames[i].c_str());
        if (thip_status_t s = launchOp(e, i, e->ops[i], bp, LaunchCtx{e->stream, &e->tuning, nullptr, 0, e->device->ordinal})) return s;
        logEvent(e, e->invocation, (int32_t)i, "NSS_START", "END", e->kernelNames[i].c_str());
        if (!e->device->dumpBuffersDir.empty()) {
            // buffer dumps: each record runs to its end and what it wrote is read back before the next one starts
            if (thip_status_t s = waitBounded(e, "waiting for a record before its dump")) return s;
            if (thip_status_t s = dumpOpOutput(e, i, bp)) return s;
        }
    }
    return THIP_OK;
}

// Sets of binding pointers with a graph of their own.  A caller that prepares its next inputs while a dispatch runs rotates over
// two or three; with one graph only, every dispatch of such a caller was launched kernel by kernel (MobileNetV2, one image, three
// sets: 151 us, the host's launches; 142 replayed).
constexpr size_t kGraphsKept = 8;
// A set that has not come back for this many dispatches makes room for a new one; one that has is not replaced, so a caller
// that rotates over more sets than are kept does not capture a graph per dispatch.
constexpr uint64_t kReplayMaxAge = 64;

static void dropReplay(thip_executable_t::Replay *r) {
    if (r->exec) (void)hipGraphExecDestroy(r->exec);
    if (r->graph) (void)hipGraphDestroy(r->graph);
    r->exec = nullptr;
    r->graph = nullptr;
}

// Frees the graphs put aside whose last replay is done; `all`: the caller knows that the stream is idle.
static void freeRetired(thip_executable_t *e, bool all) {
    size_t kept = 0;
    for (auto &r : e->retired) {
        if (!all && hipEventQuery(r.done) != hipSuccess) {
            (void)hipGetLastError();  // not-ready is no error
            e->retired[kept++] = r;
            continue;
        }
        (void)hipGraphExecDestroy(r.exec);
        (void)hipGraphDestroy(r.graph);
        (void)hipEventDestroy(r.done);
    }
    e->retired.resize(kept);
}

// Makes an unused set's entry free for another, without waiting: replays of its graph may still be on the stream, so the graph is put
// aside behind an event.  False where as many graphs as are kept lie there already.
static bool retireReplay(thip_executable_t *e, thip_executable_t::Replay *r) {
    if (!r->exec) return true;  // dispatched once, eagerly
    freeRetired(e, false);
    if (e->retired.size() >= kGraphsKept) return false;
    hipEvent_t done = nullptr;
    if (hipEventCreateWithFlags(&done, hipEventDisableTiming) != hipSuccess || hipEventRecord(done, e->stream) != hipSuccess) {
        (void)hipGetLastError();
        if (done) (void)hipEventDestroy(done);
        return false;
    }
    e->retired.push_back({r->graph, r->exec, done});
    r->graph = nullptr;
    r->exec = nullptr;
    return true;
}

// Takes the turn of a dispatch, if its launches are such that executables take turns.  *apart: it runs record by record what otherwise is one launch;
// `logged`: where a log or a dump is told of the records, in any case.
static thip_status_t takeTurn(thip_executable_t *e, uint8_t *const *bp, ChainTurns::Turn *turn, bool logged, bool *apart) {
    bool chained = true;
    if (e->chained) {
        const bool wanted = !(logged && tellsRecords(e)) && !chainAliased(e, bp);
        THIP_HIP(turn->take(&ChainTurns::of(e->device->ordinal), &e->chain, wanted, &chained), "waiting for another executable's launch");
    }
    *apart = !chained;
    return THIP_OK;
}

// Enqueues one dispatch on device bindings, through the set's graph when there is one.
static thip_status_t enqueueDevice(thip_executable_t *e, uint8_t *const *bp) {
    ChainTurns::Turn turn;
    bool apart;
    if (thip_status_t s = takeTurn(e, bp, &turn, true, &apart)) return s;
    if (apart) return enqueueOps(e, bp, true);
    const uint32_t nb = e->header.binding_count;
    const bool eligible = !e->graphsDisabled && replayPays(e->steps.size(), e->header.total_size - e->header.data_offset) && !tellsRecords(e);
    if (!eligible) return enqueueOps(e, bp);
    thip_executable_t::Replay *r = nullptr, *oldest = nullptr;
    for (auto &x : e->replays) {
        if (std::equal(x.ptrs.begin(), x.ptrs.end(), bp)) {
            r = &x;
            break;
        }
        if (!oldest || x.lastUse < oldest->lastUse) oldest = &x;
    }
    if (!r) {  // first time with these pointers: run eagerly (this also configures the kernels)
        if (e->replays.size() < kGraphsKept) {
            e->replays.emplace_back();
            r = &e->replays.back();
        } else if (e->invocation - oldest->lastUse > kReplayMaxAge && retireReplay(e, oldest)) {
            r = oldest;
        }
        if (r) {
            r->ptrs.assign(bp, bp + nb);
            r->lastUse = e->invocation;
        }
        return enqueueOps(e, bp);
    }
    r->lastUse = e->invocation;
    if (r->exec) {
        THIP_HIP(hipGraphLaunch(r->exec, e->stream), "hipGraphLaunch");
        return THIP_OK;
    }
    THIP_HIP(hipStreamBeginCapture(e->stream, hipStreamCaptureModeThreadLocal), "hipStreamBeginCapture");
    const thip_status_t launched = enqueueOps(e, bp);
    const hipError_t ended = hipStreamEndCapture(e->stream, &r->graph);
    if (launched != THIP_OK || ended != hipSuccess || !r->graph || hipGraphInstantiate(&r->exec, r->graph, nullptr, nullptr, 0) != hipSuccess) {
        r->exec = nullptr;
        dropReplay(r);
        e->graphsDisabled = true;  // fall back to eager launches for good
        (void)hipGetLastError();
        if (launched != THIP_OK) return launched;
        return enqueueOps(e, bp);
    }
    THIP_HIP(hipGraphLaunch(r->exec, e->stream), "hipGraphLaunch");
    return THIP_OK;
}

extern "C" {

thip_status_t thip_device_create(int32_t ordinal, thip_device_t **out_device) {
    if (!out_device) return fail(THIP_INVALID_ARGUMENT, "null result pointer");
    *out_device = nullptr;
    int count = 0;
    hipError_t e = hipGetDeviceCount(&count);
    if (e != hipSuccess || count <= 0) {
        (void)hipGetLastError();
        return fail(THIP_UNAVAILABLE, "no HIP device is visible (%s)", e == hipSuccess ? "count is 0" : hipGetErrorString(e));
    }
    if (ordinal < 0 || ordinal >= count) return fail(THIP_INVALID_ARGUMENT, "device ordinal %d is outside 0..%d", ordinal, count - 1);
    hipDeviceProp_t prop;
    THIP_HIP(hipGetDeviceProperties(&prop, ordinal), "hipGetDeviceProperties");
    std::string arch = prop.gcnArchName;
    const size_t colon = arch.find(':');
    if (colon != std::string::npos) arch.resize(colon);
    if (arch != "gfx950") return fail(THIP_UNAVAILABLE, "device %d is %s; the kernels are built for gfx950 only", ordinal, arch.c_str());
    THIP_HIP(hipSetDevice(ordinal), "hipSetDevice");
    thip_device_t *d = new (std::nothrow) thip_device_t();
    if (!d) return fail(THIP_RESOURCE_EXHAUSTED, "out of memory");
    d->ordinal = ordinal;
    d->arch = arch;
    d->computeUnits = prop.multiProcessorCount;
    {
        // the address of this device's copy of the scratch array (the device is current)
        void *ptr = nullptr;
        const hipError_t se = staticScratchAddress(&ptr);
        if (se != hipSuccess) {
            delete d;
            return hipFail(se, "locating the static scratch array");
        }
        d->staticScratch = (uint8_t *)ptr;
    }
    *out_device = d;
    return THIP_OK;
}

void thip_device_destroy(thip_device_t *device) {
    if (!device) return;
    if (device->eventLog) fclose(device->eventLog);
    delete device;
}

thip_status_t thip_device_name(thip_device_t *device, char *name, size_t capacity) {
    if (!device || !name || capacity == 0) return fail(THIP_INVALID_ARGUMENT, "null argument");
    snprintf(name, capacity, "%s", device->arch.c_str());
    return THIP_OK;
}

thip_status_t thip_device_alloc(thip_device_t *device, size_t size, void **out_ptr) {
    if (!device || !out_ptr) return fail(THIP_INVALID_ARGUMENT, "null argument");
    *out_ptr = nullptr;
    THIP_HIP(hipSetDevice(device->ordinal), "hipSetDevice");
    THIP_HIP(hipMalloc(out_ptr, size ? size : 1), "hipMalloc");
    return THIP_OK;
}

thip_status_t thip_device_free(thip_device_t *device, void *ptr) {
    if (!device) return fail(THIP_INVALID_ARGUMENT, "null device");
    if (ptr) THIP_HIP(hipFree(ptr), "hipFree");
    return THIP_OK;
}

thip_status_t thip_device_h2d(thip_device_t *device, void *dst_device, const void *src_host, size_t size) {
    if (!device || (size && (!dst_device || !src_host))) return fail(THIP_INVALID_ARGUMENT, "null argument");
    if (size) THIP_HIP(hipMemcpy(dst_device, src_host, size, hipMemcpyHostToDevice), "hipMemcpy H2D");
    return THIP_OK;
}

thip_status_t thip_device_d2h(thip_device_t *device, void *dst_host, const void *src_device, size_t size) {
    if (!device || (size && (!dst_host || !src_device))) return fail(THIP_INVALID_ARGUMENT, "null argument");
    if (size) THIP_HIP(hipMemcpy(dst_host, src_device, size, hipMemcpyDeviceToHost), "hipMemcpy D2H");
    return THIP_OK;
}

thip_status_t thip_device_synchronize(thip_device_t *device) {
    if (!device) return fail(THIP_INVALID_ARGUMENT, "null device");
    THIP_HIP(hipDeviceSynchronize(), "hipDeviceSynchronize");
    return THIP_OK;
}

thip_status_t thip_device_set_event_log(thip_device_t *device, const char *csv_path) {
    if (!device) return fail(THIP_INVALID_ARGUMENT, "null device");
    std::lock_guard<std::mutex> lock(device->logMutex);
    if (device->eventLog) {
        fclose(device->eventLog);
        device->eventLog = nullptr;
    }
    if (csv_path && csv_path[0]) {
        device->eventLog = fopen(csv_path, "w");
        if (!device->eventLog) return fail(THIP_INVALID_ARGUMENT, "cannot open event log %s", csv_path);
        fprintf(device->eventLog, "dispatch_name,invocation_id,action_id,timestamp_us,event,kernel\n");
    }
    return THIP_OK;
}

thip_status_t thip_device_mfma_rate(thip_device_t *device, int32_t random_operands, int32_t workgroups, int32_t iterations, double *out_tops) {
    if (!device || !out_tops) return fail(THIP_INVALID_ARGUMENT, "null argument");
    if (workgroups <= 0 || iterations <= 0) return fail(THIP_INVALID_ARGUMENT, "workgroups and iterations must be positive");
    THIP_HIP(hipSetDevice(device->ordinal), "hipSetDevice");
    THIP_HIP(measureMfmaRate(random_operands, workgroups, iterations, nullptr, out_tops), "measuring the MFMA rate");
    return THIP_OK;
}

thip_status_t thip_device_stream_floor(thip_device_t *device, int32_t reads_per_write, size_t write_bytes, int32_t cold, double *out_microseconds) {
    return thip_device_stream_floor_tuned(device, reads_per_write, write_bytes, cold, out_microseconds, nullptr, 0);
}

thip_status_t thip_device_stream_floor_tuned(thip_device_t *device, int32_t reads_per_write, size_t write_bytes, int32_t cold, double *out_microseconds,
                                             char *out_variant, size_t variant_capacity) {
    if (!device || !out_microseconds) return fail(THIP_INVALID_ARGUMENT, "null argument");
    THIP_HIP(hipSetDevice(device->ordinal), "hipSetDevice");
    const hipError_t err = measureStreamRate(reads_per_write, write_bytes, cold, nullptr, out_microseconds, out_variant, variant_capacity);
    if (err == hipErrorInvalidValue) return fail(THIP_INVALID_ARGUMENT, "reads_per_write is 1, 2 or 4; write_bytes a multiple of 16 from 4 KiB to 2 GiB");
    THIP_HIP(err, "measuring the streaming floor");
    return THIP_OK;
}

thip_status_t thip_device_set_dump_dirs(thip_device_t *device, const char *io_data_dir, const char *buffers_dir) {
    if (!device) return fail(THIP_INVALID_ARGUMENT, "null device");
    const std::string io = io_data_dir ? io_data_dir : "", buffers = buffers_dir ? buffers_dir : "";
    for (const std::string *dir : {&io, &buffers}) {
        if (!dir->empty() && !makeDirs(*dir)) return fail(THIP_INVALID_ARGUMENT, "cannot create dump directory %s", dir->c_str());
    }
    device->dumpIoDir = io;
    device->dumpBuffersDir = buffers;
    return THIP_OK;
}

thip_status_t thip_executable_set_wait_timeout(thip_executable_t *e, int64_t milliseconds) {
    if (!e) return fail(THIP_INVALID_ARGUMENT, "null executable");
    std::lock_guard<std::mutex> lock(e->mutex);
    e->waitTimeoutMs = milliseconds;
    return THIP_OK;
}

static void dropPinned(thip_executable_t *e) {
    if (e->pinned.in) (void)hipHostFree(e->pinned.in);
    if (e->pinned.out) (void)hipHostFree(e->pinned.out);
    e->pinned.in = e->pinned.out = nullptr;
    for (hipEvent_t &event : e->pinned.done) {
        if (event) (void)hipEventDestroy(event);
        event = nullptr;
    }
}

void thip_executable_destroy(thip_executable_t *e) {
    if (!e) return;
    if (e->abandoned) {
        // a wait on this executable timed out.  If its work has finished since, clean up as usual; if not, kernels may
        // still be using its buffers: leave everything in place (the caller is expected to end the process)
        if (!e->stream || hipStreamQuery(e->stream) != hipSuccess) {
            (void)hipGetLastError();
            return;
        }
    }
    if (e->stream) (void)hipStreamSynchronize(e->stream);
    if (e->chained) ChainTurns::of(e->device->ordinal).leave(&e->chain);
    for (auto &r : e->replays) dropReplay(&r);
    freeRetired(e, true);
    for (uint8_t *p : e->tempPtrs) {
        if (p) (void)hipFree(p);
    }
    for (uint8_t *p : e->staging) {
        if (p) (void)hipFree(p);
    }
    for (uint8_t *p : e->stepBuffers) {
        if (p) (void)hipFree(p);
    }
    dropPinned(e);
    if (e->chain.gaveUp) (void)hipHostFree(e->chain.gaveUp);
    if (e->constData) (void)hipFree(e->constData);
    if (e->evStart) (void)hipEventDestroy(e->evStart);
    if (e->evStop) (void)hipEventDestroy(e->evStop);
    if (e->evDone) (void)hipEventDestroy(e->evDone);
    if (e->stream) (void)hipStreamDestroy(e->stream);
    delete e;
}

// Adds a launch to the executable's, with the buffers of its own that it needs.  It is asked for its kernels now, as the records were.  False:
// its launchers do not take it, or there is no memory for its buffers; its records, which need none, then run one by one.
static bool addStep(thip_executable_t *e, Step &&planned) {
    e->steps.push_back(std::move(planned));
    e->stepBuffers.insert(e->stepBuffers.end(), 2, nullptr);
    Step &step = e->steps.back();
    hipError_t err = hipSuccess;
    if (step.kind == kStepPadded) {
        uint8_t **buffers = &e->stepBuffers[e->stepBuffers.size() - 2];
        const size_t rows = (size_t)step.rows * step.to, constants = step.constants.size();
        auto room = [e](size_t bytes) { return e->tuning.stepBytes < 0 || (long long)bytes <= e->tuning.stepBytes; };
        if (step.copies) err = room(rows + constants) ? hipMalloc((void **)&buffers[0], rows) : hipErrorOutOfMemory;
        if (step.asIs && err != hipSuccess) {  // goes without
            (void)hipGetLastError();
            buffers[0] = nullptr;
            err = hipSuccess;
        }
        if (err == hipSuccess && !room(constants)) err = hipErrorOutOfMemory;
        if (err == hipSuccess) err = hipMalloc((void **)&buffers[1], step.constants.size());
        if (err == hipSuccess) err = hipMemcpy(buffers[1], step.constants.data(), step.constants.size(), hipMemcpyHostToDevice);
        std::vector<uint8_t>().swap(step.constants);
    }
    if (step.kind == kStepDecChain) {
        uint8_t **buffers = &e->stepBuffers[e->stepBuffers.size() - 2];
        // operands that are no bindings lie where they will stay
        auto at = [e](const DescRef &r) { return r.space == kSpaceBinding ? ((ChainRef)(r.index + 1) << 56) | r.offset : (ChainRef)(uintptr_t)resolve(e, r, nullptr); };
        const Chain chain = layoutChain(viewOf(e), step.first, step.count, e->device->computeUnits, at);
        if (chain.phases.size() != step.count) err = hipErrorInvalidValue;
        step.xRoom = chain.xRoom;
        step.redRoom = chain.redRoom;
        const size_t tableBytes = chain.phases.size() * sizeof(ChainPhase), syncBytes = 4 * (kChainSyncHead + chain.exchangeWords);
        if (e->tuning.stepBytes >= 0 && (long long)(tableBytes + syncBytes) > e->tuning.stepBytes) err = hipErrorOutOfMemory;
        if (err == hipSuccess) err = hipMalloc((void **)&buffers[0], tableBytes);
        if (err == hipSuccess) err = hipMalloc((void **)&buffers[1], syncBytes);
        if (err == hipSuccess) err = hipMemcpy(buffers[0], chain.phases.data(), tableBytes, hipMemcpyHostToDevice);
        if (err == hipSuccess) err = hipMemset(buffers[1], 0, syncBytes);
        if (err == hipSuccess && !e->chain.gaveUp) {
            err = hipHostMalloc((void **)&e->chain.gaveUp, sizeof(uint32_t), hipHostMallocMapped | hipHostMallocCoherent);
            if (err == hipSuccess) *e->chain.gaveUp = 0;
        }
        void *tell = nullptr;
        if (err == hipSuccess) err = hipHostGetDevicePointer(&tell, e->chain.gaveUp, 0);
        if (err == hipSuccess) err = hipMemcpy(buffers[1] + 4 * kChainTell, &tell, sizeof(tell), hipMemcpyHostToDevice);
        if (err == hipSuccess && !e->chained) {
            e->chain.stream = e->stream;
            e->chain.always = e->tuning.decChain == 1;
            err = ChainTurns::of(e->device->ordinal).join(&e->chain);
            e->chained = err == hipSuccess;
        }
    }
    if (err == hipSuccess) {
        uint8_t *placeholder[64];
        for (auto &ptr : placeholder) ptr = (uint8_t *)(uintptr_t)0x1000000;
        char name[96] = "";
        if (launchStep(e, step, placeholder, LaunchCtx{nullptr, &e->tuning, name, sizeof(name), e->device->ordinal}) == THIP_OK) {
            if (step.kind == kStepPadded && !step.asIs) e->launchNames.push_back("pad_rows_i8");
            e->launchNames.push_back(name[0] ? name : opKernelName(e->ops[step.first]));
            return true;
        }
    }
    (void)hipGetLastError();
    for (int k = 0; k < 2; k++) {
        if (uint8_t *p = e->stepBuffers.back()) (void)hipFree(p);
        e->stepBuffers.pop_back();
    }
    e->steps.pop_back();
    return false;
}

thip_status_t thip_executable_create(thip_device_t *device, const void *blob, size_t size, const uint32_t *constants,
                                     size_t constant_count, thip_executable_t **out_executable) {
    if (!out_executable) return fail(THIP_INVALID_ARGUMENT, "null result pointer");
    *out_executable = nullptr;
    if (!device) return fail(THIP_INVALID_ARGUMENT, "null device");
    if (constant_count > 0 && !constants) return fail(THIP_INVALID_ARGUMENT, "constants pointer is NULL");
    DescHeader h;
    if (thip_status_t s = validateDescriptor((const uint8_t *)blob, size, &h)) return s;
    thip_executable_t *e = new (std::nothrow) thip_executable_t();
    if (!e) return fail(THIP_RESOURCE_EXHAUSTED, "out of memory");
    e->device = device;
    e->blob.assign((const uint8_t *)blob, (const uint8_t *)blob + h.total_size);
    if (constant_count) e->constants.assign(constants, constants + constant_count);
    e->header = h;
    e->ops = (const DescOp *)(e->blob.data() + h.ops_offset);
    e->bindings = (const DescBinding *)(e->blob.data() + h.bindings_offset);
    e->temps = (const DescTemp *)(e->blob.data() + h.temps_offset);
    e->consts = (const DescConst *)(e->blob.data() + h.consts_offset);
    thip_status_t s = THIP_OK;
    {
        const DescriptorView view = viewOf(e);
        for (uint32_t i = 0; i < h.op_count && s == THIP_OK; i++) s = checkOpFootprint(&view, i);
    }
    auto bail = [&](thip_status_t code) {
        thip_executable_destroy(e);
        return code;
    };
    if (s != THIP_OK) return bail(s);
    hipError_t err = hipSetDevice(device->ordinal);
    if (err == hipSuccess) err = hipStreamCreate(&e->stream);  // default priority
    if (err == hipSuccess) err = hipEventCreate(&e->evStart);
    if (err == hipSuccess) err = hipEventCreate(&e->evStop);
    if (err == hipSuccess) err = hipEventCreateWithFlags(&e->evDone, hipEventDisableTiming);
    if (err != hipSuccess) return bail(hipFail(err, "creating the stream"));
    const uint64_t dataSize = h.total_size - h.data_offset;
    if (dataSize) {
        err = hipMalloc((void **)&e->constData, dataSize);
        if (err == hipSuccess) err = hipMemcpy(e->constData, e->blob.data() + h.data_offset, dataSize, hipMemcpyHostToDevice);
        if (err != hipSuccess) return bail(hipFail(err, "uploading the constant segment"));
    }
    e->tempPtrs.assign(h.temp_count, nullptr);
    for (uint32_t i = 0; i < h.temp_count; i++) {
        const uint64_t bytes = e->temps[i].size ? e->temps[i].size : 1;
        err = hipMalloc((void **)&e->tempPtrs[i], bytes);
        // zero-filled once: padding regions of packed run-time operands rely on it
        if (err == hipSuccess) err = hipMemset(e->tempPtrs[i], 0, bytes);
        if (err != hipSuccess) return bail(hipFail(err, "allocating an intermediate"));
    }
    e->staging.assign(h.binding_count, nullptr);
    e->graphsDisabled = getenv("THIP_NO_GRAPH") != nullptr;
    if (const char *t = getenv("THIP_WAIT_TIMEOUT_MS")) e->waitTimeoutMs = atoll(t);
    // Which kernel each record runs is settled now, from the record, the alignment of its operands and the
    // environment's switches, and kept: the launchers are asked in naming mode (they also configure their kernels,
    // which must not happen later inside a stream capture).  Bindings stand in as aligned placeholder addresses:
    // device bindings must be 16-byte aligned and staged host bindings are, so a dispatch resolves the same way.
    e->scratchOffset.assign(h.op_count, 0);
    for (uint32_t i = 0; i < h.op_count; i++) {
        const DescOp &op = e->ops[i];
        if (op.kind != kKindFcBf16 || op.w0 <= 1) continue;
        e->scratchOffset[i] = e->scratchBytes;
        e->scratchBytes += (fcBf16WorkspaceBytes(op.M, op.Nn, op.w0) + 255) / 256 * 256;
    }
    e->tuning = tuningFromEnvironment();
    e->kernelNames.assign(h.op_count, std::string());
    {
        uint8_t *placeholder[64];
        for (auto &ptr : placeholder) ptr = (uint8_t *)(uintptr_t)0x1000000;
        for (uint32_t i = 0; i < h.op_count; i++) {
            char name[96] = "";
            if (thip_status_t st = launchOp(e, i, e->ops[i], placeholder, LaunchCtx{nullptr, &e->tuning, name, sizeof(name), e->device->ordinal})) return bail(st);
            e->kernelNames[i] = name[0] ? name : opKernelName(e->ops[i]);
        }
    }
    std::vector<Step> planned;
    try {
        planned = planSteps(viewOf(e), e->tuning);
    } catch (const std::bad_alloc &) {  // no room on the host to lay a launch's operands out
        Tuning plain = e->tuning;
        plain.plainRecords = true;
        planned = planSteps(viewOf(e), plain);
    }
    for (Step &step : planned) {
        const uint32_t first = step.first, count = step.count;
        if (addStep(e, std::move(step))) continue;
        for (uint32_t i = first; i < first + count; i++) {
            Step record{};
            record.kind = kStepRecord;
            record.first = i;
            record.count = 1;
            if (!addStep(e, std::move(record))) return bail(fail(THIP_INTERNAL, "op %u (%s): no kernel takes it", i, e->kernelNames[i].c_str()));
        }
    }
    *out_executable = e;
    return THIP_OK;
}

static thip_status_t refuseAbandoned(const thip_executable_t *e) {
    if (!e->abandoned) return THIP_OK;
    return fail(THIP_FAILED_PRECONDITION, "an earlier wait on this executable timed out; it cannot be used any more");
}

// ---- host bindings -----------------------------------------------------------------------------------------------
// The runtime copies a program's own (pageable) memory with one thread, and then into device memory, or pins and unpins its pages: 4.8 MB take 180 us,
// 64 KB 33, and back 300 and 34.  Out of pinned memory they are 91 and 9.  So a dispatch copies to pinned memory itself, with the device's CopyCrew,
// while what is already there is on its way, and goes on to launch its kernels behind it: 32 images of 224 x 224 through a mobile network 442 us -> 415,
// 128 of them 1093 -> 985, one 185 -> 178.  (Its launches replayed as a graph instead: 178, 422 and 986.)
// The link carries 53 bytes/ns and a copy more costs 9 us (4.8 MB in one 92 us, in two 101, in five 130), so what is there is sent when the link is
// about to run dry, and not before.
constexpr size_t kLinkBytesPerNs = 53, kCopyStartNs = 8000;
constexpr size_t kPinnedHalf = 8u << 20;     // two of them: bindings that are larger go through them piece by piece
constexpr size_t kPinnedResult = 1u << 20;   // a larger result comes back by the runtime: through pinned memory the copy behind it would cost as much
constexpr size_t kPinnedResults = 4u << 20;
static_assert(2 * kPinnedHalf <= CopyCrew::kMaxPieces * CopyCrew::kPiece, "");
static size_t pinnedBytes(uint64_t bytes) { return (size_t)((bytes + 255) / 256 * 256); }

static void makePinned(thip_executable_t *e) {
    if (e->pinned.tried) return;
    e->pinned.tried = true;
    uint64_t in = 0, out = 0;
    for (uint32_t i = 0; i < e->header.binding_count; i++) {
        const DescBinding &b = e->bindings[i];
        if (b.flags & kBindingRead) in = std::min<uint64_t>(in + pinnedBytes(std::min<uint64_t>(b.size, 2 * kPinnedHalf)), 2 * kPinnedHalf);
        if ((b.flags & kBindingWritten) && b.size <= kPinnedResult && out + pinnedBytes(b.size) <= kPinnedResults) out += pinnedBytes(b.size);
    }
    // what fits has no boundary to be cut at, and needs no second half
    const bool fits = in < 2 * kPinnedHalf;
    e->pinned.half = fits ? std::max<size_t>(in, 256) : kPinnedHalf;
    bool ok = hipHostMalloc((void **)&e->pinned.in, fits ? e->pinned.half : 2 * e->pinned.half, hipHostMallocDefault) == hipSuccess;
    ok = ok && hipHostMalloc((void **)&e->pinned.out, std::max<size_t>(out, 256), hipHostMallocDefault) == hipSuccess;
    for (hipEvent_t &event : e->pinned.done) ok = ok && hipEventCreateWithFlags(&event, hipEventDisableTiming) == hipSuccess;
    if (!ok) {
        (void)hipGetLastError();
        dropPinned(e);
    }
}

// Memory that the runtime knows (pinned by the caller, or on a device): it copies that without a detour.
static bool runtimeKnows(const void *p) {
    hipPointerAttribute_t at;
    if (hipPointerGetAttributes(&at, p) == hipSuccess) return at.type != hipMemoryTypeUnregistered;
    (void)hipGetLastError();
    return false;
}

// A dispatch's place in the two halves.
struct PinnedPlace {
    size_t at = 0;                     // of both
    bool used[2] = {false, false};     // copies out of it have been enqueued
    std::chrono::steady_clock::time_point idle;  // about when the link is through with them
};

// Copies host memory to `device` on the executable's stream; the host memory has been read when it returns.
static thip_status_t stageIn(thip_executable_t *e, PinnedPlace *place, uint8_t *device, const uint8_t *host, size_t bytes) {
    const size_t half = e->pinned.half;
    while (bytes > 0) {
        if (place->at == 2 * half) place->at = 0;
        const int h = place->at >= half;
        if (place->at == (size_t)h * half && place->used[h]) {
            if (thip_status_t s = waitBounded(e, e->pinned.done[h], "staging a binding")) return s;
        }
        const size_t n = std::min(bytes, (size_t)(h + 1) * half - place->at);
        uint8_t *pinned = e->pinned.in + place->at;
        CopyCrew::Copy copy(&e->device->crew, pinned, host, n);
        for (size_t sent = 0; sent < n;) {
            const bool copied = copy.step();
            const size_t there = copy.ready();
            const auto now = std::chrono::steady_clock::now();
            if (there > sent && (there == n || now >= place->idle)) {
                THIP_HIP(hipMemcpyAsync(device + sent, pinned + sent, there - sent, hipMemcpyHostToDevice, e->stream), "staging a binding");
                place->idle = std::max(now, place->idle) + std::chrono::nanoseconds(kCopyStartNs + (there - sent) / kLinkBytesPerNs);
                sent = there;
            } else if (!copied) {
                std::this_thread::yield();  // the last pieces are others'
            }
        }
        device += n;
        host += n;
        bytes -= n;
        place->at += std::min(pinnedBytes(n), (size_t)(h + 1) * half - place->at);
        place->used[h] = true;
        if (place->at == (size_t)(h + 1) * half) THIP_HIP(hipEventRecord(e->pinned.done[h], e->stream), "staging a binding");
    }
    return THIP_OK;
}

static thip_status_t runLocked(thip_executable_t *e, const thip_dispatch_state_t *st) {
    if (thip_status_t s = refuseAbandoned(e)) return s;
    THIP_HIP(hipSetDevice(e->device->ordinal), "hipSetDevice");
    uint8_t *bp[64] = {nullptr};
    const int32_t lastOp = (int32_t)e->header.op_count - 1;
    logEvent(e, e->invocation, 0, "DISPATCH", "BEGIN", "");
    logEvent(e, e->invocation, 0, "DISPATCH_SYNC_BINDINGS_IN", "BEGIN", "");
    PinnedPlace place;
    // writeInputs: host bindings are staged into device memory (TorqExecutable::writeInputs)
    for (uint32_t i = 0; i < e->header.binding_count; i++) {
        if (e->bindings[i].flags == 0) continue;
        const bool isDevice = st->binding_flags && (st->binding_flags[i] & THIP_BINDING_DEVICE);
        if (isDevice) {
            bp[i] = (uint8_t *)st->binding_ptrs[i];
            continue;
        }
        if (!e->staging[i]) {
            THIP_HIP(hipMalloc((void **)&e->staging[i], e->bindings[i].size ? e->bindings[i].size : 1), "allocating binding staging");
        }
        bp[i] = e->staging[i];
        if (e->bindings[i].flags & kBindingRead) {
            dumpBinding(e, i, st->binding_ptrs[i], e->bindings[i].size, true);
            makePinned(e);
            if (e->pinned.in && !runtimeKnows(st->binding_ptrs[i])) {
                if (thip_status_t s = stageIn(e, &place, bp[i], (const uint8_t *)st->binding_ptrs[i], e->bindings[i].size)) return s;
            } else {
                THIP_HIP(hipMemcpyAsync(bp[i], st->binding_ptrs[i], e->bindings[i].size, hipMemcpyHostToDevice, e->stream), "staging a binding");
            }
        }
    }
    logEvent(e, e->invocation, 0, "DISPATCH_SYNC_BINDINGS_IN", "END", "");
    bool allDevice = true;
    for (uint32_t i = 0; i < e->header.binding_count; i++) {
        if (e->bindings[i].flags != 0 && !(st->binding_flags && (st->binding_flags[i] & THIP_BINDING_DEVICE))) allDevice = false;
    }
    logEvent(e, e->invocation, 0, "DISPATCH_EXECUTE_ACTIONS", "BEGIN", "");
    auto enqueueStaged = [&] {
        ChainTurns::Turn turn;
        bool apart;
        const thip_status_t s = takeTurn(e, bp, &turn, true, &apart);
        return s != THIP_OK ? s : enqueueOps(e, bp, apart);
    };
    if (thip_status_t s = allDevice ? enqueueDevice(e, bp) : enqueueStaged()) {
        // what was enqueued before the failure still runs: wait for it (bounded; the launch error is what is reported)
        std::string message = thip_status_message();
        if (!e->abandoned) (void)waitBounded(e, "waiting after a failed launch");
        e->invocation++;
        return fail(s, "%s", message.c_str());
    }
    logEvent(e, e->invocation, lastOp, "DISPATCH_EXECUTE_ACTIONS", "END", "");
    logEvent(e, e->invocation, lastOp, "DISPATCH_SYNC_BINDINGS_OUT", "BEGIN", "");
    uint8_t *fromPinned[64] = {nullptr};
    size_t results = 0;
    // readOutputs (TorqExecutable::readOutputs, runtime/driver/TorqExecutable.cc:860-918)
    for (uint32_t i = 0; i < e->header.binding_count; i++) {
        const bool isDevice = st->binding_flags && (st->binding_flags[i] & THIP_BINDING_DEVICE);
        if (isDevice || !(e->bindings[i].flags & kBindingWritten)) continue;
        const size_t size = e->bindings[i].size;
        makePinned(e);
        uint8_t *to = (uint8_t *)st->binding_ptrs[i];
        if (e->pinned.out && size <= kPinnedResult && results + pinnedBytes(size) <= kPinnedResults && !runtimeKnows(to)) {
            to = fromPinned[i] = e->pinned.out + results;
            results += pinnedBytes(size);
        }
        THIP_HIP(hipMemcpyAsync(to, bp[i], size, hipMemcpyDeviceToHost, e->stream), "reading back a binding");
    }
    logEvent(e, e->invocation, lastOp, "NSS_WAIT", "BEGIN", "");
    const thip_status_t waited = waitBounded(e, "waiting for the dispatch");
    const std::string waitMessage = waited == THIP_OK ? std::string() : std::string(thip_status_message());
    logEvent(e, e->invocation, lastOp, "NSS_WAIT", "END", "");
    logEvent(e, e->invocation, lastOp, "DISPATCH_SYNC_BINDINGS_OUT", "END", "");
    logEvent(e, e->invocation, lastOp, "DISPATCH", "END", "");
    e->invocation++;
    if (waited != THIP_OK) return fail(waited, "%s", waitMessage.c_str());
    for (uint32_t i = 0; i < e->header.binding_count; i++) {
        if (fromPinned[i]) memcpy(st->binding_ptrs[i], fromPinned[i], e->bindings[i].size);
        const bool isDevice = st->binding_flags && (st->binding_flags[i] & THIP_BINDING_DEVICE);
        if (!isDevice && (e->bindings[i].flags & kBindingWritten)) dumpBinding(e, i, st->binding_ptrs[i], e->bindings[i].size, false);
    }
    return THIP_OK;
}

thip_status_t thip_executable_run(thip_executable_t *e, const thip_dispatch_state_t *st) {
    if (!e) return fail(THIP_INVALID_ARGUMENT, "null executable");
    if (thip_status_t s = checkState(e, st, false)) return s;
    std::lock_guard<std::mutex> lock(e->mutex);
    return runLocked(e, st);
}

thip_status_t thip_executable_enqueue(thip_executable_t *e, const thip_dispatch_state_t *st) {
    if (!e) return fail(THIP_INVALID_ARGUMENT, "null executable");
    if (thip_status_t s = checkState(e, st, true)) return s;
    std::lock_guard<std::mutex> lock(e->mutex);
    if (thip_status_t s = refuseAbandoned(e)) return s;
    THIP_HIP(hipSetDevice(e->device->ordinal), "hipSetDevice");
    uint8_t *bp[64] = {nullptr};
    for (uint32_t i = 0; i < e->header.binding_count; i++) bp[i] = (uint8_t *)st->binding_ptrs[i];
    const thip_status_t s = enqueueDevice(e, bp);
    e->invocation++;
    return s;
}

thip_status_t thip_executable_enqueue_noalloc(thip_executable_t *e, const thip_dispatch_state_t *st) {
    if (!e) return fail(THIP_INVALID_ARGUMENT, "null executable");
    if (thip_status_t s = checkState(e, st, true)) return s;
    if (e->scratchBytes > kStaticScratchBytes) {
        return fail(THIP_RESOURCE_EXHAUSTED, "the program's kernels need %llu bytes of scratch, the static array holds %llu",
                    (unsigned long long)e->scratchBytes, (unsigned long long)kStaticScratchBytes);
    }
    std::lock_guard<std::mutex> lock(e->mutex);
    if (thip_status_t s = refuseAbandoned(e)) return s;
    THIP_HIP(hipSetDevice(e->device->ordinal), "hipSetDevice");
    uint8_t *scratch = e->device->staticScratch;  // the address hipGetSymbolAddress gave for this device
    if (!scratch) return fail(THIP_INTERNAL, "the static scratch array was not located");
    uint8_t *bp[64] = {nullptr};
    for (uint32_t i = 0; i < e->header.binding_count; i++) bp[i] = (uint8_t *)st->binding_ptrs[i];
    const LaunchCtx ctx{e->stream, &e->tuning, nullptr, 0, e->device->ordinal};
    ChainTurns::Turn turn;
    bool apart;
    thip_status_t result = takeTurn(e, bp, &turn, false, &apart);
    for (const Step &s : e->steps) {
        // the array keeps what the last call left there, whoever made it; nothing in a K-split workspace has to start
        // at zero (every slot that is read has been written by the same dispatch)
        if (result == THIP_OK) result = launchStep(e, s, bp, ctx, scratch, apart);
    }
    e->invocation++;
    return result;
}

thip_status_t thip_executable_wait(thip_executable_t *e) {
    if (!e) return fail(THIP_INVALID_ARGUMENT, "null executable");
    std::lock_guard<std::mutex> lock(e->mutex);
    if (thip_status_t s = refuseAbandoned(e)) return s;
    return waitBounded(e, "waiting for the dispatch");
}

thip_status_t thip_executable_time(thip_executable_t *e, const thip_dispatch_state_t *st, int32_t iterations, float *out_ms) {
    if (!e || !out_ms) return fail(THIP_INVALID_ARGUMENT, "null argument");
    if (iterations <= 0) return fail(THIP_INVALID_ARGUMENT, "iterations must be positive");
    if (thip_status_t s = checkState(e, st, true)) return s;
    std::lock_guard<std::mutex> lock(e->mutex);
    if (thip_status_t as = refuseAbandoned(e)) return as;
    THIP_HIP(hipSetDevice(e->device->ordinal), "hipSetDevice");
    uint8_t *bp[64] = {nullptr};
    for (uint32_t i = 0; i < e->header.binding_count; i++) bp[i] = (uint8_t *)st->binding_ptrs[i];
    THIP_HIP(hipEventRecord(e->evStart, e->stream), "hipEventRecord");
    for (int32_t it = 0; it < iterations; it++) {
        const thip_status_t s = enqueueDevice(e, bp);
        e->invocation++;
        if (s != THIP_OK) {
            (void)hipStreamSynchronize(e->stream);
            return s;
        }
    }
    THIP_HIP(hipEventRecord(e->evStop, e->stream), "hipEventRecord");
    if (thip_status_t ws = waitBounded(e, "waiting for the timed dispatches")) return ws;
    float ms = 0.f;
    THIP_HIP(hipEventElapsedTime(&ms, e->evStart, e->evStop), "hipEventElapsedTime");
    *out_ms = ms / (float)iterations;
    return THIP_OK;
}

thip_status_t thip_executable_time_rotating(thip_executable_t *e, const thip_dispatch_state_t *states, uint32_t state_count,
                                            int32_t iterations, float *out_ms) {
    if (!e || !out_ms || !states) return fail(THIP_INVALID_ARGUMENT, "null argument");
    if (iterations <= 0 || state_count == 0) return fail(THIP_INVALID_ARGUMENT, "iterations and state_count must be positive");
    for (uint32_t s = 0; s < state_count; s++) {
        if (thip_status_t st = checkState(e, &states[s], true)) return st;
    }
    std::lock_guard<std::mutex> lock(e->mutex);
    if (thip_status_t as = refuseAbandoned(e)) return as;
    THIP_HIP(hipSetDevice(e->device->ordinal), "hipSetDevice");
    THIP_HIP(hipEventRecord(e->evStart, e->stream), "hipEventRecord");
    for (int32_t it = 0; it < iterations; it++) {
        const thip_dispatch_state_t &st = states[(uint32_t)it % state_count];
        uint8_t *bp[64] = {nullptr};
        for (uint32_t i = 0; i < e->header.binding_count; i++) bp[i] = (uint8_t *)st.binding_ptrs[i];
        const thip_status_t s = enqueueDevice(e, bp);
        e->invocation++;
        if (s != THIP_OK) {
            (void)hipStreamSynchronize(e->stream);
            return s;
        }
    }
    THIP_HIP(hipEventRecord(e->evStop, e->stream), "hipEventRecord");
    if (thip_status_t ws = waitBounded(e, "waiting for the timed dispatches")) return ws;
    float ms = 0.f;
    THIP_HIP(hipEventElapsedTime(&ms, e->evStart, e->evStop), "hipEventElapsedTime");
    *out_ms = ms / (float)iterations;
    return THIP_OK;
}

thip_status_t thip_executable_op_count(thip_executable_t *e, uint32_t *out_count) {
    if (!e || !out_count) return fail(THIP_INVALID_ARGUMENT, "null argument");
    *out_count = e->header.op_count;
    return THIP_OK;
}

thip_status_t thip_executable_op_kernel(thip_executable_t *e, uint32_t index, char *name, size_t capacity) {
    if (!e || !name || capacity == 0) return fail(THIP_INVALID_ARGUMENT, "null argument");
    if (index >= e->header.op_count) return fail(THIP_OUT_OF_RANGE, "op %u of %u", index, e->header.op_count);
    snprintf(name, capacity, "%s", e->kernelNames[index].c_str());
    return THIP_OK;
}

thip_status_t thip_executable_launch_count(thip_executable_t *e, uint32_t *out_count) {
    if (!e || !out_count) return fail(THIP_INVALID_ARGUMENT, "null argument");
    *out_count = (uint32_t)e->launchNames.size();
    return THIP_OK;
}

thip_status_t thip_executable_launch_kernel(thip_executable_t *e, uint32_t index, char *name, size_t capacity) {
    if (!e || !name || capacity == 0) return fail(THIP_INVALID_ARGUMENT, "null argument");
    if (index >= e->launchNames.size()) return fail(THIP_OUT_OF_RANGE, "launch %u of %zu", index, e->launchNames.size());
    snprintf(name, capacity, "%s", e->launchNames[index].c_str());
    return THIP_OK;
}

thip_status_t thip_executable_binding_count(thip_executable_t *e, uint32_t *out_count) {
    if (!e || !out_count) return fail(THIP_INVALID_ARGUMENT, "null argument");
    *out_count = e->header.binding_count;
    return THIP_OK;
}

thip_status_t thip_executable_binding_size(thip_executable_t *e, uint32_t binding, size_t *out_size) {
    if (!e || !out_size) return fail(THIP_INVALID_ARGUMENT, "null argument");
    if (binding >= e->header.binding_count) return fail(THIP_OUT_OF_RANGE, "binding %u of %u", binding, e->header.binding_count);
    *out_size = (size_t)e->bindings[binding].size;
    return THIP_OK;
}

}  // extern "C"
