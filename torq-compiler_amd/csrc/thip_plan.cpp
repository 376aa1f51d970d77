#include "thip_plan.h"

#include <math.h>
#include <string.h>

#include <algorithm>

#include "../../include/thip.h"
#include "thip_kernels.h"

namespace thip {

static int64_t roundUp(int64_t v, int64_t to) { return (v + to - 1) / to * to; }
static size_t elemBytes(int32_t dtype) { return dtype == 1 ? 1 : dtype == 2 ? 2 : 4; }
static bool sameRef(const DescRef &a, const DescRef &b) { return a.space == b.space && a.index == b.index && a.offset == b.offset; }
static bool sameBuffer(const DescRef &a, const DescRef &b) { return a.space == b.space && a.index == b.index; }

// How often `n` records from `first` on name each intermediate.
static std::vector<uint32_t> tempUses(const DescriptorView &v, uint32_t first, uint32_t n) {
    std::vector<uint32_t> uses(v.header.temp_count, 0);
    auto count = [&](const DescRef &r) {
        if (r.space == kSpaceTemp) uses[r.index]++;
    };
    for (uint32_t i = first; i < first + n; i++) {
        const DescOp &op = v.ops[i];
        for (const DescRef *r : {&op.in0, &op.in1, &op.weights, &op.bias, &op.scale, &op.table, &op.out}) count(*r);
        if (op.kind == kKindDecLinear) {
            DecLinearExt x;
            memcpy(&x, v.blob + v.header.data_offset + v.consts[op.table.index].offset + op.table.offset, sizeof(x));
            for (int m = 0; m < 3; m++) {
                for (const DescRef *r : {&x.weights[m], &x.bias[m], &x.out[m]}) count(*r);
            }
            count(x.res);
            count(x.add_out);
        }
    }
    return uses;
}

// Whether a GEMM-shaped record stores into the bytes of the buffer that it reads.
static bool inPlace(const DescOp &op) {
    if (!sameBuffer(op.in0, op.out)) return false;
    const uint64_t in = (uint64_t)op.N * op.H * op.W * op.C, out = (uint64_t)op.M * op.Nn * elemBytes(op.out_dtype);
    return op.in0.offset < op.out.offset + out && op.out.offset < op.in0.offset + in;
}

// The value all `n` words of a constant have; false where they differ or are none.
static bool uniformWords(const DescriptorView &v, const DescRef &r, int n, int32_t *out) {
    if (r.space != kSpaceConst) return false;
    const uint8_t *p = v.blob + v.header.data_offset + v.consts[r.index].offset + r.offset;
    for (int i = 0; i < n; i++) {
        int32_t w;
        memcpy(&w, p + (size_t)i * 4, 4);
        if (i == 0) *out = w;
        else if (w != *out) return false;
    }
    return n > 0;
}

// Transposes of one matrix (or of one per batch element) into intermediates, and behind them the GEMMs that read these.
static bool matchMatmulRt(const DescriptorView &v, const std::vector<uint32_t> &uses, uint32_t first, Step *s) {
    uint32_t n = first;
    while (n < v.header.op_count && v.ops[n].kind == kKindTranspose) n++;
    const uint32_t matrices = n - first;
    if (matrices == 0 || n == v.header.op_count) return false;
    const DescOp &t0 = v.ops[first], &g0 = v.ops[n];
    if (g0.kind != kKindIgemm || (g0.loader != kLoaderDense && g0.loader != kLoaderGather) || g0.in1.space != kSpaceNone) return false;
    const int64_t M = g0.M, K = g0.K, N = g0.Nn;
    // a 1 x 1 window over a [M][K] matrix: what torq_hl.matmul becomes under either loader
    if (g0.H != 1 || g0.W != 1 || g0.OH != 1 || g0.OW != 1 || g0.KH != 1 || g0.KW != 1 || g0.PT != 0 || g0.PL != 0 || g0.N != M || g0.C != K) return false;
    for (uint32_t i = 0; i < matrices; i++) {
        const DescOp &t = v.ops[first + i];
        if (t.gran == 2 || t.TB != 1 || t.TR != K || t.TS != N || t.TP != g0.Kp || t.out.space != kSpaceTemp || t.out.offset != 0) return false;
        if (!sameBuffer(t.in0, t0.in0) || t.in0.offset != t0.in0.offset + (uint64_t)i * (uint64_t)(K * N)) return false;
    }
    uint32_t batches = 0;
    while (n + batches < v.header.op_count) {
        const DescOp &g = v.ops[n + batches];
        if (g.kind != kKindIgemm || g.weights.space != kSpaceTemp) break;
        if (!sameRef(g.weights, v.ops[first + (matrices == 1 ? 0 : batches < matrices ? batches : 0)].out)) break;
        batches++;
        if (matrices > 1 && batches == matrices) break;
    }
    if (batches == 0 || (matrices > 1 && batches != matrices)) return false;
    const uint64_t aStep = batches > 1 ? v.ops[n + 1].in0.offset - g0.in0.offset : 0, outStep = (uint64_t)(M * N) * elemBytes(g0.out_dtype);
    if (aStep != 0 && aStep != (uint64_t)(M * K)) return false;
    for (uint32_t i = 0; i < batches; i++) {
        const DescOp &g = v.ops[n + i];
        if (!sameBuffer(g.in0, g0.in0) || g.in0.offset != g0.in0.offset + i * aStep || !sameBuffer(g.out, g0.out) || g.out.offset != g0.out.offset + i * outStep) return false;
        // everything else of the records is the same (their constants hold the same words)
        DescOp x = g, y = g0;
        for (DescOp *o : {&x, &y}) {
            for (DescRef *r : {&o->in0, &o->out, &o->weights, &o->bias, &o->scale, &o->table}) memset(r, 0, sizeof(*r));
        }
        int32_t bias, scale;
        if (memcmp(&x, &y, sizeof(x)) != 0 || !uniformWords(v, g.bias, (int)N, &bias) || !uniformWords(v, g.scale, (int)N, &scale)) return false;
        if (i == 0) {
            s->bias = bias;
            s->scale = scale;
        } else if (bias != s->bias || scale != s->scale) {
            return false;
        }
    }
    for (uint32_t i = 0; i < matrices; i++) {
        // written by its transpose, read by its GEMMs, and the operands are not what the step writes
        const DescRef &t = v.ops[first + i].out;
        if (uses[t.index] != 1 + (matrices == 1 ? batches : 1)) return false;
        for (uint32_t j = 0; j < i; j++) {
            if (v.ops[first + j].out.index == t.index) return false;
        }
    }
    if (sameBuffer(g0.out, g0.in0) || sameBuffer(g0.out, t0.in0)) return false;
    // a product this large is worth its transpose: the ring kernel behind it is faster per multiply-add (4096x2048x4096 48.9 us
    // against 57; 2048x1024x2048 16.0 against 13.0)
    if (M * N * K > (1LL << 34)) return false;
    if (!matmulRtFits((aStep ? (int64_t)batches : 1) * M * K, (int64_t)matrices * K * N, M, N, K)) return false;
    s->kind = kStepMatmulRt;
    s->first = first;
    s->count = matrices + batches;
    s->a = g0.in0;
    s->b = t0.in0;
    s->out = g0.out;
    s->batches = (int32_t)batches;
    s->a_stride = (int64_t)aStep;
    s->b_stride = matrices > 1 ? K * N : 0;
    s->out_stride = M * N;
    return true;
}

// Where an operand lies, for the rules that ask for alignments only: aligned as a dispatch's are.
static uint8_t *plannedAt(const DescriptorView &v, const DescRef &r) {
    return r.space == kSpaceNone ? nullptr : (uint8_t *)(uintptr_t)(0x1000000 + (r.space == kSpaceConst ? v.consts[r.index].offset : 0) + r.offset);
}

// Whether the requant of a record has a tail of 32-bit arithmetic (see WideRequant).
static bool narrowRequant(const DescOp &op) { return op.shift == 32 || (int64_t)op.shift + op.pre_shift >= 33; }

// Behind the two records that `s` stands for, the pointwise convolution that alone reads their result, its add folded into it or none.
static void matchBlock(const DescriptorView &v, const Tuning &tuning, const std::vector<uint32_t> &uses, Step *s) {
    const uint32_t last = s->first + 2;
    if (last >= v.header.op_count) return;
    const DescOp &e = v.ops[s->first], &d = v.ops[s->first + 1], &g = v.ops[last];
    if (g.kind != kKindIgemm || g.loader != kLoaderDense || g.KH != 1 || g.KW != 1 || g.SH != 1 || g.SW != 1 || g.out_dtype != 1) return;
    if (d.out.space != kSpaceTemp || !sameRef(d.out, g.in0) || uses[d.out.index] != 2 || g.K != d.C || g.M != (int64_t)d.N * d.OH * d.OW) return;
    for (const DescRef *r : {&g.weights, &g.bias, &g.scale, &g.out}) {
        if (r->offset % 16 != 0) return;
    }
    if (g.in1.space != kSpaceNone && g.in1.offset % 16 != 0) return;
    // workgroups read the rows around their own (what bindings share is only known with a dispatch: writesWhatItReads)
    for (const DescRef *r : {&e.in0, &e.weights, &e.bias, &e.scale, &d.weights, &d.bias, &d.scale, &g.in1, &g.weights, &g.bias, &g.scale}) {
        if (sameBuffer(g.out, *r)) return;
    }
    const IrBlockArgs a = irBlockArgs(v, *s, [&](const DescRef &r) { return plannedAt(v, r); });
    if (tuning.irBlock >= 0 ? tuning.irBlock != 0 && irBlockFits(a) : irBlockBetter(a)) s->count = 3;
}

// A pointwise convolution, or one over few channels, whose only reader is the 3 x 3 depthwise convolution right behind it, and with them the
// pointwise convolution behind that where the three are ahead as one launch.
static bool matchExpandDw(const DescriptorView &v, const Tuning &tuning, const std::vector<uint32_t> &uses, uint32_t first, Step *s) {
    if (first + 1 >= v.header.op_count) return false;
    const DescOp &e = v.ops[first], &d = v.ops[first + 1];
    const bool runs = e.loader == kLoaderRuns;
    if (e.kind != kKindIgemm || (!runs && (e.loader != kLoaderDense || e.KH != 1 || e.KW != 1)) || e.in1.space != kSpaceNone || e.out_dtype != 1) return false;
    if (runs && (e.SH != e.SW || e.OH != d.H || e.OW != d.W || e.N != d.N || (int64_t)e.N * e.H * e.W * e.C < 16 || (int64_t)e.H * e.W * e.C > (1LL << 27))) return false;
    if (d.kind != kKindDepthwise || d.variant != kDepthwiseDot4Rows || d.KH != 3 || d.KW != 3 || d.SH != d.SW) return false;
    if (e.out.space != kSpaceTemp || !sameRef(e.out, d.in0) || uses[e.out.index] != 2) return false;
    if (d.C != e.Nn || d.C > kIrMaxChannels || (int64_t)d.N * d.H * d.W != e.M || !narrowRequant(e) || !narrowRequant(d)) return false;
    if (!irExpandDwFits(e.K, runs ? e.KH : 0, d.OW, d.SW, d.PT, d.PL) || e.Kp < (runs ? (e.KH + 1) / 2 : (e.K + 31) / 32) * 32 || e.Np < (e.Nn + 31) / 32 * 32) return false;
    if ((int64_t)d.H * d.W * e.K >= (1LL << 31) || (d.OH - 1) * d.SH - d.PT >= d.H || (d.OW - 1) * d.SW - d.PL >= d.W) return false;
    for (const DescRef *r : {&e.in0, &e.weights, &e.bias, &e.scale, &d.weights, &d.bias, &d.scale, &d.out}) {
        if (r->offset % 16 != 0 && !(runs && r == &e.in0)) return false;
    }
    if (sameBuffer(d.out, e.in0)) return false;
    s->kind = kStepExpandDw;
    s->first = first;
    s->count = 2;
    IrExpandDwArgs a{};
    a.N = d.N; a.H = d.H; a.W = d.W; a.K = e.K; a.C = d.C; a.OH = d.OH; a.OW = d.OW; a.S = d.SW; a.PT = d.PT; a.PL = d.PL; a.CKH = runs ? e.KH : 0;
    if (irExpandDwTime(&a) < HUGE_VAL) {
        s->images = a.images;
        s->stripRows = a.stripRows;
    }
    matchBlock(v, tuning, uses, s);
    if (s->count == 3 || irExpandDwBetter((int64_t)d.N * d.H * d.W * d.C, d.OW, d.SW)) return true;
    *s = Step{};
    return false;
}

// Whether the copy of the rows and a kernel of aligned operands behind it are ahead of a record's own gather kernel, by the time that
// either takes (us; storing the results costs both the same).  A k-tile of 64 costs the gather 0.55, 0.85, 1.5 or 2.5 in pieces of 8, 4, 2 or
// 1 bytes and the aligned kernels 0.09, both more where the tiles outnumber the CUs; the copy is a launch (2.3) and its bytes at
// 4.2 TB/s.  Fitted to 429 linears and convolutions of 3 .. 8004 channels and 4 .. 204 800 rows; the choice costs 1.5 % of the better
// one's time over them, always padding 9 %.  Padded / own:
//   taken   1500x1333 -> 48 7.8 / 65.4, 4096x500 -> 1024 9.3 / 16.6, 60x776 -> 256 6.0 / 10.2, 200000x17 -> 16 8.7 / 20.4,
//           3x3 7x7x33 -> 64 5.5 / 15.4, 28x28x100 -> 64 6.3 / 15.6, 56x56x13 -> 24 by 5x5, batch 16 11.5 / 27.5
//   left    60x24 -> 64 5.4 / 3.2, 30000x72 -> 40 9.7 / 5.3, 100000x776 -> 64 44.0 / 39.0, 3x3 112x112x8 -> 32 6.3 / 4.3,
//           stride 2 112x112x40 -> 32, batch 32 22.3 / 15.6, 1x1 stride 2 56x56x264 -> 96, batch 4 7.3 / 5.9
//   wrong   30000x130 -> 40 11.2 / 9.5 (taken), 100000x500 -> 64 29.7 / 37.9, pointwise 56x56x24 -> 96, batch 32 9.6 / 14.4 (left)
static double gatherTime(const DescOp &g) {
    auto tilesOf = [](int64_t n) { return (double)((n + 63) / 64); };
    const double tiles = tilesOf(g.M) * tilesOf(g.Nn), beyond = tiles > 256 ? tiles - 256 : 0;
    const double step = g.gran >= 8 ? 0.55 : g.gran >= 4 ? 0.85 : g.gran >= 2 ? 1.5 : 2.5;
    return 2.8 + step * tilesOf(g.K) * (1 + beyond / 600);
}
static bool paddingPays(const DescOp &g, int64_t rows, int64_t Cp, int64_t K) {
    auto tilesOf = [](int64_t n) { return (double)((n + 63) / 64); };
    const double tiles = tilesOf(g.M) * tilesOf(g.Nn), beyond = tiles > 256 ? tiles - 256 : 0;
    const double padded = 5.1 + 0.24e-6 * (double)rows * (double)(g.C + Cp) + 0.09 * tilesOf(K) * (1 + beyond / 170);
    return padded + 0.8 < gatherTime(g);
}

// Whether igemm_direct_i8 takes the rows of the gathered record `g` as they are, as `op` (with its weights spread, or itself), and is ahead of its own
// kernel.  It is ahead of the copy and a kernel behind it as well, by that launch: over the 256 of 330 drawn linears and convolutions of 5 .. 7972
// channels that it takes, own kernel / copied rows / rows as they are cost 3.79 / 1.52 / 1.00 times the best, the choice over all 330 1.01 times (us: linear 9x100 -> 2303 5.5 / 6.4 / 4.0,
// 554x604 -> 117 13.4 / 6.6 / 4.0, 5x1379 -> 48 57.4 / 6.4 / 4.5; 3x3 30x30x98 -> 316 stride 2, batch 3 7.1 / 6.6 / 4.0, 56x56x40 -> 32, batch 2 6.5 / 6.5 / 4.0; stride 2
// 1x1 56x56x264 -> 96, batch 4 6.1 / 7.8 / 4.2).  Left where the gather is short (60x24 -> 64 3.6 / 6.1 / 3.8, 3x3 112x112x8 -> 32 4.5 / 6.7 / 4.1) and
// where K is long enough for the worse loads to cost that launch: 3x2801 -> 1608 - / 6.2 / 6.6 (few rows have a faster kernel behind the copy), 5x5
// 19x19x387 -> 134 452 / 18.2 / 19.7.
static bool asIsBetter(const DescriptorView &v, const Tuning &tuning, const DescOp &g, const DescOp &op) {
    if (tuning.padRows == 0 || tuning.padRows == 1 || g.kind != kKindIgemm || g.loader != kLoaderGather || inPlace(g)) return false;
    return igemmDirectBetter(raggedArgs(v, op, g.C, [&](const DescRef &r) { return plannedAt(v, r); })) && (tuning.padRows == 2 || (gatherTime(g) > 4.0 && g.K <= (g.M <= kFcSkinnyMaxRows ? 2500 : 9000)));
}

// Whether the weights of a window of one pixel are zeros from K to the end of the last chunk that igemm_direct_i8 reads, as they are packed.
static bool zerosBehindRows(const DescriptorView &v, const DescOp &op) {
    const int64_t end = roundUp(op.K, 32);
    if (op.weights.space != kSpaceConst || op.K != op.C || op.Kp < end) return false;
    const uint8_t *w = v.blob + v.header.data_offset + v.consts[op.weights.index].offset + op.weights.offset;
    for (int64_t n = 0; n < op.Nn; n++) {
        for (int64_t k = op.K; k < end; k++) {
            if (w[n * op.Kp + k] != 0) return false;
        }
    }
    return true;
}

// A convolution, fully_connected or matmul over a channel count that is no multiple of 16.  Its own kernel gathers the
// operand in the pieces that divide the channels, down to single bytes; with every row padded to whole chunks the kernels of
// aligned operands take it, the packed weights spread to match, with zeros against the padding.
static bool matchPadded(const DescriptorView &v, const Tuning &tuning, uint32_t first, Step *s) {
    const DescOp &g = v.ops[first];
    if (g.kind != kKindIgemm || g.loader != kLoaderGather || g.in1.space != kSpaceNone || g.weights.space != kSpaceConst || g.C % 16 == 0) return false;
    const bool pointwise = g.KH == 1 && g.KW == 1 && g.SH == 1 && g.SW == 1 && g.PT == 0 && g.PL == 0 && g.OH == g.H && g.OW == g.W;
    const int64_t C = g.C, Cp = roundUp(C, 16), taps = (int64_t)g.KH * g.KW, rows = (int64_t)g.N * g.H * g.W, K = taps * Cp, N = g.Nn;
    if (g.K != taps * C || g.Kp < g.K || g.PT < 0 || g.PL < 0 || rows * Cp >= (1LL << 31) || K >= (1LL << 31)) return false;
    if (tuning.padRows == 0) return false;
    DescOp op = g;
    op.C = (int32_t)Cp;
    op.K = (int32_t)K;
    op.gran = 16;
    op.loader = pointwise ? kLoaderDense : kLoaderWindow;
    // the (bias, scale) arrays were padded for the record's own tile
    auto padded = [&](int64_t Kp, int64_t Np) {
        op.Kp = (int32_t)Kp;
        op.Np = (int32_t)Np;
        for (const DescRef *r : {&g.bias, &g.scale}) {
            if (r->space != kSpaceConst || v.consts[r->index].size - r->offset < (uint64_t)Np * 4) return false;
        }
        return true;
    };
    // rows as they are: the weights of a window of one pixel serve without being spread (igemmRoute)
    const bool pays = paddingPays(g, rows, Cp, K), asIs = (pays || taps > 1) && padded(roundUp(K, 32), roundUp(N, 32)) && asIsBetter(v, tuning, g, op);
    if (!asIs) {
        if (tuning.padRows == 2 || (tuning.padRows < 0 && !pays)) return false;
        int64_t Kp = Cp, Np = N;
        if (pointwise && g.M <= kFcSkinnyMaxRows) {
            op.kind = kKindFcSkinny;
            op.loader = g.loader;
        } else {
            uint32_t variant;
            if (thip_gemm_tile_choice((int32_t)op.loader, g.M, N, K, Cp, g.out_dtype, 0, &variant, nullptr, 0) != THIP_OK) return false;
            if (variant == kIgemmStream && g.out.offset % 16 != 0) return false;  // it stores whole 16-byte pieces; the record's kernel any
            const IgemmTile &t = igemmTile(variant);
            Kp = roundUp(K, t.bk);
            Np = roundUp(N, t.bn);
            op.variant = variant;
        }
        if (!padded(Kp, Np)) return false;
        op.in0 = DescRef{kSpacePlan, 0, 0};
    }
    const uint64_t weightBytes = (uint64_t)roundUp((int64_t)op.Np * op.Kp, 256);
    s->constants.assign(weightBytes + 128, 0);
    const uint8_t *w = v.blob + v.header.data_offset + v.consts[g.weights.index].offset + g.weights.offset;
    for (int64_t n = 0; n < N; n++) {
        for (int64_t tap = 0; tap < taps; tap++) memcpy(&s->constants[(size_t)(n * op.Kp + tap * Cp)], w + n * g.Kp + tap * C, (size_t)C);
    }
    memset(&s->constants[weightBytes], g.input_zp, 128);  // what a tap outside the image reads
    op.weights = DescRef{kSpacePlan, 1, 0};
    op.table = op.kind == kKindIgemm && op.loader == kLoaderWindow ? DescRef{kSpacePlan, 1, weightBytes} : DescRef{kSpaceNone, 0, 0};
    s->kind = kStepPadded;
    s->first = first;
    s->count = 1;
    s->rows = rows;
    s->from = (int32_t)C;
    s->to = (int32_t)Cp;
    s->asIs = asIs;
    s->copies = !asIs || (g.in0.space == kSpaceBinding && g.out.space == kSpaceBinding && g.in0.index != g.out.index);
    s->op = op;
    return true;
}

// A grouped linear or small matmul as a phase of dec_chain, but for what the exchange carries; false: not one of its.
static bool chainPhase(const DescriptorView &v, const DescOp &op, int workgroups, const std::function<ChainRef(const DescRef &)> &at, ChainPhase *out) {
    ChainPhase t;
    memset(&t, 0, sizeof(t));
    auto asFloat = [](int32_t bits) {
        float f;
        memcpy(&f, &bits, 4);
        return f;
    };
    t.xTag = t.resTag = t.outTag[0] = t.outTag[1] = t.outTag[2] = t.addTag = -1;
    t.lo = asFloat(op.output_min);
    t.hi = asFloat(op.output_max);
    t.M = op.M;
    t.K = op.K;
    t.split = t.nmat = t.nseg = 1;
    if (op.kind == kKindDecLinear) {
        DecLinearExt x;
        memcpy(&x, v.blob + v.header.data_offset + v.consts[op.table.index].offset + op.table.offset, sizeof(x));
        if (op.M > kChainMaxRows || (long long)op.M * op.K > (1 << 20)) return false;
        if (asFloat(op.bias0) != -INFINITY || asFloat(op.scale0) != INFINITY) return false;  // a clamped expansion
        const bool pair = (op.w1 & kDecPair) != 0;
        long long tiles = 0;
        for (int m = 0; m < op.w0; m++) {
            if (x.weights[m].space != kSpaceConst || x.bias[m].space != kSpaceConst) return false;
            t.w[m] = at(x.weights[m]);
            t.bias[m] = at(x.bias[m]);
            t.out[m] = x.out[m].space == kSpaceNone ? 0 : at(x.out[m]);
            t.N[m] = x.N[m];
            if (m == 0 || !pair) tiles += x.N[m] / 16;
        }
        if (tiles > (1 << 20)) return false;
        t.x = at(op.in0);
        t.nseg = op.w0;
        t.nmat = pair ? 2 : 1;
        t.slotBytes = decSlotBytes(x.has_qbias != 0);
        // two jobs share a tile where K has more units than a workgroup has waves and the chip has workgroups to spare
        t.split = op.K / 128 > kChainWaves && tiles * 2 <= workgroups ? 2 : 1;
        t.units = (op.K / 128 + t.split - 1) / t.split;
        t.perPass = kChainResults / t.nmat;
        t.jobs = (int32_t)tiles * t.split;
        t.addMode = (op.w1 & kDecAddResidual) ? (op.w1 & kDecResFirst ? 3 : 1) : (op.w1 & kDecAddPair) ? 2 : 0;
        if (t.addMode) {
            if (t.addMode != 2) t.res = at(x.res);
            t.addOut = at(x.add_out);
            t.aw0 = asFloat((int32_t)((uint32_t)x.aw0 << 16));
            t.aw1 = asFloat((int32_t)((uint32_t)x.aw1 << 16));
            t.abias = asFloat(x.abias);
            t.alo = asFloat(x.alo);
            t.ahi = asFloat(x.ahi);
        }
    } else if (op.kind == kKindDecMatmul) {
        const long long tiles = ((long long)op.Nn + 15) / 16, rows = (long long)op.M * op.K;
        if (op.M > kChainMaxHeads || tiles * op.TB > (1 << 20) || rows > (1 << 20) || (long long)(op.w1 ? 1 : op.TB) * op.Nn * op.K >= (1 << 30)) return false;
        t.x = at(op.in0);
        t.w[0] = at(op.weights);
        t.out[0] = at(op.out);
        t.N[0] = op.Nn;
        t.tiles = (int32_t)tiles;
        t.jobs = (int32_t)tiles * op.TB;
        t.units = (op.K + 63) / 64;
        // the rows of every job of a pass are in LDS at once
        t.perPass = (int32_t)std::max<long long>(1, std::min<long long>(kChainResults, 32 * 1024 / (rows * 2)));
        t.aStride = op.w0 ? 0 : op.M * op.K;
        t.wStride = op.w1 ? 0 : op.Nn * op.K;
        t.outStride = op.M * op.Nn;
        t.wBytes = (uint32_t)((uint64_t)(op.w1 ? 1 : op.TB) * op.Nn * op.K * 2);
        t.bias0 = asFloat(op.bias0);
        const FastDiv d = makeFastDiv((uint32_t)t.tiles);
        t.tilesMul = d.mul;
        t.tilesShift = d.shift;
    } else {
        return false;
    }
    const FastDiv units = makeFastDiv((uint32_t)t.units), items = makeFastDiv((uint32_t)(t.M * 16 / t.split));
    t.unitsMul = units.mul;
    t.unitsShift = units.shift;
    t.itemsMul = items.mul;
    t.itemsShift = items.shift;
    *out = t;
    return true;
}

// What a phase reads that the chain makes is read from the exchange, so it has to be one result of a phase before it, or a part of one.  Weights and
// caches are fetched ahead: none of them is written in the chain.  Everything else that is read is there when the launch starts, and written by no phase.
Chain layoutChain(const DescriptorView &v, uint32_t first, uint32_t most, int workgroups, const std::function<ChainRef(const DescRef &)> &at) {
    struct Range {
        DescRef ref;
        uint64_t bytes;
        int32_t *tag;    // of a result: where the exchange has it
        ChainRef *plain;
    };
    Chain chain;
    std::vector<Range> reads, writes;
    auto meet = [](const Range &a, const Range &b) { return sameBuffer(a.ref, b.ref) && a.ref.offset < b.ref.offset + b.bytes && b.ref.offset < a.ref.offset + a.bytes; };
    auto anyMeets = [&](const std::vector<Range> &list, const Range &r) {
        for (const Range &x : list) {
            if (meet(x, r)) return true;
        }
        return false;
    };
    chain.phases.reserve(kChainMaxPhases);  // tags point into it
    most = std::min(most, std::min<uint32_t>(kChainMaxPhases, v.header.op_count - first));
    for (uint32_t n = 0; n < most; n++) {
        const DescOp &op = v.ops[first + n];
        ChainPhase t;
        if (!chainPhase(v, op, workgroups, at, &t)) break;
        chain.phases.push_back(t);
        ChainPhase &p = chain.phases.back();
        std::vector<Range> in, ahead, out;
        if (p.slotBytes == 0) {
            in.push_back({op.in0, (uint64_t)(op.w0 ? 1 : op.TB) * op.M * op.K * 2, &p.xTag, nullptr});
            ahead.push_back({op.weights, (uint64_t)(op.w1 ? 1 : op.TB) * op.Nn * op.K * 2, nullptr, nullptr});
            out.push_back({op.out, (uint64_t)op.TB * op.M * op.Nn * 2, &p.outTag[0], &p.out[0]});
        } else {
            DecLinearExt x;
            memcpy(&x, v.blob + v.header.data_offset + v.consts[op.table.index].offset + op.table.offset, sizeof(x));
            in.push_back({op.in0, (uint64_t)op.M * op.K * 2, &p.xTag, nullptr});
            if (p.addMode & 1) in.push_back({x.res, (uint64_t)op.M * x.N[0] * 2, &p.resTag, nullptr});
            if (p.addMode) out.push_back({x.add_out, (uint64_t)op.M * x.N[0] * 2, &p.addTag, &p.addOut});
            for (int m = 0; m < op.w0; m++) {
                if (x.out[m].space != kSpaceNone) out.push_back({x.out[m], (uint64_t)op.M * x.N[m] * 2, &p.outTag[m], &p.out[m]});
            }
        }
        bool fits = true;
        std::vector<int32_t *> exchanged;  // results that this phase is the first to read
        for (const Range &r : ahead) fits = fits && !anyMeets(writes, r);
        for (const Range &r : out) fits = fits && !anyMeets(writes, r) && !anyMeets(reads, r) && !anyMeets(in, r) && !anyMeets(ahead, r);
        uint64_t words = chain.exchangeWords;
        for (const Range &r : in) {
            if (!fits || !anyMeets(writes, r)) continue;
            const Range *source = nullptr;
            for (const Range &x : writes) {
                if (sameBuffer(x.ref, r.ref) && x.ref.offset <= r.ref.offset && r.ref.offset + r.bytes <= x.ref.offset + x.bytes) source = &x;
            }
            // 16-byte loads
            if (!source || (r.ref.offset - source->ref.offset) % 8 != 0 || words + source->bytes / 2 + 32 > (1u << 30)) {
                fits = false;
                break;
            }
            if (*source->tag < 0) {
                *source->tag = (int32_t)words;
                exchanged.push_back(source->tag);
                words = (uint64_t)roundUp((int64_t)(words + source->bytes / 2), 32);
            }
            *r.tag = *source->tag + (int32_t)((r.ref.offset - source->ref.offset) / 2);
        }
        const int32_t x = std::max(chain.xRoom, (p.slotBytes == 0 ? p.perPass : 1) * p.M * p.K * 2), red = std::max(chain.redRoom, kChainResults * kChainWaves * p.M * 64);
        if (!fits || (int64_t)(n + 1) * (int64_t)sizeof(ChainPhase) + x + red > kChainLds) {
            for (int32_t *tag : exchanged) *tag = -1;
            chain.phases.pop_back();
            break;
        }
        p.start = n == 0 ? 0 : (chain.phases[n - 1].start + chain.phases[n - 1].jobs) % workgroups;
        chain.exchangeWords = words;
        chain.xRoom = x;
        chain.redRoom = red;
        reads.insert(reads.end(), in.begin(), in.end());
        reads.insert(reads.end(), ahead.begin(), ahead.end());
        writes.insert(writes.end(), out.begin(), out.end());
    }
    // an intermediate that only the chain reads is nowhere but in the exchange
    const uint32_t count = (uint32_t)chain.phases.size();
    const std::vector<uint32_t> all = tempUses(v, 0, v.header.op_count), here = tempUses(v, first, count);
    for (const Range &r : writes) {
        if (r.ref.space == kSpaceTemp && *r.tag >= 0 && all[r.ref.index] == here[r.ref.index]) *r.plain = 0;
    }
    return chain;
}

// Whether a chain is ahead of its records' own launches.  It saves 1.5 us a phase: what a launch costs beyond handing its results to the next
// one, and the weights that are fetched meanwhile.  It costs 5 us once, and 0.25 us for every 1000 elements that a workgroup brings as input rows: it
// reads them as dwords past its L2, where a launch reads 16-bit elements through it.  Fitted to 60 decoder steps of one to four rows, 1 to 6 layers,
// hidden 256 .. 2048, one by one / as a chain, us:
//   taken   26 layers, 1152, 6912, one row 843 / 616, 4 layers of it 117 / 88 (two rows 117 / 99), 4 x 1664, 640, one row 104 / 65,
//           5 x 256, 8064, three rows 136 / 109, 1 x 1152, 6912 34.0 / 30.5
//   left    6 x 384, 6272, four rows 169 / 180, 4 x 2048, 8192, 8 heads of 256 on 2048 positions, one row 182 / 185
static bool chainPays(const Chain &chain, int workgroups) {
    double gain = -6;  // 1 us more than measured: boxes differ
    for (const ChainPhase &t : chain.phases) {
        const int jobs = (t.jobs + workgroups - 1) / workgroups;
        gain += 1.54 - 0.253e-3 * (double)t.M * t.K * (t.slotBytes == 0 ? std::min(jobs, (int)t.perPass) : 1);
    }
    return gain > 0;
}

static bool matchDecChain(const DescriptorView &v, const Tuning &tuning, uint32_t first, Step *s) {
    if (tuning.decChain == 0 || v.header.binding_count > 64) return false;
    if (v.ops[first].kind != kKindDecLinear && v.ops[first].kind != kKindDecMatmul) return false;
    const Chain chain = layoutChain(v, first, v.header.op_count, kChainWorkgroups, [](const DescRef &) { return (ChainRef)1; });
    if (chain.phases.size() < (size_t)kChainMinPhases || (tuning.decChain < 0 && !chainPays(chain, kChainWorkgroups))) return false;
    s->kind = kStepDecChain;
    s->first = first;
    s->count = (uint32_t)chain.phases.size();
    return true;
}

// The kernel that is ahead for a GEMM-shaped record.  In place a record has its own, whose tiles take 64 columns or more: those of igemm_direct_i8 take 32,
// and others of the same rows may still be reading where one stores.
static IgemmRoute igemmRoute(const DescriptorView &v, const Tuning &tuning, const DescOp &op) {
    const IgemmArgs a = igemmArgs(v, op, [&](const DescRef &r) { return plannedAt(v, r); });
    if (op.loader == kLoaderGather && op.KH == 1 && op.KW == 1 && zerosBehindRows(v, op) && asIsBetter(v, tuning, op, op)) return kIgemmDirect;
    return !inPlace(op) && igemmDirectBetter(a) ? kIgemmDirect : convPatchBetter(a) ? kIgemmPatch : !tuning.noK128 && igemmWideBetter(a, op.variant) ? kIgemmWide : kIgemmOwnTile;
}

// A replay starts about 5 us later than a launch behind another, and costs the host 12 - 20 us in place of 3 per launch.  Launches that
// stream weights take the device longer than that, so the host stays ahead and the program is faster launch by launch, by the same 5 us
// whatever its length: decoder steps of 7, 13, 25 and 37 launches 25.6 / 30.8, 48.1 / 53.7, 91.6 / 97.6 and 135.4 / 141.1 us (one by
// one / replayed; 2.4 MB of weights each), chains of 6, 18 and 30 convolutions 30.4 / 33.9, 92.4 / 97.2 and 154.2 / 158.9 (370 KB).
// At 48 convolutions that is 1.5 % (246.6 / 250.5) for 123 us of the host's time in place of 17: beyond 40 launches the replay is taken
// again.  An image network's 37 launches (95 KB each) take 141 us replayed, 151 one by one.
bool replayPays(size_t launches, uint64_t constantBytes) {
    const bool streams = constantBytes >= launches * 256 * 1024;
    return launches >= 4 && !(streams && launches <= 40);
}

// Intermediates between grouped linears (and the result of a small matmul that is one's input) are laid out in blocks of 32 columns, which the
// reader's loads bring in whole lines, where every record that touches one knows how: one writes all of it, the others take it as rows or as the
// residual sum.  Up to kDecLdsRows rows come through LDS, as they lie.  us, row by row / in blocks, 32 rows: 1152 -> 2 x 6912 11.0 / 9.9, 6912 -> 1152
// 10.6 / 9.3, 1152 -> 1536 5.0 / 4.8, 1024 -> 1152 4.9 / 4.7.
static void blockRows(const DescriptorView &v, std::vector<Step> &steps) {
    struct Use {
        size_t step;
        int32_t bit;
    };
    struct Temp {
        bool other = false;  // somebody takes it as it is
        int writers = 0, readers = 0;
        int64_t rows = 0, columns = 0;
        std::vector<Use> uses;
    };
    std::vector<Temp> temps(v.header.temp_count);
    auto asIs = [&](const DescRef &r) {
        if (r.space == kSpaceTemp) temps[r.index].other = true;
    };
    for (size_t i = 0; i < steps.size(); i++) {
        auto use = [&](const DescRef &r, int64_t rows, int64_t columns, int32_t bit, bool writes, bool reads) {
            if (r.space != kSpaceTemp) return;
            Temp &t = temps[r.index];
            if (t.uses.empty()) {
                t.rows = rows;
                t.columns = columns;
            }
            if (r.offset != 0 || t.rows != rows || t.columns != columns || rows <= kDecLdsRows || columns % 32 != 0) t.other = true;
            t.writers += writes;
            t.readers += reads;
            t.uses.push_back({i, bit});
        };
        const Step &s = steps[i];
        for (uint32_t n = s.first; n < s.first + s.count; n++) {
            const DescOp &op = v.ops[n];
            DecLinearExt x;
            if (op.kind == kKindDecLinear) memcpy(&x, v.blob + v.header.data_offset + v.consts[op.table.index].offset + op.table.offset, sizeof(x));
            if (s.kind == kStepRecord && op.kind == kKindDecLinear) {
                for (const DescRef *r : {&op.in1, &op.weights, &op.bias, &op.scale, &op.table}) asIs(*r);
                if (!sameRef(op.out, x.add_out) && !sameRef(op.out, x.out[0])) asIs(op.out);  // names one of them again
                use(op.in0, op.M, op.K, kDecBlockedX, false, true);
                for (int m = 0; m < op.w0 && m < kDecMaxSegments; m++) use(x.out[m], op.M, x.N[m], kDecBlockedOut << m, true, false);
                if (op.w1 & kDecAddResidual) use(x.res, op.M, x.N[0], kDecBlockedRes, false, false);
                if (op.w1 & (kDecAddResidual | kDecAddPair)) use(x.add_out, op.M, x.N[0], kDecBlockedAdd, true, false);
            } else if (s.kind == kStepRecord && op.kind == kKindDecMatmul) {
                for (const DescRef *r : {&op.in0, &op.in1, &op.weights, &op.bias, &op.scale, &op.table}) asIs(*r);
                use(op.out, op.TB, (int64_t)op.M * op.Nn, kDecBlockedOut, true, false);
                if (op.Nn % 4 != 0 || (int64_t)op.TB * op.M * op.Nn >= (1LL << 31)) asIs(op.out);
            } else {
                for (const DescRef *r : {&op.in0, &op.in1, &op.weights, &op.bias, &op.scale, &op.table, &op.out}) asIs(*r);
                if (op.kind == kKindDecLinear) {
                    for (int m = 0; m < kDecMaxSegments; m++) {
                        for (const DescRef *r : {&x.weights[m], &x.bias[m], &x.out[m]}) asIs(*r);
                    }
                    asIs(x.res);
                    asIs(x.add_out);
                }
            }
        }
    }
    for (const Temp &t : temps) {
        if (t.other || t.writers != 1 || t.readers < 1) continue;
        for (const Use &u : t.uses) steps[u.step].blocked |= u.bit;
    }
}

bool writesWhatItReads(const DescriptorView &v, const Step &s, uint8_t *const *bp) {
    const DescRef &out = v.ops[s.first + s.count - 1].out;
    if (out.space != kSpaceBinding) return false;
    const uint8_t *begin = bp[out.index], *end = begin + v.bindings[out.index].size;
    for (uint32_t i = s.first; i < s.first + s.count; i++) {
        const DescOp &op = v.ops[i];
        for (const DescRef *r : {&op.in0, &op.in1, &op.weights, &op.bias, &op.scale, &op.table}) {
            if (r->space == kSpaceBinding && r->index != out.index && bp[r->index] < end && begin < bp[r->index] + v.bindings[r->index].size) return true;
        }
    }
    return false;
}

std::vector<Step> planSteps(const DescriptorView &v, const Tuning &tuning) {
    const bool plain = tuning.plainRecords;
    const std::vector<uint32_t> uses = tempUses(v, 0, v.header.op_count);
    std::vector<Step> steps;
    for (uint32_t i = 0; i < v.header.op_count;) {
        Step s{};
        if (plain || (!matchDecChain(v, tuning, i, &s) && !matchExpandDw(v, tuning, uses, i, &s) && !matchMatmulRt(v, uses, i, &s) && !matchPadded(v, tuning, i, &s))) {
            s.kind = kStepRecord;
            s.first = i;
            s.count = 1;
        }
        const DescOp *op = s.kind == kStepRecord ? &v.ops[i] : s.kind == kStepPadded ? &s.op : nullptr;
        if (s.kind == kStepExpandDw && s.count == 3) op = &v.ops[i + 2];
        s.route = plain || !op || op->kind != kKindIgemm ? kIgemmOwnTile : s.kind == kStepPadded && s.asIs ? kIgemmDirect : igemmRoute(v, tuning, *op);
        i += s.count;
        steps.push_back(std::move(s));
    }
    if (!plain) blockRows(v, steps);
    return steps;
}

}  // namespace thip
