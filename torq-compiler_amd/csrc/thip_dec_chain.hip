// gfx950 kernel of a decoder's step: a run of grouped linears and small matmuls as one launch of one workgroup per CU.
#include "thip_dec_chain.h"
#include "thip_kernels_common.h"

#include <stddef.h>

namespace thip {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kChainThreads = (kChainWaves + kChainPollers + 1) * 64;

// A pointer into global memory: addresses that come out of the table are generic to the compiler, and a generic load also counts as one of LDS.
template <typename T>
__device__ __forceinline__ T globalLoad(const void *p) {
    return *(const __attribute__((address_space(1))) T *)(uintptr_t)p;
}
// Memory that other workgroups of the launch read or write: past this XCD's L2 (the compiler's agent scope).
template <typename T>
__device__ __forceinline__ T sharedLoad(const T *p) {
    return __hip_atomic_load((const __attribute__((address_space(1))) T *)(uintptr_t)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void sharedStore(T *p, T v) {
    __hip_atomic_store((__attribute__((address_space(1))) T *)(uintptr_t)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// A barrier of the workgroup for data in LDS; loads from memory stay in flight across it.
__device__ __forceinline__ void ldsBarrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory"); }

// A lane holds a dword of the phase's entry: fields are read across lanes, without a trip to LDS each.
#define PHASE_INT(entry, field) __builtin_amdgcn_readlane(entry, (int)(offsetof(ChainPhase, field) / 4))
#define PHASE_FLOAT(entry, field) __builtin_bit_cast(float, PHASE_INT(entry, field))
#define PHASE_DIV(entry, name) FastDiv{(uint32_t)PHASE_INT(entry, name##Mul), (uint32_t)PHASE_INT(entry, name##Shift), 0}
#define PHASE_REF(entry, field, index) phaseRef(entry, (int)(offsetof(ChainPhase, field) / 4) + 2 * (index))
__device__ __forceinline__ ChainRef phaseRef(int entry, int at) {
    return (ChainRef)(uint32_t)__builtin_amdgcn_readlane(entry, at) | (ChainRef)(uint32_t)__builtin_amdgcn_readlane(entry, at + 1) << 32;
}
__device__ __forceinline__ uint8_t *chainAddress(const DecChainArgs &p, ChainRef r) {
    const uint32_t binding = (uint32_t)(r >> 56);
    const uint64_t offset = r & 0xffffffffffffffull;
    return binding ? p.bindings[binding - 1] + offset : (uint8_t *)offset;
}

// What every wave of a workgroup knows.
struct ChainGroup {
    const int *table;           // LDS: the entries
    const v2i *jobsOf;          // LDS: jobs and first workgroup of each phase once more, one behind the other
    int8_t *xs;                 // LDS: the input rows
    float *red;                 // LDS: partial sums
    int *say;                   // LDS: 0: this workgroup gives up, written between the end of a pass and the start of the next and read between start and end;
                                // 1: launches done, then whether any workgroup gave up; 2: it is the last one; 3: zero
    uint32_t *exchange;
    uint32_t tag;               // of this launch, in the upper half
    int count, wg, G;
    FastDiv byGrid;
    bool alone;                 // this workgroup makes everything by itself
    int lane, wave;
};

// Where a wave is among the units of its workgroup; uniform but for `entry`.
struct ChainWalk {
    int entry;
    int phase, pass, block;        // kChainRing units a wave of a pass are a block
    int job, jobsHere, units;      // of the phase: the workgroup's first job, and how many; units of a result
    int nmat, perPass;
    FastDiv byUnits;
    int all, blocks;               // of the pass: units of its results, blocks (the same for all waves)
    int results;                   // of the pass: tiles of a matrix
    int u;                         // this wave's next unit of the pass, of `all`
};

// The first job of the workgroup, if the phase has as many.
__device__ __forceinline__ int chainPlace(const ChainGroup &q, int start) {
    const int place = q.wg - start;
    return q.alone ? 0 : place < 0 ? place + q.G : place;
}
// The first phase from `phase` on that the workgroup has jobs of.
__device__ __forceinline__ int chainNextPhase(const ChainGroup &q, int phase) {
    for (; phase < q.count; phase += 64) {
        const v2i jobs = phase + q.lane < q.count ? q.jobsOf[phase + q.lane] : v2i{0, 0};
        const unsigned long long mine = __ballot(jobs[0] > chainPlace(q, jobs[1]));
        if (mine) return phase + (int)__builtin_ctzll(mine);
    }
    return q.count;
}
__device__ __forceinline__ void chainEnterPass(const ChainGroup &q, ChainWalk &w) {
    const int jobs = w.jobsHere - w.pass * w.perPass;
    w.results = (jobs < w.perPass ? jobs : w.perPass) * w.nmat;
    w.all = w.results * w.units;
    w.blocks = (int)((uint32_t)(w.all + kChainWaves * kChainRing - 1) / (uint32_t)(kChainWaves * kChainRing));
    w.block = 0;
    w.u = q.wave;
}
__device__ __forceinline__ void chainEnterPhase(const ChainGroup &q, ChainWalk &w, int phase) {
    w.phase = phase;
    if (phase >= q.count) return;
    w.entry = q.table[phase * 64 + q.lane];
    const int jobs = PHASE_INT(w.entry, jobs);
    w.job = chainPlace(q, PHASE_INT(w.entry, start));
    w.jobsHere = q.alone ? jobs : (int)fastDiv((uint32_t)(jobs - w.job + q.G - 1), q.byGrid);
    w.perPass = PHASE_INT(w.entry, perPass);
    w.units = PHASE_INT(w.entry, units);
    w.byUnits = PHASE_DIV(w.entry, units);
    w.nmat = PHASE_INT(w.entry, nmat);
    w.pass = 0;
    chainEnterPass(q, w);
}
__device__ __forceinline__ bool chainLastPass(const ChainWalk &w) { return (w.pass + 1) * w.perPass >= w.jobsHere; }
__device__ __forceinline__ void chainNextBlock(const ChainGroup &q, ChainWalk &w) {
    if (++w.block < w.blocks) {
        w.u += kChainRing * kChainWaves;
    } else if (!chainLastPass(w)) {
        w.pass++;
        chainEnterPass(q, w);
    } else {
        chainEnterPhase(q, w, chainNextPhase(q, w.phase + 1));
    }
}
__device__ __forceinline__ int chainJob(const ChainGroup &q, const ChainWalk &w, int index) { return w.job + (w.pass * w.perPass + index) * q.G; }
__device__ __forceinline__ int chainBatch(const ChainWalk &w, int job) { return (int)fastDiv((uint32_t)job, PHASE_DIV(w.entry, tiles)); }

// One more look at the clock of a wait that began at `start`; true: the workgroup gives up.
__device__ __forceinline__ bool chainTired(const DecChainArgs &p, const ChainGroup &q, uint64_t start, uint32_t polls) {
    if (q.alone || (p.waitTicks > 0 && (polls & 63) != 63)) return false;
    if (p.waitTicks > 0 && sharedLoad(p.sync + 32) == 0 && __builtin_readsteadycounter() - start <= p.waitTicks) return false;
    if (q.lane == 0) sharedStore(p.sync + 32, 1u);
    return true;
}

// A unit of weights in registers.
struct ChainSlot {
    v4i p0, p1;
    float sc, bi;
};
// Where the weights of a pass lie (see ChainUnits).  Lane r: the first unit of result r, the bytes that may be read from there on, and its
// scales; then what all units have in common.
struct ChainWeights {
    uint32_t lo, hi, bytes, scales;
    ChainLane lane;
    uint32_t unitBytes, half, bias;  // uniform
};
__device__ __forceinline__ ChainWeights chainWeights(const DecChainArgs &p, const ChainGroup &q, const ChainWalk &w) {
    const int c = q.lane & 15, g = q.lane >> 4, K = PHASE_INT(w.entry, K), slotBytes = PHASE_INT(w.entry, slotBytes);
    const int result = q.lane < w.results ? q.lane : 0, job = chainJob(q, w, result >> (w.nmat - 1));
    ChainWeights t;
    ChainUnits u;
    uint64_t base;
    if (slotBytes == 0) {  // a matmul
        const int b = chainBatch(w, job);
        base = (uint64_t)(uintptr_t)chainAddress(p, PHASE_REF(w.entry, w, 0));
        u = chainMatmulUnits(K, (uint32_t)PHASE_INT(w.entry, wBytes), PHASE_INT(w.entry, wStride), b, job - b * PHASE_INT(w.entry, tiles));
        t.lane = chainMatmulLane(c, g, K);
    } else {
        const int split = PHASE_INT(w.entry, split);
        const ChainTile tile = chainTile(split == 1 ? job : job >> 1, w.nmat, PHASE_INT(w.entry, nseg), PHASE_INT(w.entry, N[0]) >> 4, PHASE_INT(w.entry, N[1]) >> 4);
        const int matrix = w.nmat > 1 ? result & 1 : tile.seg;
        const v2i first = *(const v2i *)(q.table + w.phase * 64 + (int)(offsetof(ChainPhase, w) / 4) + 2 * matrix);  // a constant: an address
        base = (uint64_t)(uint32_t)first[0] | (uint64_t)(uint32_t)first[1] << 32;
        u = chainLinearUnits(K, slotBytes, split, tile.tile, split == 1 ? 0 : job & 1);
        t.lane = chainLinearLane(c, g, slotBytes, split);
    }
    base += u.first;
    t.lo = (uint32_t)base;
    t.hi = (uint32_t)(base >> 32);
    t.bytes = u.bytes;
    t.scales = u.scales;
    t.unitBytes = u.unitBytes;
    t.half = u.half;
    t.bias = u.bias;
    return t;
}
// Unit `u` of `w`'s pass into a slot.  All of a slot is loaded or nothing: behind a branch around a single register of it the compiler
// waits for the load at once.
__device__ __forceinline__ void chainLoad(const ChainWalk &w, const ChainWeights &t, int u, ChainSlot &s) {
    if (u >= w.all) return;
    const int result = (int)fastDiv((uint32_t)u, w.byUnits), unit = u - result * w.units;
    const uint32_t at = (uint32_t)unit * (uint32_t)__builtin_amdgcn_readfirstlane((int)t.unitBytes);
    const uint64_t base = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)t.lo, result) | (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)t.hi, result) << 32) + at;
    const uint32_t bytes = (uint32_t)__builtin_amdgcn_readlane((int)t.bytes, result);
    const int scales = __builtin_amdgcn_readlane((int)t.scales, result);
    // A unit's first row exists.  The second half of a matmul's unit may not: it is told apart by the lane's own offset, which is always held against
    // `bytes`.  The uniform offset of the scales need not be (a scale that is not there lies behind weights that are not).
    const auto all = __builtin_amdgcn_make_buffer_rsrc((void *)base, 0, bytes - at, 0x00027000);
    s.p0 = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(all, (int)t.lane.weights, 0, 0));
    s.p1 = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(all, (int)t.lane.weights + __builtin_amdgcn_readfirstlane((int)t.half), 0, 0));
    s.sc = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(all, (int)t.lane.scales, scales, 0));
    s.bi = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(all, (int)t.lane.scales, scales + __builtin_amdgcn_readfirstlane((int)t.bias), 0));
}

// This wave's share of a result, to LDS.
__device__ __forceinline__ void chainLeave(const ChainGroup &q, int at, bool wanted, v4f &acc) {
    if (wanted) ((v4f *)q.red)[at] = acc;
    acc = v4f{0.0f, 0.0f, 0.0f, 0.0f};
}
// The rows of a block are there, the partial sums in LDS used up; true: the workgroup gives up (to be acted on before the next barrier).
__device__ __forceinline__ int chainStart(const ChainGroup &q, const ChainWalk &w) {
    if (w.block > 0) return 0;
    ldsBarrier();
    return q.say[0];
}

// A block of a linear.  The weights become operands while the rows are still on their way: two or three waves of a SIMD share its
// vector pipe, and 128 x 16 weights are some 350 cycles of it.
__device__ __forceinline__ int chainLinear(const ChainGroup &q, const ChainWalk &w, const ChainSlot (&slots)[kChainRing], v4f &acc) {
    const int c = q.lane & 15, g = q.lane >> 4;
    const int M = PHASE_INT(w.entry, M), K = PHASE_INT(w.entry, K), split = PHASE_INT(w.entry, split), all = w.all;
    const bool biases = PHASE_INT(w.entry, slotBytes) > kDecSlotBytes;
    // of the 16 x 16 products the two blocks on the diagonal are wanted where two jobs share a tile
    const bool wanted = split == 1 ? c < M : (c & 7) < M && (g >> 1) == (c >> 3);
    const int place = split == 1 ? c * 4 + g : ((c >> 3) * M + (c & 7)) * 2 + (g & 1), m = split == 1 ? c : c & 7;
    const int row = ((m < M ? m : 0) * K + 8 * g) * 2;
    v4i operand[kChainRing][4];
    int x[kChainRing], red[kChainRing];  // where the rows lie, and the sum behind the unit (< 0: it goes on with the next one)
#pragma unroll
    for (int s = 0; s < kChainRing; s++) {
        const int u = w.u + s * kChainWaves, next = u + kChainWaves;
        if (u < all) {
            const int result = (int)fastDiv((uint32_t)u, w.byUnits), unit = u - result * w.units;
            red[s] = next >= all || next >= (result + 1) * w.units ? (result * kChainWaves + q.wave) * M * 4 : -1;
            float sc = slots[s].sc, bi = biases ? slots[s].bi : 0.0f;
            x[s] = row + unit * 256;
            if (split > 1) {
                const int block = unit * 2 + (c >> 3);
                x[s] = row + block * 256;
                if (block >= (K >> 7)) {
                    sc = bi = 0.0f;
                    x[s] = -1;  // the rows end before
                }
            }
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const v4i d = j < 2 ? slots[s].p0 : slots[s].p1;
                int o[4];
                expandQ8<false>(d[(2 * j) & 3], sc, bi, 0.0f, 0.0f, &o[0], &o[1]);
                expandQ8<false>(d[(2 * j + 1) & 3], sc, bi, 0.0f, 0.0f, &o[2], &o[3]);
                operand[s][j] = v4i{o[0], o[1], o[2], o[3]};
            }
        }
        __builtin_amdgcn_sched_barrier(0);  // one unit after the other: all at once they don't fit the registers
    }
    const int givenUp = chainStart(q, w);
#pragma unroll
    for (int s = 0; s < kChainRing; s++) {
        if (w.u + s * kChainWaves < all) {
            const bool beyond = x[s] < 0;
            const int8_t *rows = q.xs + (beyond ? 0 : x[s]);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                v4i v = *(const v4i *)(rows + 64 * j);
                if (beyond) v = v4i{0, 0, 0, 0};
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, operand[s][j]), __builtin_bit_cast(v8bf, v), acc, 0, 0, 0);
            }
            if (red[s] >= 0) chainLeave(q, red[s] + place, wanted, acc);
        }
    }
    return givenUp;
}

// A block of a matmul.
__device__ __forceinline__ int chainMatmul(const ChainGroup &q, const ChainWalk &w, const ChainSlot (&slots)[kChainRing], v4f &acc) {
    const int c = q.lane & 15, g = q.lane >> 4;
    const int M = PHASE_INT(w.entry, M), K = PHASE_INT(w.entry, K), all = w.all;
    const int givenUp = chainStart(q, w);
#pragma unroll
    for (int s = 0; s < kChainRing; s++) {
        const int u = w.u + s * kChainWaves, next = u + kChainWaves;
        if (u < all) {
            const int result = (int)fastDiv((uint32_t)u, w.byUnits), unit = u - result * w.units, k = unit * 64 + 8 * g;
            const int8_t *rows = q.xs + (result * M * K + (c < M ? c : 0) * K) * 2;
#pragma unroll
            for (int j = 0; j < 2; j++) {
                // beyond K a row holds the next one or anything: zeros on both sides
                const int in = k + 32 * j < K ? -1 : 0;
                v4i v = *(const v4i *)(rows + ((k + 32 * j) & in) * 2), d = j ? slots[s].p1 : slots[s].p0;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    v[e] &= in;
                    d[e] &= in;
                }
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, d), __builtin_bit_cast(v8bf, v), acc, 0, 0, 0);
            }
            if (next >= all || next >= (result + 1) * w.units) chainLeave(q, (result * kChainWaves + q.wave) * M * 4 + c * 4 + g, c < M, acc);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    return givenUp;
}

// The waves that multiply.
__device__ __forceinline__ void chainMultiply(const DecChainArgs &p, const ChainGroup &q, int firstPhase) {
    ChainSlot slots[kChainRing];
    ChainWalk ahead;
    ChainWeights weights;
    chainEnterPhase(q, ahead, firstPhase);
    if (firstPhase < q.count) {
        weights = chainWeights(p, q, ahead);
#pragma unroll
        for (int s = 0; s < kChainRing; s++) chainLoad(ahead, weights, ahead.u + s * kChainWaves, slots[s]);
    }
    v4f acc = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    while (ahead.phase < q.count) {
        const ChainWalk now = ahead;
        chainNextBlock(q, ahead);
        if (ahead.phase >= q.count) ahead.all = 0;
        else if (ahead.block == 0) weights = chainWeights(p, q, ahead);
        const int givenUp = PHASE_INT(now.entry, slotBytes) == 0 ? chainMatmul(q, now, slots, acc) : chainLinear(q, now, slots, acc);
        if (__builtin_amdgcn_readfirstlane(givenUp)) break;
        if (now.block + 1 == now.blocks) ldsBarrier();  // the partial sums are in LDS
        ChainSlot fresh[kChainRing];  // apart from the old ones, which are used up: what is not loaded is undefined
#pragma unroll
        for (int s = 0; s < kChainRing; s++) {
            chainLoad(ahead, weights, ahead.u + s * kChainWaves, fresh[s]);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int s = 0; s < kChainRing; s++) slots[s] = fresh[s];
    }
}

// kCount times four elements of the exchange a lane, kChainStep apart, once they are all there, to LDS; false: the workgroup gives up.
constexpr int kChainStep = kChainPollers * 256;
template <int kCount>
__device__ __forceinline__ bool chainBringSome(const DecChainArgs &p, const ChainGroup &q, const uint32_t *src, int e, int elements, int8_t *dst, uint64_t start) {
    const auto all = __builtin_amdgcn_make_buffer_rsrc((void *)src, 0, (uint32_t)elements * 4u, 0x00027000);  // beyond: zeros, without a fetch
    // what is there is not asked for again: the last look is short
    v4i v[kCount];
    bool there[kCount];
#pragma unroll
    for (int i = 0; i < kCount; i++) there[i] = e + i * kChainStep >= elements;
    for (uint32_t polls = 0;; polls++) {
#pragma unroll
        for (int i = 0; i < kCount; i++) {
            if (!there[i]) v[i] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(all, (e + i * kChainStep) * 4, 0, (int)(0x80000000u | 16u)));  // volatile, sc1
        }
        bool whole = true;
#pragma unroll
        for (int i = 0; i < kCount; i++) {
            const uint32_t d = ((uint32_t)v[i][0] ^ q.tag) | ((uint32_t)v[i][1] ^ q.tag) | ((uint32_t)v[i][2] ^ q.tag) | ((uint32_t)v[i][3] ^ q.tag);
            there[i] = there[i] || d < 0x10000u;
            whole = whole && there[i];
        }
        if (__all(whole) && (q.alone || p.waitTicks > 0)) break;
        if (chainTired(p, q, start, polls)) return false;
        if (polls > 16) __builtin_amdgcn_s_sleep(2);
    }
#pragma unroll
    for (int i = 0; i < kCount; i++) {
        if (e + i * kChainStep < elements) {
            *(v2i *)(dst + (e + i * kChainStep) * 2) = v2i{(int)__builtin_amdgcn_perm((uint32_t)v[i][1], (uint32_t)v[i][0], 0x05040100u), (int)__builtin_amdgcn_perm((uint32_t)v[i][3], (uint32_t)v[i][2], 0x05040100u)};
        }
    }
    return true;
}

// The waves that bring the input rows.
__device__ __forceinline__ void chainBring(const DecChainArgs &p, const ChainGroup &q, int firstPhase) {
    const int from = (q.wave - kChainWaves) * 256, first4 = from + q.lane * 4;
    bool late = false;
    ChainWalk w;
    for (chainEnterPhase(q, w, firstPhase); w.phase < q.count; chainEnterPhase(q, w, chainNextPhase(q, w.phase + 1))) {
        const int xTag = PHASE_INT(w.entry, xTag), elements = PHASE_INT(w.entry, M) * PHASE_INT(w.entry, K), aStride = PHASE_INT(w.entry, aStride);
        const bool matmul = PHASE_INT(w.entry, slotBytes) == 0;
        const uint8_t *x = xTag < 0 ? chainAddress(p, PHASE_REF(w.entry, x, 0)) : (const uint8_t *)(q.exchange + xTag);
        for (;;) {
            const int pieces = matmul ? w.results : w.pass == 0 ? 1 : 0;
            for (int j = 0; j < pieces; j++) {
                const size_t skip = matmul ? (size_t)chainBatch(w, chainJob(q, w, j)) * (size_t)aStride : 0;
                int8_t *dst = q.xs + j * elements * 2;
                if (xTag < 0) {
                    for (int e = first4 * 2; e < elements; e += kChainStep * 2) *(v4i *)(dst + e * 2) = globalLoad<v4i>(x + (skip + (size_t)e) * 2);
                } else {
                    const uint64_t start = __builtin_readsteadycounter();
                    // as many loads at once as there is to bring: one behind the other they are a trip to memory each
                    const uint32_t *src = (const uint32_t *)x + skip;
                    for (int e = 0; e + from < elements && !late; e += 16 * kChainStep) {
                        const int left = elements - from - e;
                        late = !(left <= 2 * kChainStep   ? chainBringSome<2>(p, q, src, first4 + e, elements, dst, start)
                                 : left <= 4 * kChainStep ? chainBringSome<4>(p, q, src, first4 + e, elements, dst, start)
                                 : left <= 8 * kChainStep ? chainBringSome<8>(p, q, src, first4 + e, elements, dst, start)
                                                          : chainBringSome<16>(p, q, src, first4 + e, elements, dst, start));
                    }
                }
            }
            if (late && q.lane == 0) q.say[0] = 1;
            ldsBarrier();
            if (__builtin_amdgcn_readfirstlane(q.say[0])) return;
            ldsBarrier();
            if (chainLastPass(w)) break;
            w.pass++;
            chainEnterPass(q, w);
        }
    }
}

// An element of a pass: where its partial sums lie and where it goes.
struct ChainItem {
    int part[2][kChainWaves];   // floats from the partial sums on
    int tagged[2], addTagged;   // words of the exchange; < 0: nowhere
    uint32_t where;             // elements into a result
    uint16_t *plain[2];         // null: nowhere
    float bias[2];
    uint32_t res;
    bool real;
};
// What the elements of a phase have in common.
struct ChainOut {
    int M, split, nseg, addMode, shares, perJob, zeroAt;
    bool matmul, resFirst;
    float lo, hi, aw0, aw1, abias, alo, ahi;
    FastDiv byItems;
    uint16_t *addOut;
    int addTag, resTag;
};
__device__ __forceinline__ void globalStore16(uint16_t *p, uint16_t v) { *(__attribute__((address_space(1))) uint16_t *)(uintptr_t)p = v; }

__device__ __forceinline__ ChainItem chainItem(const DecChainArgs &p, const ChainGroup &q, const ChainWalk &w, const ChainOut &o, int item, bool real, bool &late) {
    ChainItem it;
    const int jl = (int)fastDiv((uint32_t)item, o.byItems), rest = item - jl * o.perJob;
    const int m = o.split == 1 ? rest >> 4 : rest >> 3, column = o.split == 1 ? rest & 15 : rest & 7, job = chainJob(q, w, jl);
    int seg = 0, N = PHASE_INT(w.entry, N[0]);
    it.bias[0] = it.bias[1] = 0.0f;
    it.res = 0;
    it.real = real;
    if (o.matmul) {
        const int b = chainBatch(w, job), n = (job - b * PHASE_INT(w.entry, tiles)) * 16 + column;
        it.real = real && n < N;
        it.where = (uint32_t)b * (uint32_t)PHASE_INT(w.entry, outStride) + (uint32_t)(m * N + n);
        it.bias[0] = PHASE_FLOAT(w.entry, bias0);
    } else {
        const int N1 = PHASE_INT(w.entry, N[1]), N2 = PHASE_INT(w.entry, N[2]);
        const ChainTile t = chainTile(o.split == 1 ? job : job >> 1, w.nmat, o.nseg, N >> 4, N1 >> 4);
        seg = t.seg;
        N = seg == 0 ? N : seg == 1 ? N1 : N2;
        const int n = t.tile * 16 + (o.split == 1 ? 0 : (job & 1) * 8) + column;
        it.where = (uint32_t)(m * N + n);
        // constants: addresses
        const ChainRef b0 = PHASE_REF(w.entry, bias, 0), b1 = PHASE_REF(w.entry, bias, 1), b2 = PHASE_REF(w.entry, bias, 2);
        it.bias[0] = globalLoad<float>((const float *)(seg == 0 ? b0 : seg == 1 ? b1 : b2) + n);
        if (w.nmat == 2) it.bias[1] = globalLoad<float>((const float *)b1 + n);
    }
#pragma unroll
    for (int mat = 0; mat < 2; mat++) {
        const int result = jl * w.nmat + (mat < w.nmat ? mat : 0);
        int from = result * w.units;
        from -= (int)((uint32_t)from / kChainWaves) * kChainWaves;
        const int base = result * kChainWaves * o.M * 16 + rest;
#pragma unroll
        for (int i = 0; i < kChainWaves; i++) {
            it.part[mat][i] = i < o.shares ? base + from * o.M * 16 : o.zeroAt;
            from = from + 1 == kChainWaves ? 0 : from + 1;
        }
    }
    {
        auto optional = [&](ChainRef r) { return r ? (uint64_t)(uintptr_t)chainAddress(p, r) : 0; };
        const int t0 = PHASE_INT(w.entry, outTag[0]), t1 = PHASE_INT(w.entry, outTag[1]), t2 = PHASE_INT(w.entry, outTag[2]);
        const uint64_t p0 = optional(PHASE_REF(w.entry, out, 0)), p1 = optional(PHASE_REF(w.entry, out, 1)), p2 = optional(PHASE_REF(w.entry, out, 2));
        const int t = seg == 0 ? t0 : seg == 1 ? t1 : t2;
        it.tagged[0] = t < 0 ? -1 : t + (int)it.where;
        it.tagged[1] = w.nmat < 2 || t1 < 0 ? -1 : t1 + (int)it.where;
        it.plain[0] = (uint16_t *)(uintptr_t)(seg == 0 ? p0 : seg == 1 ? p1 : p2);
        it.plain[1] = w.nmat < 2 ? nullptr : (uint16_t *)(uintptr_t)p1;
    }
    it.addTagged = o.addTag < 0 ? -1 : o.addTag + (int)it.where;
    if (o.addMode == 1) {
        if (o.resTag < 0) {
            it.res = (uint32_t)globalLoad<uint16_t>((const uint16_t *)chainAddress(p, PHASE_REF(w.entry, res, 0)) + it.where);
        } else {
            // the other operand of the add, once it is there
            const uint32_t *at = q.exchange + (uint32_t)o.resTag + it.where;
            const uint64_t start = __builtin_readsteadycounter();
            it.res = sharedLoad(at);
            for (uint32_t polls = 0; __any(it.real && (it.res ^ q.tag) >= 0x10000u); polls++) {
                it.res = sharedLoad(at);
                if (chainTired(p, q, start, polls)) {
                    late = true;
                    break;
                }
            }
        }
    }
    if (late) it.real = false;  // nothing wrong is handed on
    return it;
}

__device__ __forceinline__ void chainStore(const ChainGroup &q, const ChainWalk &w, const ChainOut &o, const ChainItem &it) {
    // all reads at once: one after the other they are a trip to LDS each
    float part[2][kChainWaves], half[2][kChainWaves], sum[2] = {0.0f, 0.0f};
#pragma unroll
    for (int mat = 0; mat < 2; mat++) {
        if (mat < w.nmat) {
#pragma unroll
            for (int i = 0; i < kChainWaves; i++) part[mat][i] = q.red[it.part[mat][i]];
            if (o.split > 1) {
#pragma unroll
                for (int i = 0; i < kChainWaves; i++) half[mat][i] = q.red[i < o.shares ? it.part[mat][i] + o.perJob : o.zeroAt];
            }
        }
    }
#pragma unroll
    for (int mat = 0; mat < 2; mat++) {
        if (mat < w.nmat) {
            if (o.split > 1) {
#pragma unroll
                for (int i = 0; i < kChainWaves; i++) part[mat][i] += half[mat][i];
            }
#pragma unroll
            for (int i = 0; i < kChainWaves; i++) sum[mat] += part[mat][i];
        }
    }
    uint16_t y[2];
#pragma unroll
    for (int mat = 0; mat < 2; mat++) {
        const float t0 = sum[mat] + it.bias[mat];
        y[mat] = bf16Bits(t0 < o.lo ? o.lo : (t0 > o.hi ? o.hi : t0));
    }
    if (!it.real) return;
    if (o.addMode) {
        const uint16_t r = (uint16_t)it.res;
        const uint16_t a = o.addMode == 2 ? y[0] : o.resFirst ? r : y[0], b = o.addMode == 2 ? y[1] : o.resFirst ? y[0] : r;
        const uint16_t z = addBf16One(a, b, o.aw0, o.aw1, o.abias, o.alo, o.ahi);
        if (it.addTagged >= 0) sharedStore(q.exchange + it.addTagged, q.tag | z);
        if (o.addOut) globalStore16(o.addOut + it.where, z);
    }
    if (it.tagged[0] >= 0) sharedStore(q.exchange + it.tagged[0], q.tag | y[0]);
    if (it.plain[0]) globalStore16(it.plain[0] + it.where, y[0]);
    if (it.tagged[1] >= 0) sharedStore(q.exchange + it.tagged[1], q.tag | y[1]);
    if (it.plain[1]) globalStore16(it.plain[1] + it.where, y[1]);
}

// The wave that adds up and stores.
__device__ __forceinline__ void chainFinish(const DecChainArgs &p, const ChainGroup &q, int firstPhase) {
    bool late = false;
    ChainWalk w;
    for (chainEnterPhase(q, w, firstPhase); w.phase < q.count; chainEnterPhase(q, w, chainNextPhase(q, w.phase + 1))) {
        ChainOut o;
        o.M = PHASE_INT(w.entry, M);
        o.split = PHASE_INT(w.entry, split);
        o.nseg = PHASE_INT(w.entry, nseg);
        o.addMode = PHASE_INT(w.entry, addMode);
        o.matmul = PHASE_INT(w.entry, slotBytes) == 0;
        o.resFirst = o.addMode == 3;
        if (o.addMode == 3) o.addMode = 1;
        o.shares = w.units < kChainWaves ? w.units : kChainWaves;
        o.perJob = o.M * 16 / o.split;
        o.zeroAt = (p.redRoom >> 2) + 3;  // say[3]
        o.lo = PHASE_FLOAT(w.entry, lo);
        o.hi = PHASE_FLOAT(w.entry, hi);
        o.aw0 = PHASE_FLOAT(w.entry, aw0);
        o.aw1 = PHASE_FLOAT(w.entry, aw1);
        o.abias = PHASE_FLOAT(w.entry, abias);
        o.alo = PHASE_FLOAT(w.entry, alo);
        o.ahi = PHASE_FLOAT(w.entry, ahi);
        o.byItems = PHASE_DIV(w.entry, items);
        const ChainRef ra = PHASE_REF(w.entry, addOut, 0);
        o.addOut = ra ? (uint16_t *)chainAddress(p, ra) : nullptr;
        o.addTag = PHASE_INT(w.entry, addTag);
        o.resTag = PHASE_INT(w.entry, resTag);
        for (;;) {
            const int items = (w.results >> (w.nmat - 1)) * o.perJob;
            ChainItem it = chainItem(p, q, w, o, q.lane < items ? q.lane : 0, q.lane < items, late);
            if (late && q.lane == 0) q.say[0] = 1;
            ldsBarrier();
            if (__builtin_amdgcn_readfirstlane(q.say[0])) return;
            ldsBarrier();  // the partial sums are in LDS
            chainStore(q, w, o, it);
            for (int item = 64; item < items; item += 64) {
                it = chainItem(p, q, w, o, item + q.lane < items ? item + q.lane : 0, item + q.lane < items, late);
                chainStore(q, w, o, it);
            }
            if (chainLastPass(w)) break;
            w.pass++;
            chainEnterPass(q, w);
        }
    }
}

// ---------------------------------------------------------------------------
// dec_chain: a decoder's step at one to four rows as one launch.  Its phases (a layer: q, k, v; scores; context; output projection and residual;
// gate, up and their sum; down and residual) each read what all workgroups made of the one before.  As launches they cost 3.3 - 4.5 us each
// however little they do: 2.3 us from the end of one to the start of the next, a trip to memory for the rows, and the weights are only asked for then.
//
// One workgroup per CU stays for the whole step.  Results pass through an exchange in memory, a dword for a bf16: a reader sees by the tag next to the value
// that it is there, so handing on costs a store and a load that meet in the memory-side cache (0.9 - 1.3 us for 1024 - 4096 elements,
// 2.0 for 6912) and no barrier.  (A barrier over counters, the writes drained first and the rows read through L2 behind it: 2.2 us and
// 0.8 for the rows.)  Nine waves multiply: they fetch the next block of weights as soon as a block is used up and make it operands (the int8 weights expanded
// to bf16) before its rows are there; two bring rows to LDS; one adds the waves' sums up in LDS and stores.  Each of these keeps its address
// arithmetic out of the time between a row's arrival and its result: with one wave doing the bringing and the adding a phase took 5.2 us in place of 3.5.
// Jobs are dealt on from phase to phase, so that who worked in one has its weights of the next but one in time (26 layers 678 -> 646 us).
//
// Measured, us, one launch per record / this one: 26 layers of hidden 1152, feed-forward 6912, four heads of 256 on 1024 positions, one row,
// with the 262144-column projection behind it 843 / 616 (its bytes at 5.05 TB/s: 207); 4 layers without that 117 / 88, two rows 117 / 99.  What bounds it: of 21 us a
// layer 6 x 1.0 are the exchange, 6 x 0.7 the adding up and storing, 4.0 the products and 6 waits of the gate / up and down phases for weights and their expansion.
// Weights by LDS-DMA two blocks ahead, through LDS: 616 -> 609 there, 72 -> 77 at 512, 2048; the vector pipes are busy as it is.
//
// Workgroups wait for one another, so all must get a CU.  The driver lets no two such launches run at once (ChainTurns); where something else keeps a CU for
// longer than waitTicks, whoever waits gives up, everyone returns, and the last workgroup makes the whole step by itself and tells the host.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kChainThreads) void dec_chain(DecChainArgs p) {
    extern __shared__ __attribute__((aligned(16))) int8_t smem[];
    const int tid = threadIdx.x;
    ChainGroup q;
    int *const table = (int *)smem;
    v2i *const jobsOf = (v2i *)(table + p.count * 64);
    q.table = table;
    q.jobsOf = jobsOf;
    q.xs = (int8_t *)(jobsOf + kChainMaxPhases);
    q.red = (float *)(q.xs + p.xRoom);
    q.say = (int *)(q.xs + p.xRoom + p.redRoom);
    q.exchange = p.sync + kChainSyncHead;
    q.lane = tid & 63;
    q.wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    q.count = p.count;
    q.wg = (int)blockIdx.x;
    q.G = (int)gridDim.x;
    q.byGrid = FastDiv{p.byGridMul, p.byGridShift, 0};
    for (int i = tid; i < p.count * 16; i += kChainThreads) ((v4i *)table)[i] = globalLoad<v4i>((const v4i *)p.phases + i);
    if (tid < p.count) jobsOf[tid] = v2i{globalLoad<int>(&p.phases[tid].jobs), globalLoad<int>(&p.phases[tid].start)};
    if (tid == 0) {
        q.say[0] = q.say[3] = 0;
        q.say[1] = (int)sharedLoad(p.sync);
    }
    ldsBarrier();
    const uint32_t epoch = (uint32_t)__builtin_amdgcn_readfirstlane(q.say[1]);
    for (int attempt = 0;; attempt++) {
        q.alone = attempt > 0;
        q.tag = (2u * epoch + 1u + (uint32_t)attempt) << 16;  // what the first attempt left is none of the second's
        const int firstPhase = chainNextPhase(q, 0);
        if (q.wave < kChainWaves) {
            chainMultiply(p, q, firstPhase);
        } else {
            __builtin_amdgcn_s_setprio(3);  // few instructions, but every workgroup waits for them
            if (q.wave < kChainWaves + kChainPollers) chainBring(p, q, firstPhase);
            else chainFinish(p, q, firstPhase);
        }
        if (attempt > 0) break;
        // The last workgroup to get here ends the launch.  If one gave up, because not all of them got a CU at the same time, it
        // makes everything again by itself.
        waitVmcnt<0>();
        ldsBarrier();
        if (tid == 0) q.say[2] = __hip_atomic_fetch_add(p.sync + 64, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u == gridDim.x;
        ldsBarrier();
        if (!__builtin_amdgcn_readfirstlane(q.say[2])) return;
        if (tid == 0) q.say[1] = (int)sharedLoad(p.sync + 32);
        ldsBarrier();
        const bool again = __builtin_amdgcn_readfirstlane(q.say[1]) != 0;
        if (tid == 0) {
            sharedStore(p.sync, epoch + 1u);
            sharedStore(p.sync + 32, 0u);
            sharedStore(p.sync + 64, 0u);
            // (an argument of the launch would be one more to keep all the way)
            if (again) __hip_atomic_store((uint32_t *)(uintptr_t)globalLoad<uint64_t>(p.sync + kChainTell), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            q.say[0] = 0;
        }
        if (!again) return;
        ldsBarrier();
        q.G = 1;
    }
}

hipError_t launchDecChain(const DecChainArgs &in, int workgroups, const LaunchCtx &ctx) {
    DecChainArgs a = in;
    const FastDiv byGrid = makeFastDiv((uint32_t)workgroups);
    a.byGridMul = byGrid.mul;
    a.byGridShift = byGrid.shift;
    const size_t lds = (size_t)a.count * sizeof(ChainPhase) + 8 * kChainMaxPhases + a.xRoom + a.redRoom + 16;
    if (!a.phases || !a.sync || a.count < 1 || a.count > kChainMaxPhases || workgroups < 1 || lds > 160 * 1024) return hipErrorInvalidValue;
    static std::once_flag once;
    static hipError_t configured = hipSuccess;
    std::call_once(once, [&] { configured = hipFuncSetAttribute((const void *)dec_chain, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024); });
    if (configured != hipSuccess) return configured;
    if (ctx.name) {  // a workgroup per CU: they wait for one another
        int fit = 0;
        const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&fit, dec_chain, kChainThreads, lds);
        if (e != hipSuccess) return e;
        if (fit < 1) return hipErrorInvalidValue;
    }
    THIP_ENQUEUE(ctx, "dec_chain", dec_chain, dim3((unsigned)workgroups), dim3(kChainThreads), lds, a);
    return hipGetLastError();
}

}  // namespace thip
