// The weights that dec_chain loads, for the chains that the library plans for a serialised program (the file in argv[1]): every dword that may be
// fetched lies inside its operand, and every dword that a product needs is fetched.  A load is held against the bytes of its unit by the offset
// of the lane, and the uniform offset beside it may count or not: both readings are checked.  Prints "phases linear matmul shared odd": how many there
// are, of which kind, with two jobs to a tile, and of these with an odd number of k-blocks.
#include <stdio.h>

#include <vector>

#include "thip_plan.h"

using namespace thip;

static int phase, job;
static int fail(const char *what, int unit, int lane, long long at) {
    printf("phase %d, job %d, unit %d, lane %d: %s (%lld)\n", phase, job, unit, lane, what, at);
    return 1;
}

// `count` dwords from `lane` + `uniform` on of a unit that starts at `unit` of an operand, `bytes` of it to be read.
static int load(uint64_t operand, uint64_t unit, uint32_t bytes, uint32_t lane, uint32_t uniform, int count, bool needed, int u, int l) {
    for (int d = 0; d < count; d++) {
        const uint32_t own = lane + 4 * d;
        const uint64_t at = unit + own + uniform;
        // where the uniform offset counts it is taken off the bytes, which may pass below zero
        const bool counted = (uint64_t)own + 4 <= (uint32_t)(bytes - uniform), plain = (uint64_t)own + 4 <= bytes;
        if ((counted || plain) && at + 4 > operand) return fail("fetched behind the operand", u, l, (long long)at);
        if (needed && !(counted && plain)) return fail("needed and not fetched", u, l, (long long)at);
    }
    return 0;
}

int main(int argc, char **argv) {
    if (argc != 2) return 2;
    std::vector<uint8_t> blob;
    FILE *f = fopen(argv[1], "rb");
    if (!f) return 2;
    fseek(f, 0, SEEK_END);
    blob.resize((size_t)ftell(f));
    rewind(f);
    const size_t n = fread(blob.data(), 1, blob.size(), f);
    fclose(f);
    DescHeader h;
    if (n != blob.size() || validateWhole(blob.data(), blob.size(), &h) != THIP_OK) return 3;
    const DescriptorView v{blob.data(), h, (const DescOp *)(blob.data() + h.ops_offset), (const DescBinding *)(blob.data() + h.bindings_offset),
                           (const DescTemp *)(blob.data() + h.temps_offset), (const DescConst *)(blob.data() + h.consts_offset)};
    int linear = 0, matmul = 0, shared = 0, odd = 0, phases = 0;
    for (const Step &s : planSteps(v, tuningFromEnvironment())) {
        if (s.kind != kStepDecChain) continue;
        const Chain chain = layoutChain(v, s.first, s.count, kChainWorkgroups, [](const DescRef &) { return (ChainRef)1; });
        for (const ChainPhase &t : chain.phases) {
            phase = phases++;
            const int blocks = t.K >> 7;
            (t.slotBytes ? linear : matmul)++;
            shared += t.split > 1;
            odd += t.split > 1 && blocks % 2 != 0;
            for (job = 0; job < t.jobs; job++) {
                for (int mat = 0; mat < t.nmat; mat++) {
                    ChainUnits u;
                    ChainTile tile{0, 0};
                    uint64_t operand = t.wBytes;
                    int batch = 0;
                    if (t.slotBytes) {
                        tile = chainTile(t.split == 1 ? job : job >> 1, t.nmat, t.nseg, t.N[0] >> 4, t.N[1] >> 4);
                        const int matrix = t.nmat > 1 ? mat : tile.seg;
                        if (tile.tile < 0 || tile.tile * 16 >= t.N[matrix]) return fail("a tile beyond its matrix", tile.seg, tile.tile, 0);
                        operand = decWeightBytes(t.N[matrix], t.K, t.slotBytes > kDecSlotBytes);
                        u = chainLinearUnits(t.K, t.slotBytes, t.split, tile.tile, t.split == 1 ? 0 : job & 1);
                    } else {
                        batch = job / t.tiles;
                        tile.tile = job % t.tiles;
                        u = chainMatmulUnits(t.K, t.wBytes, t.wStride, batch, tile.tile);
                    }
                    for (int unit = 0; unit < t.units; unit++) {
                        const uint32_t at = (uint32_t)unit * u.unitBytes, bytes = u.bytes - at;
                        const uint64_t where = u.first + at;
                        if (at >= u.bytes) return fail("nothing of a unit is there", unit, 0, at);
                        for (int lane = 0; lane < 64; lane++) {
                            const int c = lane & 15, g = lane >> 4;
                            if (t.slotBytes) {
                                const ChainLane l = chainLinearLane(c, g, t.slotBytes, t.split);
                                const int block = t.split == 1 ? unit : unit * 2 + (c >> 3), column = t.split == 1 ? c : (job & 1) * 8 + (c & 7);
                                const bool needed = block < blocks;
                                // what is loaded is this column's of this k-block
                                const uint64_t slot = (uint64_t)(tile.tile * blocks + block) * t.slotBytes;
                                if (where + l.weights != slot + (uint64_t)(g * 16 + column) * 16) return fail("other weights", unit, lane, 0);
                                if (where + l.scales + u.scales != slot + 2048 + column * 4) return fail("another scale", unit, lane, 0);
                                if (load(operand, where, bytes, l.weights, 0, 4, needed, unit, lane) || load(operand, where, bytes, l.weights + u.half, 0, 4, needed, unit, lane) ||
                                    load(operand, where, bytes, l.scales, u.scales, 1, needed, unit, lane) || load(operand, where, bytes, l.scales, u.scales + u.bias, 1, needed, unit, lane)) return 1;
                            } else {
                                const ChainLane l = chainMatmulLane(c, g, t.K);
                                const int column = tile.tile * 16 + c, k = unit * 64 + 8 * g;
                                const bool real = column < t.N[0];
                                if (where + l.weights != ((uint64_t)batch * t.wStride + (uint64_t)column * t.K + k) * 2) return fail("other weights", unit, lane, 0);
                                if (load(operand, where, bytes, l.weights, 0, 4, real && k < t.K, unit, lane) || load(operand, where, bytes, l.weights + u.half, 0, 4, real && k + 32 < t.K, unit, lane) ||
                                    load(operand, where, bytes, l.scales, u.scales, 1, false, unit, lane)) return 1;
                            }
                        }
                    }
                }
            }
        }
    }
    printf("%d %d %d %d %d\n", phases, linear, matmul, shared, odd);
    return 0;
}
