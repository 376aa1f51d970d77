// The launches that the library plans for a serialised program (the file in argv[1]), one a line: what it is, its records, and the
// kernel of a GEMM-shaped record; then whether dispatches on buffers that come back are replayed as a graph.  Further arguments: where the
// bindings lie, for a line to say that its launch would write what it reads.
#include <stdio.h>
#include <stdlib.h>

#include <vector>

#include "thip_plan.h"

using namespace thip;

int main(int argc, char **argv) {
    if (argc < 2) return 2;
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
    if (argc > 2 && (uint32_t)argc != 2 + h.binding_count) return 2;
    std::vector<uint8_t *> bindings;
    for (int i = 2; i < argc; i++) bindings.push_back((uint8_t *)(uintptr_t)strtoull(argv[i], nullptr, 0));
    const std::vector<Step> steps = planSteps(v, tuningFromEnvironment());
    const char *kinds[] = {"record", "ir_expand_dw_i8", "padded", "igemm_rt_i8", "dec_chain"}, *routes[] = {"", " igemm_direct_i8", " conv_patch_i8", " igemm_dense_k128_i8"};
    for (const Step &s : steps) {
        printf("%s %u %u%s", s.kind == kStepExpandDw && s.count == 3 ? "ir_block_i8" : kinds[s.kind], s.first, s.count, routes[s.route]);
        // the input's rows in no whole 16-byte chunks, read all the same
        if (s.asIs || (s.kind == kStepRecord && s.route == kIgemmDirect && v.ops[s.first].loader == kLoaderGather)) printf(" as it is");
        if (s.blocked) printf(" blocked %d", s.blocked);
        if (!bindings.empty() && writesWhatItReads(v, s, bindings.data())) printf(" shared");
        puts("");
    }
    puts(replayPays(steps.size(), h.total_size - h.data_offset) ? "replayed" : "one by one");
    return 0;
}
