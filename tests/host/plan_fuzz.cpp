// The launches of mutated descriptors (files argv[2] ...; argv[1]: mutants of each): whatever the validation lets through is planned, with
// the sanitizers watching.
#include <stdio.h>
#include <stdlib.h>

#include <random>
#include <vector>

#include "thip_plan.h"

using namespace thip;

int main(int argc, char **argv) {
    if (argc < 3) return 2;
    std::mt19937 rng(20);
    long planned = 0, records = 0;
    for (int a = 2; a < argc; a++) {
        FILE *f = fopen(argv[a], "rb");
        if (!f) return 2;
        fseek(f, 0, SEEK_END);
        const size_t size = (size_t)ftell(f);
        rewind(f);
        std::vector<uint64_t> whole((size + 7) / 8);
        const size_t n = fread(whole.data(), 1, size, f);
        fclose(f);
        if (n != size) return 2;
        for (int it = 0; it < atoi(argv[1]); it++) {
            std::vector<uint64_t> copy(whole);
            uint8_t *p = (uint8_t *)copy.data();
            const size_t tables = (size_t)((const DescHeader *)p)->data_offset;  // records and tables lie below
            for (int k = it ? 1 + (int)(rng() % 3) : 0; k > 0; k--) {
                static const uint32_t words[] = {0, 1, 2, 3, 7, 16, 32, 100, 0x7fffffff, 0xffffffff};
                const size_t at = sizeof(DescHeader) + rng() % (tables - sizeof(DescHeader));
                if (rng() % 2) p[at] ^= (uint8_t)(1u << (rng() % 8));
                else memcpy(p + (at & ~(size_t)3), &words[rng() % 10], 4);
            }
            DescHeader h;
            if (validateWhole(p, size, &h) != THIP_OK) continue;
            const DescriptorView v{p, h, (const DescOp *)(p + h.ops_offset), (const DescBinding *)(p + h.bindings_offset), (const DescTemp *)(p + h.temps_offset),
                                   (const DescConst *)(p + h.consts_offset)};
            Tuning t;
            t.padRows = it % 2 ? 1 : -1;
            uint32_t next = 0;
            for (const Step &s : planSteps(v, t)) {  // every record belongs to one step, in order
                if (s.first != next || s.count == 0) return 1;
                next += s.count;
            }
            if (next != h.op_count) return 1;
            planned++;
            records += next;
        }
    }
    printf("planned %ld programs of %ld records\n", planned, records);
    return 0;
}
