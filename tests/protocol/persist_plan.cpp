// Every launch of many iterations that persist_plan.h chooses has no more
// workgroups than the device has compute units; prints the sizes swept, or the
// first violation.
#include <cstdio>
#include <initializer_list>

#include "persist_plan.h"

using namespace nlhip;

int main() {
    const uint32_t xcd = 8;
    long swept = 0, taken = 0;
    for (uint32_t cus : {0u, 1u, 4u, 8u, 16u, 31u, 32u, 38u, 64u, 128u, 224u, 256u, 304u})
        for (int blk = 0; blk < 2; ++blk)
            for (uint32_t sps = 1; sps <= 5; ++sps)
                for (uint32_t chunk : {1u, 64u, 128u, 129u, 256u, 257u, 512u, 513u})
                    for (uint32_t P = 0; P <= 1300; ++P) {
                        const PersistShape s = persist_resident(
                            persist_shape(blk != 0, P, sps, chunk, xcd), cus, xcd);
                        ++swept;
                        if (!s.kind) continue;
                        ++taken;
                        const uint32_t units = s.stride > 1 ? cus / xcd : cus;
                        const uint32_t subs = s.threads / (s.kind == kPersistSmall ? 128 : 256);
                        if (s.wgs == 0 || s.wgs > units || s.threads > 512 || subs * s.wgs < P) {
                            std::printf("cus %u blk %d sps %u chunk %u P %u: kind %d, %u "
                                        "workgroups of %u threads, stride %u\n",
                                        cus, blk, sps, chunk, P, s.kind, s.wgs, s.threads,
                                        s.stride);
                            return 1;
                        }
                    }
    std::printf("swept %ld taken %ld\n", swept, taken);
    return 0;
}
