// A grid-wide barrier whose wait may be given up, over words of device memory
// (k_cg_persist.hip) or of a model of it (tests/protocol/grid_barrier.cpp).
//
// Arrivals are counted per group of workgroups, and the last of a group adds
// one to the root word.  A workgroup whose polls run out sets kPersistFail in
// the root, and only from a value below the target: the bit and the completed
// count exclude one another at every barrier, so all workgroups pass it or
// none does.  (Set whatever the count, the bit could land just behind the last
// arrival: those that had seen the count would go on, the others leave.)
#pragma once

#include <cstdint>

#ifdef __HIPCC__
#define NLHIP_BARRIER_FN __host__ __device__ __forceinline__
#else
#define NLHIP_BARRIER_FN inline
#endif

namespace nlhip {

constexpr uint32_t kPersistFail = 0x80000000u;  // bit of the root: a wait was given up
constexpr uint32_t kPersistLong = 0x40000000u;  // with it: by a workgroup whose rows are too long

// Word: load(), add(v) and cas(expected, desired), which returns the value it
// found, each one atomic access; pause() between polls.
// epoch: 1 for the first barrier over these words, then 2, ...
template <typename Word>
NLHIP_BARRIER_FN void barrier_arrive(Word group, Word root, uint32_t group_size, uint32_t epoch) {
    if (group.add(1u) + 1u == group_size * epoch) root.add(1u);
}

// True when all `ngroups` groups have arrived and no wait was given up.
template <typename Word>
NLHIP_BARRIER_FN bool barrier_wait(Word root, uint32_t ngroups, uint32_t epoch, uint32_t polls) {
    const uint32_t target = ngroups * epoch;
    uint32_t seen = 0;
    for (uint32_t k = 0; k < polls; ++k) {
        seen = root.load();  // with the bit set it is above every target
        if (seen >= target) return !(seen & kPersistFail);
        root.pause();
    }
    while (seen < target) {
        const uint32_t found = root.cas(seen, seen | kPersistFail);
        if (found == seen) return false;
        seen = found;  // an arrival or a bit since: at most one turn per workgroup
    }
    return !(seen & kPersistFail);
}

}  // namespace nlhip
