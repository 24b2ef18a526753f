// The launch of many PCG iterations (k_cg_persist.hip) for a system, by its
// sizes and by what the device holds.  Host code without HIP.
#pragma once

#include <cstdint>

namespace nlhip {

constexpr int kPersistSmall = 1, kPersistRows = 2, kPersistBlocks = 3;

struct PersistShape {
    int kind = 0;          // 0: not for this system
    uint32_t wgs = 0;      // workgroups that take part
    uint32_t stride = 1;   // every stride-th workgroup of the grid does
    uint32_t threads = 0;  // per workgroup
};

// P logical workgroups of sps tiles and chunk rows each, with at most one tile
// per wavefront:
//   small  up to 128 rows each, in two wavefronts
//   rows   up to 256 rows each
//   blocks up to 512 rows (256 row pairs) each
// Logical workgroups per physical one: fewer, larger workgroups wait for one
// another faster until their gathers queue up (us per iteration with 1, 2, 4:
// 8 k rows 5.6, 5.3, 5.9; 24 k 8.9, 6.0, 5.6; with 1, 2: 100 k 14.9, 9.3).  On
// one XCD (stride) up to 16 workgroups: 4.0 against 4.3 at 1,150 rows; the
// gathers of more of them crowd its L2 (8 k rows 7.0 against 5.3).
inline PersistShape persist_shape(bool blk, uint32_t P, uint32_t sps, uint32_t chunk,
                                  uint32_t num_xcd) {
    PersistShape s;
    uint32_t subs = 2;
    if (P == 0) return s;
    if (!blk && sps <= 2 && chunk <= 128 && P <= 256) {
        s.kind = kPersistSmall;
        if (P > 128) subs = 4;
        if (P <= 32) s.stride = num_xcd;
        s.threads = 128 * subs;
    } else if (sps <= 4 && chunk <= (blk ? 512u : 256u)) {
        s.kind = blk ? kPersistBlocks : kPersistRows;
        s.threads = 256 * subs;
    }
    s.wgs = (P + subs - 1) / subs;
    return s;
}

// The workgroups wait for one another, so all of them have to be resident:
// one on each of cus compute units (the registers of FP64 kernels hold no
// second), with a stride on those of one XCD of num_xcd (a partition of the
// device with fewer units takes the others too).
inline PersistShape persist_resident(PersistShape s, uint32_t cus, uint32_t num_xcd) {
    if (s.stride > 1 && s.wgs > cus / num_xcd) s.stride = 1;
    if (s.wgs > cus) s.kind = 0;
    return s;
}

}  // namespace nlhip
