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

// Entries (2x2 blocks) of the longest row (row pair) it takes: 16 (8) are in
// registers, and the rest of a row is fetched by its lane one after another in
// every iteration, 0.2 to 0.3 us each, while everyone waits.  The launches
// lose little to one long row (their tiles' entries are read side by side), but
// few workgroups, as small systems have, take long to stream long rows.
// us per iteration, three launches against this:
//   24 k rows, one of 41 entries among 5: 12.8, 12.0; of 53 13.0, 14.4; of 505
//   20.4, 149; all of 49 22.9, 20.9, of 65 27.4, 31.0
//   8 k, all of 49 22.9, 14.9, of 257 179, 77.5; 1 k, one of 53 14.3, 11.2, of
//   101 15.3, 21.6, all of 257 186, 76.5
//   100 k, one of 41 15.2, 14.0, of 53 15.6, 16.5; all of 21 19.8, 12.3, of 25
//   21.7, 17.5, of 33 23.8, 28.5
//   100 k pairs, one of 37 blocks 19.6, 18.1, of 69 20.7, 26.3; all of 11 22.5,
//   18.1, of 13 24.2, 24.3
inline uint32_t persist_longest(const PersistShape& s, uint64_t nnz, uint32_t n) {
    const uint32_t mean = uint32_t((nnz + n - 1) / n);  // entries of a row
    if (s.kind == kPersistSmall) return 40 + (s.threads <= 256 ? mean : mean / 4);
    if (mean <= 16) return 40;
    return s.kind == kPersistBlocks ? 12 : 24;
}

}  // namespace nlhip
