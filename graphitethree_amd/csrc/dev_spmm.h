// Multi-vector SpMM row engine shared by the multi-right-hand-side PCG
// (k_spmm.hip) and the eigensolver's Chebyshev filter (k_eigen.hip).
#pragma once

#include "dev_common.h"

namespace nlhip {

constexpr int kSpmmU = 8;  // gathers in flight per lane

// Rows of an XCD's blocks [lo, hi) of P: an even share of the m rows.
__device__ __forceinline__ void spmm_xcd_rows(uint32_t m, uint32_t lo, uint32_t hi, uint32_t P,
                                              uint32_t& r0, uint32_t& r1) {
    r0 = uint32_t(uint64_t(m) * lo / P);
    r1 = uint32_t(uint64_t(m) * hi / P);
}

// A lane's V adjacent columns of an interleaved vector (V = 2: an aligned
// pair), loaded and stored as one word.  Stores are non-temporal: the result
// must not push the gathered rows out of the L2.  At every size: with plain
// stores the eigensolver is as fast where its blocks fit the last-level cache
// (88.0 and 88.3 ms at 300^2, 477 and 476 at 500^2) and slower beyond it (925
// and 963 ms at 600^2, 6.18 and 6.35 s at 1000^2), the multi-RHS iteration
// between 5% faster and 2.5% slower without a pattern (us, non-temporal and plain:
// 300^2 x 32 76 and 77, 500^2 x 32 154 and 158, 700^2 x 32 287 and 275, 1000^2 x 32
// 559 and 571, 1500^2 x 32 1281 and 1299).
template <int V, typename T>
struct Lane {
    T v[V];
};
template <int V, bool NT = false, typename T>
__device__ __forceinline__ Lane<V, T> lane_load(const T* p) {
    Lane<V, T> r;
    if constexpr (!NT) {
        __builtin_memcpy(r.v, p, sizeof(T) * V);
    } else if constexpr (V == 2) {
        using V2 = T __attribute__((ext_vector_type(2)));
        const V2 w = __builtin_nontemporal_load(reinterpret_cast<const V2*>(p));
        r.v[0] = w.x;
        r.v[1] = w.y;
    } else {
        r.v[0] = __builtin_nontemporal_load(p);
    }
    return r;
}
template <int V, bool NT = true, typename T>
__device__ __forceinline__ void lane_store(T* p, const T (&v)[V]) {
    if constexpr (!NT) {
        __builtin_memcpy(p, v, sizeof(T) * V);
    } else if constexpr (V == 2) {
        using V2 = T __attribute__((ext_vector_type(2)));
        V2 w;
        w.x = v[0];
        w.y = v[1];
        __builtin_nontemporal_store(w, reinterpret_cast<V2*>(p));
    } else {
        __builtin_nontemporal_store(v[0], p);
    }
}

// Row engine: G lanes per row (V = 1 or 2 adjacent columns each, gathered as
// one copy per entry; G V >= k), 64 / G rows per wavefront and step.  The
// blocks that run on one XCD share an even part of the rows and take its
// steps in turn, so at any time they work on neighbouring rows and the X rows
// that those gather (a stencil's rows i - w .. i + w) stay in that XCD's L2;
// a wavefront's step is short (4 rows at 16 lanes), which keeps that window at
// a megabyte for 256-byte X rows.
//
// A wavefront's rows are one contiguous range of entries: its lanes load them
// coalesced, a step ahead, stage them in the wavefront's own LDS and each
// row's lanes read them back (one address per row: a broadcast) for the
// gathers of X[col * k + j].  No workgroup barrier: the wavefronts of a CU
// drift apart and cover one another's latency.  The row pointers are loaded
// two steps ahead, the next step's entries behind the first gathers (loads
// return in order).
//
// Row sums are left to right with one rounding per product and per add.  For
// each row, the lane with columns j .. j + V - 1 calls pre(row, j) (loads the
// epilogue needs that do not depend on the sums) and then fin(row, j, sums,
// pre value).  Columns with
// done[j] set gather nothing (their sums are not used).  zero_x: X is all
// zeros; the rows' sums are +0 (what the sums would give) and the matrix is
// not read.
//
// Against the engine it replaces (passes of 64 rows staged by the whole
// workgroup between barriers, and row shares rounded up to 64 rows per
// block, which left most XCDs without rows below some 300 k rows):
// the Chebyshev step at 90 k rows and 32 columns 37 -> 20 us, the SpMM of 2.25 M
// rows and 32 columns 498 -> 428 us (1.12 GB fetched where 0.78 are needed,
// 1.64 before; 471 us with plain stores; more wavefronts with fewer registers
// spill: 445 us).  Grids are what is resident: with more workgroups the
// waiting ones come back to rows that have left the L2 (550 us).
template <int G, int V, typename T, typename Pre, typename Fin>
__device__ __forceinline__ void spmm_rows_v(uint32_t m, uint32_t k, uint32_t L,
                                            const uint32_t* __restrict__ rp,
                                            const uint32_t* __restrict__ ci,
                                            const T* __restrict__ val, const T* __restrict__ X,
                                            Pre& pre, Fin& fin, const int32_t* done = nullptr,
                                            bool zero_x = false) {
    static_assert(V == 1 || V == 2, "one or two columns per lane");
    constexpr uint32_t Rw = kWave / G;           // rows per wavefront and step
    constexpr int C = G <= 8 ? 2 : 1;            // staged entries per lane
    constexpr uint32_t kChunk = 64u * C;
    __shared__ uint32_t s_ci[kWavesPerBlock][kChunk];
    __shared__ T s_val[kWavesPerBlock][kChunk];
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint32_t w = uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x / kWave)));
    uint32_t* const sc = s_ci[w];
    T* const sv = s_val[w];
    const uint32_t g = lane / G, jb = (lane % G) * V;
    const bool mine = jb < k;  // the lane owns at least one column
    bool active_col = false;
#pragma unroll
    for (int v = 0; v < V; ++v)
        active_col |= jb + v < k && !(done && done[jb + v]);
    uint32_t lo, hi, r0, r1;
    xcd_block_range(L, gridDim.x, lo, hi);
    spmm_xcd_rows(m, lo, hi, gridDim.x, r0, r1);
    const uint64_t stride = uint64_t(hi - lo) * kWavesPerBlock * Rw;
    uint64_t a = uint64_t(r0) + (uint64_t(L - lo) * kWavesPerBlock + w) * Rw;
    using PV = decltype(pre(0u, 0u));
    if (zero_x) {
        for (; a < r1; a += stride) {
            const uint64_t row = a + g;
            if (row >= r1 || !mine) continue;
            const PV pv = pre(uint32_t(row), jb);
            T z[V];
#pragma unroll
            for (int v = 0; v < V; ++v) z[v] = T(0);
            fin(uint32_t(row), jb, z, pv);
        }
        return;
    }
    auto row_ptrs = [&](uint64_t at, uint32_t& b, uint32_t& e) {
        const uint64_t row = at + g;
        b = rp[row < r1 ? uint32_t(row) : r1];
        e = rp[row + 1 < r1 ? uint32_t(row) + 1u : r1];
    };
    uint32_t cn[C] = {};
    T vn[C] = {};
    auto load = [&](uint32_t j0, uint32_t j1) {  // entries [j0, j0 + kChunk) up to j1
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const uint32_t j = j0 + uint32_t(c) * 64u + lane;
            if (j < j1) {
                cn[c] = ntload(ci + j);
                vn[c] = ntload(val + j);
            }
        }
    };
    if (a >= r1) return;
    uint32_t rb, re, rbn, ren;
    row_ptrs(a, rb, re);
    row_ptrs(a + stride, rbn, ren);
    uint32_t J0 = lane_word(rb, 0), J1 = lane_word(re, kWave - 1);
    load(J0, J1);
    for (;;) {
        const uint32_t row = uint32_t(a) + g;  // a + 64 < 2^32 unless past r1
        const bool in = a + g < r1;
        uint32_t rb2, re2;
        row_ptrs(a + 2 * stride, rb2, re2);
        PV pv{};
        if (in && mine) pv = pre(row, jb);
        T acc[V];
#pragma unroll
        for (int v = 0; v < V; ++v) acc[v] = T(0);
        const uint32_t K0 = lane_word(rbn, 0), K1 = lane_word(ren, kWave - 1);
        for (uint32_t c0 = J0;; c0 += kChunk) {
#pragma unroll
            for (int c = 0; c < C; ++c) {
                sc[c * 64 + lane] = cn[c];
                sv[c * 64 + lane] = vn[c];
            }
            __builtin_amdgcn_wave_barrier();
            const bool last = c0 + kChunk >= J1 || c0 + kChunk < c0;
            const uint32_t b = rb > c0 ? rb - c0 : 0u;
            const uint32_t e = re > c0 ? (re - c0 < kChunk ? re - c0 : kChunk) : 0u;
            // the next entries to load: the rest of this step's, or the next step's
            const uint32_t n0 = last ? K0 : c0 + kChunk, n1 = last ? K1 : J1;
            bool ahead = false;
            for (uint32_t p = b; p < e || !ahead; p += kSpmmU) {
                T xv[kSpmmU][V];
                if (p < e) {
#pragma unroll
                    for (int u = 0; u < kSpmmU; ++u) {
                        const uint32_t q = p + u < e ? p + u : e - 1u;
                        if (active_col) {
                            __builtin_memcpy(xv[u], X + uint64_t(sc[q]) * k + jb, sizeof(T) * V);
                        } else {
#pragma unroll
                            for (int v = 0; v < V; ++v) xv[u][v] = T(0);
                        }
                    }
                }
                if (!ahead) {
                    __builtin_amdgcn_sched_barrier(0);
                    load(n0, n1);
                    __builtin_amdgcn_sched_barrier(0);
                    ahead = true;
                }
                if (p < e) {
#pragma unroll
                    for (int u = 0; u < kSpmmU; ++u)
                        if (p + u < e) {
                            const T av = sv[p + u];
#pragma unroll
                            for (int v = 0; v < V; ++v)
                                acc[v] = add_rn(acc[v], mul_rn(av, xv[u][v]));
                        }
                }
            }
            __builtin_amdgcn_wave_barrier();
            if (last) break;
        }
        if (in && mine) fin(row, jb, acc, pv);
        a += stride;
        if (a >= r1) return;
        rb = rbn;
        re = ren;
        rbn = rb2;
        ren = re2;
        J0 = K0;
        J1 = K1;
    }
}

// ---- stream SpMM for a few right-hand sides --------------------------
//
// For k <= 4 right-hand sides the row engine above leaves lanes idle (4 lanes
// for k = 3).
// This engine streams the matrix as the scalar stream engine does (one row
// per lane, 64-row tiles, a wavefront's nonzeros as one contiguous range in
// chunks of 64E entries, the next chunk's (colind, val) loads issued before
// the current chunk is summed) and gathers the K values X[col*K + j] of every
// entry.  The K products of each entry are staged in LDS and lane l sums
// row l's products column by column, left to right with one rounding per
// product and per add: the sums of spmm_rows, bitwise.  Columns with
// act[j] false sum zeros (their sums are not used).  Block L owns tiles [L*sp, L*sp + sp), one contiguous quarter
// per wavefront; `stage` holds kStage values per wavefront.
//
// Epilogue: pv = epi.pre(row) when the row's tile starts, then
// epi.done(row, sums[K], pv), by the row's lane, rows in order.  zero_x: X
// is all zeros; the sums are +0 (what the sums would give) and the matrix
// is not read.
template <int K, int E, bool D16>
struct MultiStreamEngine {
    using Loads = StreamEngine<E, true, D16>;
    static constexpr uint32_t kStage = 64u * uint32_t(E) * uint32_t(K);

    template <typename T, typename Epi>
    __device__ __forceinline__ static void run_rows(uint32_t R0, uint32_t R1,
                                                    const uint32_t* __restrict__ rp,
                                                    const Cols& cols, const T* __restrict__ val,
                                                    const T* __restrict__ X, const bool (&act)[K],
                                                    T* __restrict__ st, int lane, Epi& epi) {
        constexpr uint32_t C = 64u * E;  // entries per chunk
        const uint32_t ul = uint32_t(lane);
        const uint32_t J1 = __builtin_amdgcn_readfirstlane(rp[R1]);
        uint32_t r0 = R0;
        uint32_t nrows = (R1 - r0) < 64u ? (R1 - r0) : 64u;
        uint32_t tile_end = rp[r0 + nrows];
        uint32_t rb = ul < nrows ? rp[r0 + ul] : tile_end;
        typename Epi::PV pv{};
        if (ul < nrows) pv = epi.pre(r0 + ul);
        uint32_t re = __shfl_down(rb, 1, kWave);
        if (ul + 1 >= nrows) re = tile_end;
        uint32_t base = __builtin_amdgcn_readfirstlane(__shfl(rb, 0, kWave));
        T acc[K];
#pragma unroll
        for (int j = 0; j < K; ++j) acc[j] = T(0);
        uint32_t c[E];
        T a[E];
        if (base < J1) Loads::load_chunk(cols, val, base, J1, lane, c, a);
        while (base < J1) {
            const uint32_t craw = base + C;
            const uint32_t cend = craw < J1 ? craw : J1;
            // each entry's K values as one copy: the widest loads the
            // alignment allows (k = 3 FP64: 16 + 8 bytes; FP32: 12 bytes),
            // so the gather instructions per entry are 1-2 instead of K
            T p[E][K];
#pragma unroll
            for (int e = 0; e < E; ++e)
                __builtin_memcpy(p[e], X + uint64_t(c[e]) * K, sizeof(T) * K);
            // every gather ahead of the prefetch (loads return in order)
            __builtin_amdgcn_sched_barrier(0);
            uint32_t cn[E];
            T an[E];
            Loads::load_chunk(cols, val, craw, J1, lane, cn, an);
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const bool in = base + uint32_t(e) * 64u + ul < J1;
#pragma unroll
                for (int j = 0; j < K; ++j)
                    st[uint32_t(j) * C + uint32_t(e) * 64u + ul] =
                        (in && act[j]) ? mul_rn(a[e], p[e][j]) : T(0);
            }
            __builtin_amdgcn_wave_barrier();
            // consume this chunk; it may complete several tiles
            for (;;) {
                const uint32_t lo = rb > base ? rb : base;
                const uint32_t hi = re < cend ? re : cend;
                for (uint32_t q = lo; q < hi; ++q) {
#pragma unroll
                    for (int j = 0; j < K; ++j) acc[j] = add_rn(acc[j], st[uint32_t(j) * C + q - base]);
                }
                if (tile_end > cend) break;
                if (ul < nrows) epi.done(r0 + ul, acc, pv);
#pragma unroll
                for (int j = 0; j < K; ++j) acc[j] = T(0);
                r0 += 64u;
                if (r0 >= R1) return;
                nrows = (R1 - r0) < 64u ? (R1 - r0) : 64u;
                tile_end = rp[r0 + nrows];
                rb = ul < nrows ? rp[r0 + ul] : tile_end;
                re = __shfl_down(rb, 1, kWave);
                if (ul + 1 >= nrows) re = tile_end;
                if (ul < nrows) pv = epi.pre(r0 + ul);
            }
            __builtin_amdgcn_wave_barrier();
            base = craw;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                c[e] = cn[e];
                a[e] = an[e];
            }
        }
        // tiles left without nonzeros (all their rows are empty)
        for (;;) {
            if (ul < nrows) epi.done(r0 + ul, acc, pv);
            r0 += 64u;
            if (r0 >= R1) return;
            nrows = (R1 - r0) < 64u ? (R1 - r0) : 64u;
            if (ul < nrows) pv = epi.pre(r0 + ul);
        }
    }

    template <typename T, typename Epi>
    __device__ __forceinline__ static void run(uint32_t m, uint32_t sp, uint32_t L,
                                               const uint32_t* __restrict__ rp,
                                               const Cols& cols, const T* __restrict__ val,
                                               const T* __restrict__ X, const bool (&act)[K],
                                               T* stage, Epi& epi, bool zero_x = false) {
        const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
        const uint64_t ntiles = (uint64_t(m) + 63) / 64;
        uint64_t tb = uint64_t(L) * sp;
        if (tb > ntiles) tb = ntiles;
        const uint64_t te = tb + sp < ntiles ? tb + sp : ntiles;
        const uint64_t q = (te - tb + kWavesPerBlock - 1) / kWavesPerBlock;
        uint64_t t0 = tb + uint64_t(w) * q;
        if (t0 > te) t0 = te;
        const uint64_t t1 = t0 + q < te ? t0 + q : te;
        if (t0 >= t1) return;
        const uint32_t R1 = uint32_t(t1 * 64 < m ? t1 * 64 : m);
        if (zero_x) {  // X = 0: the same epilogue calls, in order, with sums of +0
            T z[K];
#pragma unroll
            for (int j = 0; j < K; ++j) z[j] = T(0);
            for (uint32_t r0 = uint32_t(t0 * 64); r0 < R1; r0 += 64u) {
                const uint32_t row = r0 + uint32_t(lane);
                if (row < R1) {
                    const typename Epi::PV pv = epi.pre(row);
                    epi.done(row, z, pv);
                }
            }
            return;
        }
        run_rows(uint32_t(t0 * 64), R1, rp, cols, val, X, act, stage + w * kStage, lane, epi);
    }
};

}  // namespace nlhip
