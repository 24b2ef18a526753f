// SSOR preconditioner on the device (nlNewSSORPreconditioner(M, omega);
// Matrix::solve_iterative passes omega = 1.5 at
// src/lib/OGF/scene_graph/NL/matrix.cpp:366-368):
//   w_i = (x_i - sum_{j<i} a_ij w_j) * omega / d_i      rows in increasing order
//   y_i = (w_i (d_i / omega) - sum_{j>i} a_ij y_j) * omega / d_i
//                                                       rows in decreasing order
//   y_i = (2 - omega) y_i
// Each sweep is a triangular solve.  The host sorts the rows into levels
// (a row's level is one more than the deepest row it reads), so the rows of
// one level are independent: a level with many rows is one launch over the
// whole grid, and a run of consecutive smaller levels is one workgroup that
// steps through them with a barrier between levels (k_ssor_chain).  Each sweep keeps, in
// level order, the entries each row reads, packed in CRS order.  Every row
// sums them in that order with one rounding per product and per addition,
// so the result is that of the sequential sweep, bit for bit.
#include "dev_common.h"
#include "nlhip_internal.h"

namespace nlhip {

namespace {

// d_i = sum of row i's diagonal entries (CRS order), dscale_i = d_i / omega;
// *bad = 1 when a diagonal is zero or not finite.
__global__ void k_ssor_diag(uint32_t n, const uint32_t* rp, const uint32_t* ci, const double* val,
                            double omega, double* diag, double* dscale, uint32_t* bad) {
    const uint32_t stride = gridDim.x * blockDim.x;
    uint32_t flag = 0;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        double d = 0.0;
        for (uint32_t e = rp[i]; e < rp[i + 1]; ++e)
            if (ci[e] == i) d = add_rn(d, val[e]);
        diag[i] = d;
        dscale[i] = d / omega;
        flag |= (d == 0.0 || !isfinite(d)) ? 1u : 0u;
    }
    if (flag) atomicOr(bad, 1u);
}

constexpr int kSsorU = 8;  // packed entries loaded (and gathers issued) at a time

// The row at position k of a sweep: its packed entries come in groups of
// kSsorU (all loads of a group, then all gathers, then the additions in
// order), so a row costs one round trip per group instead of one per entry.
template <bool UPPER>
__device__ __forceinline__ void ssor_row(const SsorArgs& a, const SsorSweepArgs& sw, uint32_t k) {
    const uint32_t i = sw.rows[k];
    const uint32_t e0 = sw.eoff[k], e1 = sw.eoff[k + 1];
    const double* v = UPPER ? a.y : a.w;
    const double xi = UPPER ? mul_rn(a.w[i], a.dscale[i]) : a.x[i];
    const double di = a.diag[i];
    double S = 0.0;
    for (uint32_t e = e0; e < e1; e += kSsorU) {
        uint32_t c[kSsorU];
        double av[kSsorU], g[kSsorU];
#pragma unroll
        for (int u = 0; u < kSsorU; ++u) {
            const uint32_t q = e + u < e1 ? e + u : e1 - 1u;
            c[u] = sw.col[q];
            av[u] = sw.val[q];
        }
#pragma unroll
        for (int u = 0; u < kSsorU; ++u) g[u] = v[c[u]];
#pragma unroll
        for (int u = 0; u < kSsorU; ++u)
            if (e + uint32_t(u) < e1) S = add_rn(S, mul_rn(av[u], g[u]));
    }
    const double t = mul_rn(add_rn(xi, -S), a.omega);
    (UPPER ? a.y : a.w)[i] = t / di;
}

// One level over the whole grid.
template <bool UPPER>
__global__ __launch_bounds__(kBlock) void k_ssor_sweep(SsorArgs a, uint32_t l) {
    const SsorSweepArgs& sw = UPPER ? a.up : a.lo;
    const uint32_t stride = gridDim.x * kBlock;
    const uint32_t b = sw.off[l], e = sw.off[l + 1];
    for (uint32_t k = b + blockIdx.x * kBlock + threadIdx.x; k < e; k += stride)
        ssor_row<UPPER>(a, sw, k);
}

// A run of levels, positions [k0, k1), by one workgroup, level after level.
//
// What bounds it is the chain from level to level.  The results of the last
// kRing - kChain positions are read from LDS, by position (sw.dep); older ones,
// and those of earlier launches, are known when their chunk begins and are
// read from memory then, the product taking the place of the entry.
// Everything else a row needs is known before: its packed entries, diagonal
// and input are loaded into registers a chunk of kChain positions ahead, the
// row numbers that lead to them another chunk ahead.  A level then costs LDS
// reads, the sums, a division and a barrier: 0.73 us against 1.9 with the values
// through memory (599 levels of up to 300 rows, 300^2 grid: 431 and 518 us a
// sweep).  What must not stand in the level loop is a load or its wait (1.1
// us a level), nor a branch per entry (1.0): rows of more than kChainE entries
// take one in the chunks that have them, in groups of kChainX (entry by entry,
// and every value of such a chunk by a search for it, a level cost 3.5 us).
// 512 threads: 485 and 577 us.
//
// us per application, levels of up to 256 rows through memory in one workgroup
// and the others over the grid -> this: 300^2 cotangent 2970 -> 1630, 1000^2 14300 ->
// 10600, 317^2 LSCM 5240 -> 3060, 27-point stencil on 30^3 1080 -> 930 and on 64^3
// 4340 -> 4180, Delaunay mesh of 200 k vertices numbered by rows 6080 -> 3420, at
// random 360 -> 360.
constexpr uint32_t kChain = 1024;   // threads, positions per chunk
constexpr uint32_t kRing = 16384;   // results kept in LDS (128 KiB)
constexpr int kChainE = 8;          // entries of a row kept in registers
constexpr int kChainX = 4;          // of the others, at a time
constexpr uint32_t kKnown = ~0u;    // dep of an entry kept as its product

struct ChainRow {
    uint32_t row, e0, e1, lev;
};
struct ChainData {
    double x, d, s, v[kChainE];
    uint32_t dep[kChainE];
};

template <bool UPPER>
__global__ __launch_bounds__(kChain) void k_ssor_chain(SsorArgs a, uint32_t k0, uint32_t k1) {
    extern __shared__ double ring[];
    // a row of the chunk has more than 4, more than kChainE entries, a value
    // that is not in the ring
    __shared__ uint32_t s_lev[2], s_kind[2][3];
    const SsorSweepArgs& sw = UPPER ? a.up : a.lo;
    double* const out = UPPER ? a.y : a.w;
    // whether position k reads q's value in LDS (no position of k's chunk has
    // taken its place)
    auto in_ring = [&](uint32_t q, uint32_t k) { return q >= k0 && k - q <= kRing - kChain; };
    auto stored = [&](uint32_t q) {
        return __hip_atomic_load(out + sw.rows[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    auto row_of = [&](uint32_t k) {
        ChainRow r{0, 0, 0, 0};
        if (k < k1) {
            r.row = sw.rows[k];
            r.e0 = sw.eoff[k];
            r.e1 = sw.eoff[k + 1];
            r.lev = sw.lev[k];
        }
        return r;
    };
    auto data_of = [&](uint32_t k, const ChainRow& r) {
        ChainData c{};
        if (k < k1) {
            c.x = UPPER ? a.w[r.row] : a.x[r.row];
            c.d = a.diag[r.row];
            if (UPPER) c.s = a.dscale[r.row];
#pragma unroll
            for (int u = 0; u < kChainE; ++u)
                if (r.e0 + uint32_t(u) < r.e1) {
                    c.v[u] = sw.val[r.e0 + u];
                    c.dep[u] = sw.dep[r.e0 + u];
                }
        }
        return c;
    };
    uint32_t k = k0 + threadIdx.x;
    ChainRow r = row_of(k), rn = row_of(k + kChain);
    ChainData c = data_of(k, r);
    uint32_t chunk = 0;
    if (threadIdx.x < 6) s_kind[threadIdx.x / 3][threadIdx.x % 3] = 0;
    __syncthreads();
    for (uint32_t c0 = k0; c0 < k1; c0 += kChain, k += kChain, ++chunk) {
        // this chunk's registers, loaded a chunk ago: used here, so that the
        // compiler waits for them before the next loads are issued and not
        // (for those, too) in the level loop
        asm volatile("" : "+v"(c.x), "+v"(c.d), "+v"(c.s), "+v"(r.row), "+v"(r.e0), "+v"(r.e1),
                     "+v"(r.lev), "+v"(rn.row), "+v"(rn.e0), "+v"(rn.e1), "+v"(rn.lev));
#pragma unroll
        for (int u = 0; u < kChainE; ++u) asm volatile("" : "+v"(c.v[u]), "+v"(c.dep[u]));
        if (UPPER) c.x = mul_rn(c.x, c.s);
        const uint32_t last = k1 - c0 < kChain ? k1 - c0 - 1u : kChain - 1u;
        const uint32_t len = r.e1 - r.e0;
        if (threadIdx.x == 0) s_lev[0] = r.lev;
        if (threadIdx.x == last) s_lev[1] = r.lev;
        // Values that are not in the ring are known: read here, and kept as
        // the entry's product.  They are kRing - kChain positions back, in an
        // earlier group of four chunks, whose stores have been waited for.
        bool far = false;
#pragma unroll
        for (int u = 0; u < kChainE; ++u)
            far |= k < k1 && uint32_t(u) < len && !in_ring(c.dep[u], k);
        if (far) {
#pragma unroll
            for (int u0 = 0; u0 < kChainE; u0 += kChainX) {
                double g[kChainX];
#pragma unroll
                for (int u = u0; u < u0 + kChainX; ++u) {
                    g[u - u0] = 0.0;
                    if (uint32_t(u) < len && !in_ring(c.dep[u], k)) g[u - u0] = stored(c.dep[u]);
                }
#pragma unroll
                for (int u = u0; u < u0 + kChainX; ++u)
                    if (uint32_t(u) < len && !in_ring(c.dep[u], k)) {
                        c.v[u] = mul_rn(c.v[u], g[u - u0]);
                        c.dep[u] = kKnown;
                    }
            }
            s_kind[chunk & 1u][2] = 1;
        }
        if (len > 4u) s_kind[chunk & 1u][0] = 1;
        if (len > uint32_t(kChainE)) s_kind[chunk & 1u][1] = 1;
        if (chunk % 4 == 3) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        const uint32_t l0 = s_lev[0], l1 = s_lev[1];
        const uint32_t more = s_kind[chunk & 1u][0], most = s_kind[chunk & 1u][1],
                       known = s_kind[chunk & 1u][2];
        if (threadIdx.x < 3) s_kind[(chunk + 1u) & 1u][threadIdx.x] = 0;
        const ChainRow rnn = row_of(k + 2 * kChain);
        const ChainData cn = data_of(k + kChain, rn);
        auto finish = [&](double S) {
            const double t = mul_rn(add_rn(c.x, -S), a.omega) / c.d;
            ring[k % kRing] = t;
            out[r.row] = t;
        };
        // the sum of the first N entries; past the row's end a value that is
        // not used
        auto kept = [&](auto n, auto pre) {
            constexpr int N = decltype(n)::value;
            double S = 0.0, g[N];
#pragma unroll
            for (int u = 0; u < N; ++u) g[u] = ring[c.dep[u] % kRing];
#pragma unroll
            for (int u = 0; u < N; ++u) {
                double t = mul_rn(c.v[u], g[u]);
                if (decltype(pre)::value && c.dep[u] == kKnown) t = c.v[u];
                t = add_rn(S, t);
                S = uint32_t(u) < len ? t : S;
            }
            return S;
        };
        // no loads in here: the next chunk's stay in flight
        auto levels = [&](auto n, auto pre) {
            for (uint32_t l = l0; l <= l1; ++l) {
                if (k < k1 && r.lev == l) finish(kept(n, pre));
                __syncthreads();
            }
        };
        using N4 = std::integral_constant<int, 4>;
        using N8 = std::integral_constant<int, kChainE>;
        if (most) {
            // the entries past those kept: as many at a time, loads first
            const bool longer = __any(k < k1 && len > uint32_t(kChainE));
            for (uint32_t l = l0; l <= l1; ++l) {
                if (k < k1 && r.lev == l) {
                    double S = kept(N8{}, std::true_type{});
                    if (longer) {
                        for (uint32_t e = r.e0 + kChainE; e < r.e1; e += kChainX) {
                            uint32_t q[kChainX];
                            double v[kChainX], g[kChainX];
                            bool out = false;
#pragma unroll
                            for (int u = 0; u < kChainX; ++u) {
                                const uint32_t at = e + u < r.e1 ? e + u : r.e1 - 1u;
                                q[u] = sw.dep[at];
                                v[u] = sw.val[at];
                            }
#pragma unroll
                            for (int u = 0; u < kChainX; ++u) {
                                g[u] = ring[q[u] % kRing];
                                out |= !in_ring(q[u], k);
                            }
                            if (out) {
#pragma unroll
                                for (int u = 0; u < kChainX; ++u)
                                    if (!in_ring(q[u], k)) g[u] = stored(q[u]);
                            }
#pragma unroll
                            for (int u = 0; u < kChainX; ++u)
                                if (e + uint32_t(u) < r.e1) S = add_rn(S, mul_rn(v[u], g[u]));
                        }
                    }
                    finish(S);
                }
                __syncthreads();
            }
        } else if (known) {
            levels(N8{}, std::true_type{});
        } else if (more) {
            levels(N8{}, std::false_type{});
        } else {
            levels(N4{}, std::false_type{});
        }
        r = rn;
        rn = rnn;
        c = cn;
    }
}

__global__ void k_ssor_scale(SsorArgs a) {
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < a.n; i += stride)
        a.y[i] = mul_rn(a.post, a.y[i]);
}

uint32_t blocks_for(uint64_t n) {
    const uint64_t g = (n + kBlock - 1) / kBlock;
    return uint32_t(g < 1 ? 1 : (g > 65535 ? 65535 : g));
}

}  // namespace

hipError_t ssor_diag(uint32_t n, const uint32_t* rp, const uint32_t* ci, const double* val,
                     double omega, double* diag, double* dscale, uint32_t* bad, hipStream_t s) {
    if (n) k_ssor_diag<<<blocks_for(n), kBlock, 0, s>>>(n, rp, ci, val, omega, diag, dscale, bad);
    return hipGetLastError();
}

hipError_t ssor_level(const SsorArgs& a, bool upper, uint32_t l, uint32_t rows, hipStream_t s) {
    if (upper) k_ssor_sweep<true><<<blocks_for(rows), kBlock, 0, s>>>(a, l);
    else k_ssor_sweep<false><<<blocks_for(rows), kBlock, 0, s>>>(a, l);
    return hipGetLastError();
}

hipError_t ssor_chain_init() {
    for (const void* f : {reinterpret_cast<const void*>(&k_ssor_chain<true>),
                          reinterpret_cast<const void*>(&k_ssor_chain<false>)}) {
        const hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize,
                                                 int(kRing * sizeof(double)));
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t ssor_chain(const SsorArgs& a, bool upper, uint32_t k0, uint32_t k1, hipStream_t s) {
    if (k0 >= k1) return hipSuccess;
    if (upper) k_ssor_chain<true><<<1, kChain, kRing * sizeof(double), s>>>(a, k0, k1);
    else k_ssor_chain<false><<<1, kChain, kRing * sizeof(double), s>>>(a, k0, k1);
    return hipGetLastError();
}

hipError_t ssor_scale(const SsorArgs& a, hipStream_t s) {
    if (a.n) k_ssor_scale<<<blocks_for(a.n), kBlock, 0, s>>>(a);
    return hipGetLastError();
}

}  // namespace nlhip
