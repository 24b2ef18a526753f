// Multi right-hand-side Jacobi-PCG: k independent CG recurrences (one per
// right-hand side, as OpenNL's NL_NB_SYSTEMS loop solves them) that share
// every pass over the matrix.  Used for mesh_smooth's x, y, z solves
// (src/lib/OGF/mesh/commands/mesh_grob_surface_commands.cpp:703).
//
// Layout: vectors are n x k row-major ("interleaved"), element (i, j) at
// i*k + j, so the gather of x[col] for all right-hand sides is one
// contiguous k*8-byte segment.  The SpMM-shaped launches (SpMM step, start,
// residual) sum each row in column order with one rounding per product and
// per add, with one of two engines (dev_spmm.h), same sums:
// * k <= kMultiStreamMaxK: the stream engine, one row per lane, the matrix
//   streamed in 64-row tiles and each entry's k values gathered as one copy;
//   Pdq workgroups of sp tiles, as many as the device holds at once;
// * larger k: the row engine, G lanes per row (G = k rounded up to a power of
//   two, or half of it with two columns per lane).
//
// An iteration is the single-right-hand-side one (k_cg.hip): direction
// (x -= alpha d with the pending alpha, stopping test, d = beta d + h), SpMM
// (Q = A D, partials of d_j.q_j), update (r -= alpha q, partials of r_j.h_j
// and r_j.r_j).  h = D^-1 r is formed where it is read, from r and the one
// D^-1 of the row, and not stored: 80 n k bytes per iteration with the SpMM's
// 16, against 96 with h in memory and x updated beside r.
// * k <= kMultiStreamMaxK: three launches, whose workgroups reduce the
//   partials themselves (P k of them each);
// * larger k: the scalars in launches of one workgroup per column in between
//   (5 launches), where P k partials per workgroup would outweigh the step.
// Against five launches each with h stored, us per iteration: 1500^2 rows,
// k = 32, FP64 1700 -> 1350; 300^2, k = 3, FP64 25 -> 17 of kernel time; 1000^2,
// k = 3, FP32 57 -> 41.
// Columns whose stopping test held are left untouched (stop, raised with the
// test, becomes done in the SpMM); once every column has stopped, the
// launches exit at once.
#include <algorithm>

#include "dev_common.h"
#include "dev_spmm.h"
#include "nlhip_internal.h"
#include "nlhip_kernels.h"

namespace nlhip {

// Rows [r0, r1) of logical block L for the element-wise kernels, with the
// G-lane row groups: thread t handles column t % G of rows
// r0 + t / G, r0 + t / G + kBlock / G, ...
__device__ __forceinline__ void block_rows(const uint32_t m, const uint32_t rows_per_block,
                                           uint32_t L, uint32_t& r0, uint32_t& r1) {
    const uint64_t rb = uint64_t(L) * rows_per_block;
    r0 = rb < m ? uint32_t(rb) : m;
    r1 = (uint64_t(r0) + rows_per_block < m) ? r0 + rows_per_block : m;
}

// Whether any column's flags, written by earlier launches, are clear; the
// same answer in every thread.  The direction step runs for columns that stop
// in this iteration too (the pending update of x), the others do not.
template <typename T>
__device__ __forceinline__ bool any_open(const MultiArgs<T>& a) {
    for (uint32_t j = 0; j < a.k; ++j)
        if (!a.done[j]) return true;
    return false;
}
template <typename T>
__device__ __forceinline__ bool any_active(const MultiArgs<T>& a) {
    for (uint32_t j = 0; j < a.k; ++j)
        if (!a.done[j] && !a.stop[j]) return true;
    return false;
}
// In the SpMM launch, by one workgroup: columns that stopped in this
// iteration are done (the direction launch has updated their x).  Workgroups
// that read done[j] in this launch see stop[j] either way.
template <typename T>
__device__ __forceinline__ void close_stopped(const MultiArgs<T>& a) {
    if (blockIdx.x == 0 && threadIdx.x < a.k && a.stop[threadIdx.x]) a.done[threadIdx.x] = 1;
}

// Per-workgroup partial sums of k columns, V per lane (lane l of the lanes of
// a row holds columns l*V .. l*V + V - 1; 4 to 32 lanes): the lanes of a
// wavefront that hold a column by a butterfly over its rows, then the
// wavefronts in index order; lds holds kWavesPerBlock * 32 values.  (The lanes
// added one after another through LDS, 64 of them with 4 lanes per row, cost 3.5
// of the 7.9 us of an update step with 10 k rows and 8 columns.)  The partials of
// columns with done[j] or stop[j] set (may be null) stay as they are: a
// re-opened column continues from them.
template <int V, typename T>
__device__ __forceinline__ void column_partials_v(const T (&v)[V], uint32_t k, uint32_t lanes,
                                                  T* lds, T* out /* k values */,
                                                  const int32_t* done = nullptr,
                                                  const int32_t* stop = nullptr) {
    const uint32_t lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    __syncthreads();
#pragma unroll
    for (int c = 0; c < V; ++c) {
        T s = xor_add<32>(v[c]);
        if (lanes <= 16) s = xor_add<16>(s);
        if (lanes <= 8) s = xor_add<8>(s);
        if (lanes <= 4) s = xor_add<4>(s);
        if (lane < lanes) lds[w * 32 + lane * V + c] = s;
    }
    __syncthreads();
    if (threadIdx.x < k && !(done && (done[threadIdx.x] || stop[threadIdx.x]))) {
        T s = lds[threadIdx.x];
        for (int x = 1; x < kWavesPerBlock; ++x) s += lds[x * 32 + threadIdx.x];
        out[threadIdx.x] = s;
    }
}

// Columns per lane of the row-group SpMM kernels for k right-hand sides
// (G = k rounded up to a power of two lanes per row with one): two, gathered
// as one 16-byte copy per entry, for FP64 when k is even and at least 6.  FP64
// solves (cotangent grids, t = 1), one column per lane -> two: 300^2 k = 8 2.41 ->
// 2.42 ms, k = 32 4.42 -> 3.92; 700^2 5.51 -> 5.18, 17.8 -> 14.9; 1500^2 20.2 -> 17.9,
// 79.6 -> 66.7.  FP32 keeps one: pairs (8 bytes) take mixed solves from 3.16 to
// 3.56 ms (300^2, k = 8), 5.11 to 5.30 (700^2), but 18.2 to 16.7 at 1500^2.
template <typename T>
bool multi_two_cols(uint32_t k) {
    return std::is_same<T, double>::value && k % 2 == 0 && k >= 6;
}
template <int G>
constexpr int two_cols_v() {
    return G >= 8 ? 2 : 1;
}

template <int G, int V, typename T, bool PREC>
__global__ __launch_bounds__(kBlock) void k_m_init(MultiArgs<T> a) {
    __shared__ T lds[kWavesPerBlock * 32];
    const uint32_t L = xcd_logical_block(blockIdx.x, gridDim.x);
    const uint32_t k = a.k;
    T prh[V], prr[V], pbb[V];
#pragma unroll
    for (int c = 0; c < V; ++c) prh[c] = prr[c] = pbb[c] = T(0);
    struct PV {
        Lane<V, T> b;
        T dinv;
    };
    auto pre = [&](uint32_t row, uint32_t j) {
        return PV{lane_load<V>(a.b + uint64_t(row) * k + j), PREC ? a.dinv[row] : T(1)};
    };
    auto fin = [&](uint32_t row, uint32_t j, const T (&s)[V], const PV& pv) {
        T r[V];
#pragma unroll
        for (int c = 0; c < V; ++c) {
            const T bi = pv.b.v[c];
            r[c] = add_rn(s[c], mul_rn(T(-1), bi));
            const T hi = PREC ? mul_rn(pv.dinv, r[c]) : r[c];
            prh[c] += r[c] * hi;
            prr[c] += r[c] * r[c];
            pbb[c] += bi * bi;
        }
        lane_store<V>(a.r + uint64_t(row) * k + j, r);
    };
    const bool zero_x = a.x_nonzero && *a.x_nonzero == 0;  // X = 0: A X = 0 (block-uniform)
    spmm_rows_v<G / V, V>(a.m, k, L, a.rp, a.ci, a.val, a.x, pre, fin,
                               nullptr, zero_x);
    column_partials_v<V>(prh, k, G / V, lds, a.part_rh + size_t(L) * k);
    column_partials_v<V>(prr, k, G / V, lds, a.part_rr + size_t(L) * k);
    column_partials_v<V>(pbb, k, G / V, lds, a.part_bb + size_t(L) * k);
}

// One workgroup per column: sum of the P partials of column j (stride k) in
// a fixed order (thread t takes partials t, t + 256, ..., then the block
// sums the threads); every thread gets the total.
template <typename T>
__device__ __forceinline__ T col_sum(const T* part, uint32_t P, uint32_t k, uint32_t j,
                                     T* lds) {
    T v = T(0);
    uint32_t p = threadIdx.x;
    for (; p + 3 * kBlock < P; p += 4 * kBlock) {
        const T a = part[size_t(p) * k + j], b = part[size_t(p + kBlock) * k + j];
        const T c = part[size_t(p + 2 * kBlock) * k + j];
        const T d = part[size_t(p + 3 * kBlock) * k + j];
        v = v + a + b + c + d;
    }
    for (; p < P; p += kBlock) v += part[size_t(p) * k + j];
    return block_sum_all(v, lds);
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_m_sys_init(MultiArgs<T> a, T eps, int max_iter) {
    __shared__ T lds[kWavesPerBlock];
    const uint32_t j = blockIdx.x;
    // the start's partials: one per workgroup of the SpMM-shaped launch
    const T rho = col_sum(a.part_rh, a.Pdq, a.k, j, lds);
    const T err = col_sum(a.part_rr, a.Pdq, a.k, j, lds);
    const T bb = col_sum(a.part_bb, a.Pdq, a.k, j, lds);
    if (threadIdx.x == 0) {
        const T thresh = (eps * eps) * bb;
        a.bb[j] = bb;
        a.thresh[j] = thresh;
        a.rho[j] = rho;
        a.rho_prev[j] = T(1);
        a.err[j] = err;
        a.beta[j] = T(0);
        a.alpha[j] = T(0);
        a.iters[j] = 0;
        a.stop[j] = 0;
        const bool skip = a.skip && a.skip[j];
        a.done[j] = (skip || !(err > thresh) || max_iter <= 0) ? 1 : 0;
    }
}

// The sums of N x K interleaved partials (part[c][p K + j], p < P) over the
// workgroups, in col_sum's order, in every thread; lds holds
// kWavesPerBlock * N * K values.
template <int N, int K, typename T>
__device__ __forceinline__ void all_col_sums(const T* const (&part)[N], uint32_t P, T* lds,
                                             T (&out)[N][K]) {
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
#pragma unroll
    for (int c = 0; c < N; ++c)
#pragma unroll
        for (int j = 0; j < K; ++j) out[c][j] = T(0);
    for (uint32_t p = threadIdx.x; p < P; p += kBlock)
#pragma unroll
        for (int c = 0; c < N; ++c)
#pragma unroll
            for (int j = 0; j < K; ++j) out[c][j] += part[c][size_t(p) * K + j];
#pragma unroll
    for (int c = 0; c < N; ++c)
#pragma unroll
        for (int j = 0; j < K; ++j) {
            const T v = group_sum<kWave>(out[c][j]);
            if (lane == 0) lds[(c * K + j) * kWavesPerBlock + w] = v;
        }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < N; ++c)
#pragma unroll
        for (int j = 0; j < K; ++j) {
            const T* l = lds + (c * K + j) * kWavesPerBlock;
            out[c][j] = ((l[0] + l[1]) + l[2]) + l[3];
        }
}

// Direction step for K <= kMultiStreamMaxK columns, one row per lane: the
// scalars of every column from the last update's partials (block 0 writes
// them), then x and d.
template <int K, typename T, bool PREC>
__global__ __launch_bounds__(kBlock) void k_m_dir_few(MultiArgs<T> a, int max_iter) {
    __shared__ T lds[kWavesPerBlock * 2 * K];
    if (!any_open(a)) return;  // every column has stopped
    T sums[2][K];
    const T* const parts[2] = {a.part_rh, a.part_rr};
    all_col_sums<2, K>(parts, a.P, lds, sums);
    bool upd[K], dir[K], first[K];
    T alpha[K], beta[K];
#pragma unroll
    for (int j = 0; j < K; ++j) {
        const int it = a.iters[j];
        const bool open = !a.done[j];
        first[j] = it == 0;  // its scalars and test: the start's
        const bool stop = !first[j] && (!(sums[1][j] > a.thresh[j]) || it >= max_iter);
        alpha[j] = a.alpha[j];
        beta[j] = first[j] ? T(0) : sums[0][j] / a.rho_prev[j];
        upd[j] = open && !first[j];
        dir[j] = open && !stop;
        if (blockIdx.x == 0 && threadIdx.x == 0 && upd[j]) {
            a.rho[j] = sums[0][j];
            a.err[j] = sums[1][j];
            if (stop) a.stop[j] = 1;
            else a.beta[j] = beta[j];
        }
    }
    const uint32_t L = xcd_logical_block(blockIdx.x, gridDim.x);
    uint32_t r0, r1;
    block_rows(a.m, a.rows_per_block, L, r0, r1);
    constexpr int U = 2;
    for (uint32_t i0 = r0 + threadIdx.x; i0 < r1; i0 += U * kBlock) {
        T xv[U][K], dv[U][K], rv[U][K], pv[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t i = i0 + uint32_t(u * kBlock);
            if (i < r1) {
                __builtin_memcpy(xv[u], a.x + uint64_t(i) * K, sizeof(T) * K);
                __builtin_memcpy(dv[u], a.d + uint64_t(i) * K, sizeof(T) * K);
                __builtin_memcpy(rv[u], a.r + uint64_t(i) * K, sizeof(T) * K);
                pv[u] = PREC ? a.dinv[i] : T(1);
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t i = i0 + uint32_t(u * kBlock);
            if (i < r1) {
#pragma unroll
                for (int j = 0; j < K; ++j) {
                    const T h = PREC ? mul_rn(pv[u], rv[u][j]) : rv[u][j];
                    const T x = add_rn(xv[u][j], mul_rn(-alpha[j], dv[u][j]));
                    const T d = first[j] ? h : add_rn(mul_rn(beta[j], dv[u][j]), h);
                    xv[u][j] = upd[j] ? x : xv[u][j];
                    dv[u][j] = dir[j] ? d : dv[u][j];
                }
                __builtin_memcpy(a.x + uint64_t(i) * K, xv[u], sizeof(T) * K);
                __builtin_memcpy(a.d + uint64_t(i) * K, dv[u], sizeof(T) * K);
            }
        }
    }
}

// The scalars of the direction step, one workgroup per column (larger k).
template <typename T>
__global__ __launch_bounds__(kBlock) void k_m_beta(MultiArgs<T> a, int max_iter) {
    __shared__ T lds[kWavesPerBlock];
    const uint32_t j = blockIdx.x;
    const int it = a.iters[j];
    if (a.done[j] || it == 0) return;
    const T rho = col_sum(a.part_rh, a.P, a.k, j, lds);
    const T err = col_sum(a.part_rr, a.P, a.k, j, lds);
    if (threadIdx.x == 0) {
        a.rho[j] = rho;
        a.err[j] = err;
        if (!(err > a.thresh[j]) || it >= max_iter) a.stop[j] = 1;
        else a.beta[j] = rho / a.rho_prev[j];
    }
}

// Rows per lane and trip of the element-wise steps of larger k: their loads
// before their stores.
constexpr int kMultiU = 4;

// True when x, d, r and q together exceed the last-level cache: the
// element-wise steps of larger k then load and store past it (NT), which left
// it to the rows the SpMM gathers.  Per solve, without -> with: 1500^2 rows x
// 32 (576 MB each) 8.21 -> 7.87 ms, 1000^2 x 32 (256 MB) 4.04 -> 3.66, 1500^2
// x 8 (144 MB) 2.48 -> 2.28, 700^2 x 32 (125 MB) 2.05 -> 2.00; the same within
// 1% at 64 MB and below.
template <typename T>
bool multi_streamed(uint32_t m, uint32_t k) {
    return 4 * uint64_t(m) * k * sizeof(T) > kLastLevelCache;
}

// Direction step of larger k: V adjacent columns per lane, G / V lanes per row.
template <int V, bool NT, typename T, bool PREC>
__global__ __launch_bounds__(kBlock) void k_m_dir(MultiArgs<T> a) {
    if (!any_open(a)) return;  // every column has stopped
    const uint32_t L = xcd_logical_block(blockIdx.x, gridDim.x);
    const uint32_t k = a.k, lanes = a.G / V, per = kBlock / lanes;
    const uint32_t g = threadIdx.x / lanes, j = (threadIdx.x % lanes) * V;
    if (j >= k) return;
    bool upd[V], dir[V], first[V];
    T alpha[V], beta[V];
    bool any = false;
#pragma unroll
    for (int c = 0; c < V; ++c) {
        first[c] = a.iters[j + c] == 0;
        upd[c] = !a.done[j + c] && !first[c];
        dir[c] = !a.done[j + c] && !a.stop[j + c];
        any |= upd[c] || dir[c];
        alpha[c] = a.alpha[j + c];
        beta[c] = a.beta[j + c];
    }
    if (!any) return;
    uint32_t r0, r1;
    block_rows(a.m, a.rows_per_block, L, r0, r1);
    for (uint32_t i0 = r0 + g; i0 < r1; i0 += kMultiU * per) {
        Lane<V, T> xv[kMultiU], dv[kMultiU], rv[kMultiU];
        T pv[kMultiU];
#pragma unroll
        for (int u = 0; u < kMultiU; ++u) {
            const uint32_t row = i0 + uint32_t(u) * per;
            if (row < r1) {
                const uint64_t i = uint64_t(row) * k + j;
                xv[u] = lane_load<V, NT>(a.x + i);
                dv[u] = lane_load<V, NT>(a.d + i);
                rv[u] = lane_load<V, NT>(a.r + i);
                pv[u] = PREC ? a.dinv[row] : T(1);
            }
        }
#pragma unroll
        for (int u = 0; u < kMultiU; ++u) {
            const uint32_t row = i0 + uint32_t(u) * per;
            if (row < r1) {
                const uint64_t i = uint64_t(row) * k + j;
#pragma unroll
                for (int c = 0; c < V; ++c) {
                    const T h = PREC ? mul_rn(pv[u], rv[u].v[c]) : rv[u].v[c];
                    const T x = add_rn(xv[u].v[c], mul_rn(-alpha[c], dv[u].v[c]));
                    const T d = first[c] ? h : add_rn(mul_rn(beta[c], dv[u].v[c]), h);
                    xv[u].v[c] = upd[c] ? x : xv[u].v[c];
                    dv[u].v[c] = dir[c] ? d : dv[u].v[c];
                }
                lane_store<V, NT>(a.x + i, xv[u].v);
                lane_store<V, NT>(a.d + i, dv[u].v);
            }
        }
    }
}

template <int G, int V, typename T>
__global__ __launch_bounds__(kBlock) void k_m_spmm(MultiArgs<T> a) {
    __shared__ T lds[kWavesPerBlock * 32];
    close_stopped(a);
    if (!any_active(a)) return;  // every column has stopped (block-uniform)
    const uint32_t L = xcd_logical_block(blockIdx.x, gridDim.x);
    const uint32_t k = a.k;
    T pdq[V];
#pragma unroll
    for (int c = 0; c < V; ++c) pdq[c] = T(0);
    auto pre = [&](uint32_t row, uint32_t j) {
        return lane_load<V>(a.d + uint64_t(row) * k + j);
    };
    auto fin = [&](uint32_t row, uint32_t j, const T (&s)[V], const Lane<V, T>& d) {
        lane_store<V>(a.q + uint64_t(row) * k + j, s);
#pragma unroll
        for (int c = 0; c < V; ++c) pdq[c] += d.v[c] * s[c];
    };
    spmm_rows_v<G / V, V>(a.m, k, L, a.rp, a.ci, a.val, a.d, pre, fin,
                               a.done);
    column_partials_v<V>(pdq, k, G / V, lds, a.part_dq + size_t(L) * k);
}

// Wavefront entries per chunk / 64 of the stream kernels.
constexpr int kMultiStreamE = 4;

// The stream SpMM's epilogue: q[row, :] = sums, and d[row, j] * sums[j]
// added to column j's partial of d.q (row by row).
template <int K, typename T>
struct MultiDqEpilogue {
    const T* __restrict__ d;
    T* __restrict__ q;
    T (&pdq)[K];
    struct PV {
        T v[K];
    };
    __device__ __forceinline__ PV pre(uint32_t row) const {
        PV p;
#pragma unroll
        for (int j = 0; j < K; ++j) p.v[j] = d[uint64_t(row) * K + j];
        return p;
    }
    __device__ __forceinline__ void done(uint32_t row, const T (&s)[K], const PV& pv) {
#pragma unroll
        for (int j = 0; j < K; ++j) {
            q[uint64_t(row) * K + j] = s[j];
            pdq[j] += pv.v[j] * s[j];
        }
    }
};

// Per-workgroup partials of K columns: each wavefront's sum (xor butterfly),
// then the wavefronts in index order; out[j] for j < K.  Every thread of
// the block calls it (it synchronises the block).
template <int K, typename T>
__device__ __forceinline__ void stream_partials(const T (&v)[K], T* red, T* out,
                                                const int32_t* done = nullptr,
                                                const int32_t* stop = nullptr) {
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    __syncthreads();  // red of an earlier call has been read
#pragma unroll
    for (int j = 0; j < K; ++j) {
        const T s = group_sum<kWave>(v[j]);
        if (lane == 0) red[w * K + j] = s;
    }
    __syncthreads();
    // a stopped column's partials stay as they are (see column_partials_v)
    if (threadIdx.x < uint32_t(K) && !(done && (done[threadIdx.x] || stop[threadIdx.x]))) {
        T s = red[threadIdx.x];
        for (int x = 1; x < kWavesPerBlock; ++x) s += red[x * K + threadIdx.x];
        out[threadIdx.x] = s;
    }
}

// SpMM step for k = K <= kMultiStreamMaxK with the stream engine: Q = A D
// for the columns still iterating, Pdq workgroups of sp tiles.
template <int K, bool D16, typename T>
__global__ __launch_bounds__(kBlock) void k_m_spmm_stream(MultiArgs<T> a) {
    using Eng = MultiStreamEngine<K, kMultiStreamE, D16>;
    __shared__ T stage[kWavesPerBlock * Eng::kStage];
    __shared__ T red[kWavesPerBlock * K];
    close_stopped(a);
    if (!any_active(a)) return;  // every column has stopped (block-uniform)
    const uint32_t L = xcd_logical_block(blockIdx.x, gridDim.x);
    bool act[K];
    T pdq[K];
#pragma unroll
    for (int j = 0; j < K; ++j) {
        act[j] = !a.done[j] && !a.stop[j];
        pdq[j] = T(0);
    }
    MultiDqEpilogue<K, T> epi{a.d, a.q, pdq};
    Eng::run(a.m, a.sp, L, a.rp, a.cols, a.val, a.d, act, stage, epi);
    stream_partials<K>(pdq, red, a.part_dq + size_t(L) * K);
}

// The start's epilogue (k_m_init's, row by row): r = A x - b and, with
// h = D^-1 r, partials of r.h, r.r and b.b per column.
template <int K, typename T, bool PREC>
struct MultiInitEpilogue {
    const MultiArgs<T>& a;
    T (&prh)[K];
    T (&prr)[K];
    T (&pbb)[K];
    struct PV {
        T b[K];
        T dinv;
    };
    __device__ __forceinline__ PV pre(uint32_t row) const {
        PV p;
#pragma unroll
        for (int j = 0; j < K; ++j) p.b[j] = a.b[uint64_t(row) * K + j];
        p.dinv = PREC ? a.dinv[row] : T(1);
        return p;
    }
    __device__ __forceinline__ void done(uint32_t row, const T (&s)[K], const PV& pv) {
#pragma unroll
        for (int j = 0; j < K; ++j) {
            const uint64_t i = uint64_t(row) * K + j;
            const T bi = pv.b[j];
            const T ri = add_rn(s[j], mul_rn(T(-1), bi));
            const T hi = PREC ? mul_rn(pv.dinv, ri) : ri;
            a.r[i] = ri;
            prh[j] += ri * hi;
            prr[j] += ri * ri;
            pbb[j] += bi * bi;
        }
    }
};

// k_m_init with the stream engine (k = K <= kMultiStreamMaxK): Pdq
// workgroups, Pdq partials of each kind.
template <int K, bool D16, typename T, bool PREC>
__global__ __launch_bounds__(kBlock) void k_m_init_stream(MultiArgs<T> a) {
    using Eng = MultiStreamEngine<K, kMultiStreamE, D16>;
    __shared__ T stage[kWavesPerBlock * Eng::kStage];
    __shared__ T red[kWavesPerBlock * K];
    const uint32_t L = xcd_logical_block(blockIdx.x, gridDim.x);
    bool act[K];
    T prh[K], prr[K], pbb[K];
#pragma unroll
    for (int j = 0; j < K; ++j) {
        act[j] = true;
        prh[j] = prr[j] = pbb[j] = T(0);
    }
    MultiInitEpilogue<K, T, PREC> epi{a, prh, prr, pbb};
    const bool zero_x = a.x_nonzero && *a.x_nonzero == 0;  // X = 0: A X = 0 (block-uniform)
    Eng::run(a.m, a.sp, L, a.rp, a.cols, a.val, a.x, act, stage, epi, zero_x);
    stream_partials<K>(prh, red, a.part_rh + size_t(L) * K);
    stream_partials<K>(prr, red, a.part_rr + size_t(L) * K);
    stream_partials<K>(pbb, red, a.part_bb + size_t(L) * K);
}

// The scalars of the update step, one workgroup per column (larger k).
template <typename T>
__global__ __launch_bounds__(kBlock) void k_m_alpha(MultiArgs<T> a) {
    __shared__ T lds[kWavesPerBlock];
    const uint32_t j = blockIdx.x;
    if (a.done[j] || a.stop[j]) return;
    const T dq = col_sum(a.part_dq, a.Pdq, a.k, j, lds);
    if (threadIdx.x == 0) {
        const T rho = a.rho[j];
        a.alpha[j] = rho / dq;
        a.rho_prev[j] = rho;
        a.iters[j] = a.iters[j] + 1;
    }
}

// Update step for K <= kMultiStreamMaxK columns, one row per lane: alpha of
// every column from the SpMM's partials (block 0 writes the scalars), then r.
template <int K, typename T, bool PREC>
__global__ __launch_bounds__(kBlock) void k_m_update_few(MultiArgs<T> a) {
    __shared__ T lds[kWavesPerBlock * K];
    __shared__ T red[kWavesPerBlock * K];
    if (!any_active(a)) return;  // every column has stopped (block-uniform)
    T dq[1][K];
    const T* const parts[1] = {a.part_dq};
    all_col_sums<1, K>(parts, a.Pdq, lds, dq);
    bool act[K];
    T alpha[K], prh[K], prr[K];
#pragma unroll
    for (int j = 0; j < K; ++j) {
        act[j] = !a.done[j] && !a.stop[j];
        const T rho = a.rho[j];
        alpha[j] = rho / dq[0][j];
        prh[j] = prr[j] = T(0);
        if (blockIdx.x == 0 && threadIdx.x == 0 && act[j]) {
            a.alpha[j] = alpha[j];
            a.rho_prev[j] = rho;
            a.iters[j] = a.iters[j] + 1;
        }
    }
    const uint32_t L = xcd_logical_block(blockIdx.x, gridDim.x);
    uint32_t r0, r1;
    block_rows(a.m, a.rows_per_block, L, r0, r1);
    constexpr int U = 2;
    for (uint32_t i0 = r0 + threadIdx.x; i0 < r1; i0 += U * kBlock) {
        T rv[U][K], qv[U][K], pv[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t i = i0 + uint32_t(u * kBlock);
            if (i < r1) {
                __builtin_memcpy(rv[u], a.r + uint64_t(i) * K, sizeof(T) * K);
                __builtin_memcpy(qv[u], a.q + uint64_t(i) * K, sizeof(T) * K);
                pv[u] = PREC ? a.dinv[i] : T(1);
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t i = i0 + uint32_t(u * kBlock);
            if (i < r1) {
#pragma unroll
                for (int j = 0; j < K; ++j) {
                    const T ri = add_rn(rv[u][j], mul_rn(-alpha[j], qv[u][j]));
                    const T hi = PREC ? mul_rn(pv[u], ri) : ri;
                    rv[u][j] = act[j] ? ri : rv[u][j];
                    prh[j] += ri * hi;
                    prr[j] += ri * ri;
                }
                __builtin_memcpy(a.r + uint64_t(i) * K, rv[u], sizeof(T) * K);
            }
        }
    }
    stream_partials<K>(prh, red, a.part_rh + size_t(L) * K, a.done, a.stop);
    stream_partials<K>(prr, red, a.part_rr + size_t(L) * K, a.done, a.stop);
}

// Update step of larger k: V adjacent columns per lane, G / V lanes per row.
template <int V, bool NT, typename T, bool PREC>
__global__ __launch_bounds__(kBlock) void k_m_update(MultiArgs<T> a) {
    __shared__ T lds[kWavesPerBlock * 32];
    if (!any_active(a)) return;  // every column has stopped (block-uniform)
    const uint32_t L = xcd_logical_block(blockIdx.x, gridDim.x);
    const uint32_t k = a.k, lanes = a.G / V, per = kBlock / lanes;
    const uint32_t g = threadIdx.x / lanes, j = (threadIdx.x % lanes) * V;
    T prh[V], prr[V], alpha[V];
    bool act[V];
    bool any = false;
#pragma unroll
    for (int c = 0; c < V; ++c) {
        prh[c] = prr[c] = alpha[c] = T(0);
        act[c] = j + c < k && !a.done[j + c] && !a.stop[j + c];
        if (act[c]) alpha[c] = a.alpha[j + c];
        any |= act[c];
    }
    uint32_t r0, r1;
    block_rows(a.m, a.rows_per_block, L, r0, r1);
    if (any) {
        for (uint32_t i0 = r0 + g; i0 < r1; i0 += kMultiU * per) {
            Lane<V, T> rv[kMultiU], qv[kMultiU];
            T pv[kMultiU];
#pragma unroll
            for (int u = 0; u < kMultiU; ++u) {
                const uint32_t row = i0 + uint32_t(u) * per;
                if (row < r1) {
                    const uint64_t i = uint64_t(row) * k + j;
                    rv[u] = lane_load<V, NT>(a.r + i);
                    qv[u] = lane_load<V, NT>(a.q + i);
                    pv[u] = PREC ? a.dinv[row] : T(1);
                }
            }
#pragma unroll
            for (int u = 0; u < kMultiU; ++u) {
                const uint32_t row = i0 + uint32_t(u) * per;
                if (row < r1) {
                    const uint64_t i = uint64_t(row) * k + j;
#pragma unroll
                    for (int c = 0; c < V; ++c) {
                        const T ri = add_rn(rv[u].v[c], mul_rn(-alpha[c], qv[u].v[c]));
                        const T hi = PREC ? mul_rn(pv[u], ri) : ri;
                        rv[u].v[c] = act[c] ? ri : rv[u].v[c];
                        prh[c] += ri * hi;
                        prr[c] += ri * ri;
                    }
                    lane_store<V, NT>(a.r + i, rv[u].v);
                }
            }
        }
    }
    column_partials_v<V>(prh, k, lanes, lds, a.part_rh + size_t(L) * k, a.done, a.stop);
    column_partials_v<V>(prr, k, lanes, lds, a.part_rr + size_t(L) * k, a.done, a.stop);
}

// Re-opens the columns flagged in `again` (their loop stopped on the stopping
// test; the host has lowered their thresholds).  alpha = 0: the direction
// step that stopped has applied the pending x -= alpha d.  The next one
// recomputes rho and err from the same partials and, the test failing now,
// goes on as it would have with this threshold from the start.
template <typename T>
__global__ void k_m_reopen(MultiArgs<T> a, const int32_t* again) {
    const uint32_t j = threadIdx.x;
    if (j >= a.k || !again[j]) return;
    a.alpha[j] = T(0);
    a.stop[j] = 0;
    a.done[j] = 0;
}

// ---------------------------------------------------- layout / refinement

// interleaved[i*k + j] = colmajor[j*n + i] and back, in tiles of kLayoutRows
// rows through LDS (rows padded to an odd length): runs of 512 bytes per
// column on one side, whole rows on the other.  For 2.25 M rows and 32 columns
// 228 us in and 202 us out (368 and 557 us with a group of lanes per row).
constexpr uint32_t kLayoutRows = 64;

template <typename T, bool IN>
__global__ __launch_bounds__(kBlock) void k_layout(uint32_t n, uint32_t k,
                                                   const T* __restrict__ src,
                                                   T* __restrict__ dst, int32_t* nonzero) {
    __shared__ T tile[kLayoutRows * 33];
    const uint32_t ld = k | 1u;
    bool nz = false;
    const uint64_t step = uint64_t(gridDim.x) * kLayoutRows;
    for (uint64_t r0 = uint64_t(blockIdx.x) * kLayoutRows; r0 < n; r0 += step) {
        const uint32_t rows = n - r0 < kLayoutRows ? uint32_t(n - r0) : kLayoutRows;
        const uint32_t row = threadIdx.x % kLayoutRows;
        __syncthreads();  // the previous tile has been written
        if (IN) {
            for (uint32_t j = threadIdx.x / kLayoutRows; j < k; j += kBlock / kLayoutRows)
                if (row < rows) {
                    const T v = src[uint64_t(j) * n + r0 + row];
                    tile[row * ld + j] = v;
                    nz |= !(v == T(0));
                }
        } else {
            for (uint32_t e = threadIdx.x; e < rows * k; e += kBlock)
                tile[(e / k) * ld + e % k] = src[r0 * k + e];
        }
        __syncthreads();
        if (IN) {
            for (uint32_t e = threadIdx.x; e < rows * k; e += kBlock)
                dst[r0 * k + e] = tile[(e / k) * ld + e % k];
        } else {
            for (uint32_t j = threadIdx.x / kLayoutRows; j < k; j += kBlock / kLayoutRows)
                if (row < rows) dst[uint64_t(j) * n + r0 + row] = tile[row * ld + j];
        }
    }
    if (IN && nonzero && nz) *nonzero = 1;  // every writer stores 1
}

// R = B - A X (FP64, interleaved), per-column partial |r|^2 and |b|^2.
template <int G, int V>
__global__ __launch_bounds__(kBlock) void k_m_residual64(MultiArgs<double> a) {
    __shared__ double lds[kWavesPerBlock * 32];
    const uint32_t L = xcd_logical_block(blockIdx.x, gridDim.x);
    const uint32_t k = a.k;
    double prr[V], pbb[V];
#pragma unroll
    for (int c = 0; c < V; ++c) prr[c] = pbb[c] = 0.0;
    auto pre = [&](uint32_t row, uint32_t j) {
        return lane_load<V>(a.b + uint64_t(row) * k + j);
    };
    auto fin = [&](uint32_t row, uint32_t j, const double (&s)[V], const Lane<V, double>& b) {
        double r[V];
#pragma unroll
        for (int c = 0; c < V; ++c) {
            r[c] = b.v[c] - s[c];
            prr[c] += r[c] * r[c];
            pbb[c] += b.v[c] * b.v[c];
        }
        lane_store<V>(a.r + uint64_t(row) * k + j, r);
    };
    spmm_rows_v<G / V, V>(a.m, k, L, a.rp, a.ci, a.val, a.x, pre, fin);
    column_partials_v<V>(prr, k, G / V, lds, a.part_rr + size_t(L) * k);
    column_partials_v<V>(pbb, k, G / V, lds, a.part_bb + size_t(L) * k);
}

// k_m_residual64's epilogue for the stream engine: r = b - A x, partials of
// r.r and b.b per column.
template <int K>
struct MultiResidualEpilogue {
    const MultiArgs<double>& a;
    double (&prr)[K];
    double (&pbb)[K];
    struct PV {
        double b[K];
    };
    __device__ __forceinline__ PV pre(uint32_t row) const {
        PV p;
#pragma unroll
        for (int j = 0; j < K; ++j) p.b[j] = a.b[uint64_t(row) * K + j];
        return p;
    }
    __device__ __forceinline__ void done(uint32_t row, const double (&s)[K], const PV& pv) {
#pragma unroll
        for (int j = 0; j < K; ++j) {
            const double bi = pv.b[j];
            const double ri = bi - s[j];
            a.r[uint64_t(row) * K + j] = ri;
            prr[j] += ri * ri;
            pbb[j] += bi * bi;
        }
    }
};

template <int K, bool D16>
__global__ __launch_bounds__(kBlock) void k_m_residual64_stream(MultiArgs<double> a) {
    using Eng = MultiStreamEngine<K, kMultiStreamE, D16>;
    __shared__ double stage[kWavesPerBlock * Eng::kStage];
    __shared__ double red[kWavesPerBlock * K];
    const uint32_t L = xcd_logical_block(blockIdx.x, gridDim.x);
    bool act[K];
    double prr[K], pbb[K];
#pragma unroll
    for (int j = 0; j < K; ++j) {
        act[j] = true;
        prr[j] = pbb[j] = 0.0;
    }
    MultiResidualEpilogue<K> epi{a, prr, pbb};
    Eng::run(a.m, a.sp, L, a.rp, a.cols, a.val, a.x, act, stage, epi);
    stream_partials<K>(prr, red, a.part_rr + size_t(L) * K);
    stream_partials<K>(pbb, red, a.part_bb + size_t(L) * K);
}

__global__ __launch_bounds__(kBlock) void k_m_norms64(MultiArgs<double> a) {
    __shared__ double lds[kWavesPerBlock];
    const uint32_t j = blockIdx.x;
    const double rr = col_sum(a.part_rr, a.Pdq, a.k, j, lds);
    const double bb = col_sum(a.part_bb, a.Pdq, a.k, j, lds);
    if (threadIdx.x == 0) {
        a.err[j] = rr;
        a.bb[j] = bb;
    }
}

// b32 = float(r64 * scale[j]); x32 = 0
__global__ __launch_bounds__(kBlock) void k_m_scale_cast(MultiArgs<double> a64,
                                                         MultiArgs<float> a32,
                                                         const double* scale) {
    const uint32_t L = xcd_logical_block(blockIdx.x, gridDim.x);
    const uint32_t k = a64.k, G = a64.G;
    const uint32_t g = threadIdx.x / G, j = threadIdx.x % G;
    if (j >= k) return;
    const double sj = scale[j];
    uint32_t r0, r1;
    block_rows(a64.m, a64.rows_per_block, L, r0, r1);
    for (uint32_t row = r0 + g; row < r1; row += kBlock / G) {
        const uint64_t i = uint64_t(row) * k + j;
        const_cast<float*>(a32.b)[i] = float(a64.r[i] * sj);
        a32.x[i] = 0.0f;
    }
}

__global__ __launch_bounds__(kBlock) void k_m_ir_update(MultiArgs<double> a64,
                                                        MultiArgs<float> a32,
                                                        const double* unscale) {
    const uint32_t L = xcd_logical_block(blockIdx.x, gridDim.x);
    const uint32_t k = a64.k, G = a64.G;
    const uint32_t g = threadIdx.x / G, j = threadIdx.x % G;
    if (j >= k || a32.skip[j]) return;
    const double uj = unscale[j];
    uint32_t r0, r1;
    block_rows(a64.m, a64.rows_per_block, L, r0, r1);
    for (uint32_t row = r0 + g; row < r1; row += kBlock / G) {
        const uint64_t i = uint64_t(row) * k + j;
        a64.x[i] = a64.x[i] + uj * double(a32.x[i]);
    }
}

// ------------------------------------------------------------- launchers

#define NLHIP_G_SWITCH(G_, CALL)                         \
    switch (G_) { /* k > kMultiStreamMaxK */             \
        case 8: { constexpr int G = 8; CALL; } break;    \
        case 16: { constexpr int G = 16; CALL; } break;  \
        case 32: { constexpr int G = 32; CALL; } break;  \
        default: return hipErrorInvalidValue;            \
    }

// K = k (1 .. kMultiStreamMaxK) and D16 as constants for the stream kernels.
#define NLHIP_KD_SWITCH(K_, D16_, CALL)                                                   \
    switch (K_) {                                                                          \
        case 1: { constexpr int K = 1; if (D16_) { constexpr bool D16 = true; CALL; }      \
                  else { constexpr bool D16 = false; CALL; } } break;                      \
        case 2: { constexpr int K = 2; if (D16_) { constexpr bool D16 = true; CALL; }      \
                  else { constexpr bool D16 = false; CALL; } } break;                      \
        case 3: { constexpr int K = 3; if (D16_) { constexpr bool D16 = true; CALL; }      \
                  else { constexpr bool D16 = false; CALL; } } break;                      \
        case 4: { constexpr int K = 4; if (D16_) { constexpr bool D16 = true; CALL; }      \
                  else { constexpr bool D16 = false; CALL; } } break;                      \
        default: return hipErrorInvalidValue;                                              \
    }
static_assert(kMultiStreamMaxK == 4, "one case per k up to kMultiStreamMaxK");

namespace {
template <typename T>
hipError_t stream_spmm_kernel(uint32_t k, bool d16, const void*& f) {
    NLHIP_KD_SWITCH(k, d16, (f = reinterpret_cast<const void*>(&k_m_spmm_stream<K, D16, T>)));
    return hipSuccess;
}
}  // namespace

template <typename T>
uint32_t multi_rows_per_cu(uint32_t k) {
    uint32_t G = 8;
    while (G < k) G <<= 1;
    const bool v2 = multi_two_cols<T>(k);
    const void* f = nullptr;
    auto pick = [&] {
        NLHIP_G_SWITCH(G, (f = v2 ? reinterpret_cast<const void*>(&k_m_spmm<G, two_cols_v<G>(), T>)
                                  : reinterpret_cast<const void*>(&k_m_spmm<G, 1, T>)));
        return hipSuccess;
    };
    int per = 0;
    if (pick() != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, f, kBlock, 0) != hipSuccess || per < 1)
        return 1;
    return uint32_t(per);
}
template uint32_t multi_rows_per_cu<double>(uint32_t);
template uint32_t multi_rows_per_cu<float>(uint32_t);

// Sized for the SpMM step, the launch of every iteration; the start and the
// residual (once per solve, more registers for their epilogues at large k)
// may hold fewer workgroups per CU and then run a second, partial round.
template <typename T>
uint32_t multi_stream_per_cu(uint32_t k, bool d16) {
    const void* f = nullptr;
    int per = 0;
    if (stream_spmm_kernel<T>(k, d16, f) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, f, kBlock, 0) != hipSuccess || per < 1)
        return 1;
    return uint32_t(per);
}
template uint32_t multi_stream_per_cu<double>(uint32_t, bool);
template uint32_t multi_stream_per_cu<float>(uint32_t, bool);

template <typename T>
hipError_t multi_start(const MultiArgs<T>& a, bool precond, T eps, int max_iter, hipStream_t s) {
    const bool d16 = a.cols.ci16 != nullptr;
    const bool v2 = multi_two_cols<T>(a.k);
    if (a.sp && precond) {
        NLHIP_KD_SWITCH(a.k, d16, (k_m_init_stream<K, D16, T, true><<<a.Pdq, kBlock, 0, s>>>(a)));
    } else if (a.sp) {
        NLHIP_KD_SWITCH(a.k, d16, (k_m_init_stream<K, D16, T, false><<<a.Pdq, kBlock, 0, s>>>(a)));
    } else if (precond) {
        NLHIP_G_SWITCH(a.G, (v2 ? k_m_init<G, two_cols_v<G>(), T, true><<<a.P, kBlock, 0, s>>>(a)
                               : k_m_init<G, 1, T, true><<<a.P, kBlock, 0, s>>>(a)));
    } else {
        NLHIP_G_SWITCH(a.G, (v2 ? k_m_init<G, two_cols_v<G>(), T, false><<<a.P, kBlock, 0, s>>>(a)
                               : k_m_init<G, 1, T, false><<<a.P, kBlock, 0, s>>>(a)));
    }
    k_m_sys_init<T><<<a.k, kBlock, 0, s>>>(a, eps, max_iter);
    return hipGetLastError();
}

template <typename T, bool PREC>
static hipError_t multi_iteration_p(const MultiArgs<T>& a, int max_iter, hipStream_t s) {
    if (a.sp) {
        switch (a.k) {
            case 1: k_m_dir_few<1, T, PREC><<<a.P, kBlock, 0, s>>>(a, max_iter); break;
            case 2: k_m_dir_few<2, T, PREC><<<a.P, kBlock, 0, s>>>(a, max_iter); break;
            case 3: k_m_dir_few<3, T, PREC><<<a.P, kBlock, 0, s>>>(a, max_iter); break;
            default: k_m_dir_few<4, T, PREC><<<a.P, kBlock, 0, s>>>(a, max_iter); break;
        }
        NLHIP_KD_SWITCH(a.k, a.cols.ci16 != nullptr,
                        (k_m_spmm_stream<K, D16, T><<<a.Pdq, kBlock, 0, s>>>(a)));
        switch (a.k) {
            case 1: k_m_update_few<1, T, PREC><<<a.P, kBlock, 0, s>>>(a); break;
            case 2: k_m_update_few<2, T, PREC><<<a.P, kBlock, 0, s>>>(a); break;
            case 3: k_m_update_few<3, T, PREC><<<a.P, kBlock, 0, s>>>(a); break;
            default: k_m_update_few<4, T, PREC><<<a.P, kBlock, 0, s>>>(a); break;
        }
        return hipGetLastError();
    }
    const bool v2 = multi_two_cols<T>(a.k);
    k_m_beta<T><<<a.k, kBlock, 0, s>>>(a, max_iter);
    const bool nt = multi_streamed<T>(a.m, a.k);
    if (v2) (nt ? k_m_dir<2, true, T, PREC> : k_m_dir<2, false, T, PREC>)<<<a.P, kBlock, 0, s>>>(a);
    else (nt ? k_m_dir<1, true, T, PREC> : k_m_dir<1, false, T, PREC>)<<<a.P, kBlock, 0, s>>>(a);
    NLHIP_G_SWITCH(a.G, (v2 ? k_m_spmm<G, two_cols_v<G>(), T><<<a.P, kBlock, 0, s>>>(a)
                           : k_m_spmm<G, 1, T><<<a.P, kBlock, 0, s>>>(a)));
    k_m_alpha<T><<<a.k, kBlock, 0, s>>>(a);
    if (v2)
        (nt ? k_m_update<2, true, T, PREC> : k_m_update<2, false, T, PREC>)<<<a.P, kBlock, 0, s>>>(a);
    else
        (nt ? k_m_update<1, true, T, PREC> : k_m_update<1, false, T, PREC>)<<<a.P, kBlock, 0, s>>>(a);
    return hipGetLastError();
}

template <typename T>
hipError_t multi_iteration(const MultiArgs<T>& a, bool precond, int max_iter, hipStream_t s) {
    return precond ? multi_iteration_p<T, true>(a, max_iter, s)
                   : multi_iteration_p<T, false>(a, max_iter, s);
}

template <typename T>
hipError_t multi_layout(uint32_t n, uint32_t k, const T* src, T* dst, bool to_interleaved,
                        hipStream_t s, int32_t* nonzero) {
    if (k == 0 || k > 32) return hipErrorInvalidValue;
    const uint64_t tiles = (uint64_t(n) + kLayoutRows - 1) / kLayoutRows;
    const uint32_t g = uint32_t(tiles < 16384 ? (tiles ? tiles : 1) : 16384);
    if (to_interleaved) k_layout<T, true><<<g, kBlock, 0, s>>>(n, k, src, dst, nonzero);
    else k_layout<T, false><<<g, kBlock, 0, s>>>(n, k, src, dst, nullptr);
    return hipGetLastError();
}

hipError_t multi_reopen(const MultiArgs<double>& a, const int32_t* again, hipStream_t s) {
    k_m_reopen<double><<<1, kWave, 0, s>>>(a, again);
    return hipGetLastError();
}

hipError_t multi_residual64(const MultiArgs<double>& a, hipStream_t s) {
    const bool v2 = multi_two_cols<double>(a.k);
    if (a.sp) {
        NLHIP_KD_SWITCH(a.k, a.cols.ci16 != nullptr,
                        (k_m_residual64_stream<K, D16><<<a.Pdq, kBlock, 0, s>>>(a)));
    } else {
        NLHIP_G_SWITCH(a.G, (v2 ? k_m_residual64<G, two_cols_v<G>()><<<a.P, kBlock, 0, s>>>(a)
                               : k_m_residual64<G, 1><<<a.P, kBlock, 0, s>>>(a)));
    }
    k_m_norms64<<<a.k, kBlock, 0, s>>>(a);
    return hipGetLastError();
}

hipError_t multi_scale_cast(const MultiArgs<double>& a64, const MultiArgs<float>& a32,
                            const double* scale, hipStream_t s) {
    k_m_scale_cast<<<a64.P, kBlock, 0, s>>>(a64, a32, scale);
    return hipGetLastError();
}

hipError_t multi_ir_update(const MultiArgs<double>& a64, const MultiArgs<float>& a32,
                           const double* unscale, hipStream_t s) {
    k_m_ir_update<<<a64.P, kBlock, 0, s>>>(a64, a32, unscale);
    return hipGetLastError();
}

// dst[:, j] = src[:, j] for the columns j with flag[j] (interleaved n x k).
__global__ __launch_bounds__(kBlock) void k_m_copy_cols(uint32_t n, uint32_t k,
                                                        double* __restrict__ dst,
                                                        const double* __restrict__ src,
                                                        const int32_t* __restrict__ flag) {
    const uint64_t nk = uint64_t(n) * k;
    const uint64_t stride = uint64_t(gridDim.x) * kBlock;
    uint64_t i = uint64_t(blockIdx.x) * kBlock + threadIdx.x;
    uint32_t j = uint32_t(i % k);
    const uint32_t dj = uint32_t(stride % k);
    for (; i < nk; i += stride) {
        if (flag[j]) dst[i] = src[i];
        j += dj;
        j -= j >= k ? k : 0u;
    }
}

hipError_t multi_copy_cols(uint32_t n, uint32_t k, double* dst, const double* src,
                           const int32_t* flag, hipStream_t s) {
    const uint64_t nk = uint64_t(n) * k;
    if (nk == 0) return hipSuccess;
    const uint64_t g = (nk + kBlock - 1) / kBlock;
    k_m_copy_cols<<<uint32_t(g < 16384 ? g : 16384), kBlock, 0, s>>>(n, k, dst, src, flag);
    return hipGetLastError();
}

template hipError_t multi_start<double>(const MultiArgs<double>&, bool, double, int, hipStream_t);
template hipError_t multi_start<float>(const MultiArgs<float>&, bool, float, int, hipStream_t);
template hipError_t multi_iteration<double>(const MultiArgs<double>&, bool, int, hipStream_t);
template hipError_t multi_iteration<float>(const MultiArgs<float>&, bool, int, hipStream_t);
template hipError_t multi_layout<double>(uint32_t, uint32_t, const double*, double*, bool,
                                         hipStream_t, int32_t*);

}  // namespace nlhip
