// The fused PCG of k_cg.hip with many iterations per launch, for systems
// whose matrix (but for the ends of its longer rows) fits in the registers of
// the workgroups that are resident at once: below a few hundred thousand rows an iteration of three launches is
// all latency (14 us for 24 k rows, of which the bytes need one).
//
// Every logical workgroup L of the three launches (its 64-row tiles of the
// SpMV, its row range of the element-wise steps, its entry of the partial
// sums) becomes part of one physical workgroup, and every sum is formed in
// the order of the three launches, so iterates, scalars and iteration counts
// are theirs, bit for bit.  A lane keeps its row (or, for 2x2 blocks, its
// pair of rows) of the matrix and its rows' x, r, h, d and D^-1 in registers;
// what other workgroups read goes through memory with device-coherent
// accesses: the pairs (d, h) of every row, q where a row's SpMV lane is not
// its element-wise lane, and the partial sums.
//
// An iteration has two grid-wide waits instead of three launch boundaries:
// the direction step needs none, because a lane that gathers column c takes
// the pair (d, h) of the previous iteration and forms d = beta d + h itself,
// the same multiply and add as the owner's.  Each wait is the reduction that
// the step needs anyway: every workgroup writes its partial sums, tagged with
// the iteration, behind its other stores, and polls those of all (with
// counters, and the sums read behind them, an iteration at 1,150 rows took
// 9.0 us instead of 4.3).
//
// The launch is not cooperative: it uses at most one workgroup of 512 threads
// per CU, which one always holds, one such launch runs at a time in a process
// (GridTurn), and every wait is bounded.  A workgroup that gives up sets
// kPersistFail and leaves; the others then give up at the latest at the
// barrier before the solver's vectors, partials and status are written,
// which is complete for all or for none of them (grid_barrier.h; a wait that
// is given up between barriers sets the bit before the next one's count can
// be complete).  The caller continues with the three launches from the
// unchanged state, and keeps to them for a while (System::persist).
//
// LSCM systems, us per iteration, three launches -> this: 1,150 rows 8.2 ->
// 4.3; 8 k 14.6 -> 5.5; 24 k 14.2 -> 5.7; 60 k 13.7 -> 7.5; 100 k 17.1 -> 8.8;
// 201 k (2x2 blocks) 18.4 -> 11.1; 259 k 21.1 -> 12.2.
#include "dev_common.h"
#include "nlhip_kernels.h"

namespace nlhip {

namespace {

template <typename T>
__device__ __forceinline__ T ld_dev(const T* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void st_dev(T* p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// A barrier word in device memory (grid_barrier.h).
struct DeviceWord {
    uint32_t* p;
    __device__ __forceinline__ uint32_t load() const { return ld_dev(p); }
    __device__ __forceinline__ uint32_t add(uint32_t v) const {
        return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __device__ __forceinline__ uint32_t cas(uint32_t expected, uint32_t desired) const {
        __hip_atomic_compare_exchange_strong(p, &expected, desired, __ATOMIC_RELAXED,
                                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return expected;
    }
    __device__ __forceinline__ void pause() const { __builtin_amdgcn_s_sleep(1); }
};
// Every store of this wavefront has reached the device's point of coherence.
__device__ __forceinline__ void wait_stores() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// The (d, h) pairs: 16 bytes (FP64) or 8 (FP32) per row, device-coherent.
template <typename T>
struct Pairs;
template <>
struct Pairs<double> {
    using V4 = uint32_t __attribute__((ext_vector_type(4)));
    static constexpr int kSc1 = 16;  // cache policy of the buffer instructions: device scope
    static constexpr uint32_t kBytes = 16;
    __amdgpu_buffer_rsrc_t rs;
    __device__ Pairs(double* p, uint32_t n)
        : rs(__builtin_amdgcn_make_buffer_rsrc(p, 0, n * 16u, 0x00027000)) {}
    // of the row at byte offset o
    __device__ __forceinline__ void load(uint32_t o, double& d, double& h) const {
        const V4 v = __builtin_amdgcn_raw_buffer_load_b128(rs, o, 0, kSc1);
        d = __longlong_as_double((long long)((uint64_t(v.y) << 32) | v.x));
        h = __longlong_as_double((long long)((uint64_t(v.w) << 32) | v.z));
    }
    __device__ __forceinline__ void store(uint32_t o, double d, double h) const {
        const uint64_t a = uint64_t(__double_as_longlong(d)), b = uint64_t(__double_as_longlong(h));
        const V4 v = {uint32_t(a), uint32_t(a >> 32), uint32_t(b), uint32_t(b >> 32)};
        __builtin_amdgcn_raw_buffer_store_b128(v, rs, o, 0, kSc1);
    }
};
template <>
struct Pairs<float> {
    static constexpr uint32_t kBytes = 8;
    char* q;
    __device__ Pairs(float* p, uint32_t) : q(reinterpret_cast<char*>(p)) {}
    __device__ __forceinline__ void load(uint32_t o, float& d, float& h) const {
        const uint64_t v = ld_dev(reinterpret_cast<const uint64_t*>(q + o));
        d = __uint_as_float(uint32_t(v));
        h = __uint_as_float(uint32_t(v >> 32));
    }
    __device__ __forceinline__ void store(uint32_t o, float d, float h) const {
        st_dev(reinterpret_cast<uint64_t*>(q + o), (uint64_t(__float_as_uint(h)) << 32) | __float_as_uint(d));
    }
};

// A partial sum as other workgroups see it: two words, each one half of the
// value with the tag of its iteration, so that a reader needs no other flag.
template <typename T>
struct Tagged;
template <>
struct Tagged<double> {
    __device__ __forceinline__ static void put(uint64_t* s, double v, uint32_t tag) {
        const uint64_t b = uint64_t(__double_as_longlong(v)), t = uint64_t(tag) << 32;
        st_dev(s, t | uint32_t(b));
        st_dev(s + 1, t | (b >> 32));
    }
    __device__ __forceinline__ static bool get(const uint64_t* s, uint32_t tag, double& v) {
        const uint64_t a = ld_dev(s), b = ld_dev(s + 1);
        v = __longlong_as_double((long long)((b << 32) | uint32_t(a)));
        return uint32_t(a >> 32) == tag && uint32_t(b >> 32) == tag;
    }
};
template <>
struct Tagged<float> {
    __device__ __forceinline__ static void put(uint64_t* s, float v, uint32_t tag) {
        st_dev(s, (uint64_t(tag) << 32) | __float_as_uint(v));
    }
    __device__ __forceinline__ static bool get(const uint64_t* s, uint32_t tag, float& v) {
        const uint64_t a = ld_dev(s);
        v = __uint_as_float(uint32_t(a));
        return uint32_t(a >> 32) == tag;
    }
};

}  // namespace

// AW: wavefronts of a logical workgroup that hold rows (2 of 4 when it has at
// most 128 rows, else 4); E: element-wise rows per lane.  BLK: 2x2 blocks.
template <typename T, bool BLK, int AW, int E, int MAXT>
__global__ __launch_bounds__(MAXT) void k_cg_persist(CGArgs<T> a, CGPersist<T> p) {
    constexpr int W = BLK ? 8 : 16;        // entries (blocks) of a row kept in registers
    constexpr int NV = BLK ? 4 : 1;        // values per entry
    constexpr int NR = BLK ? 2 : 1;        // rows per lane
    constexpr int kMaxSub = MAXT / (64 * AW);
    __shared__ T s_wave[2][kMaxSub * AW];  // wavefront sums
    __shared__ T s_red[2][4];              // virtual wavefronts' sums
    __shared__ uint32_t s_ok;
    // the polls of a wait, at barriers and in sums: read where they are needed
    // (the loop has more scalars than scalar registers; held in registers they
    // cost 0.1 us per iteration)
    __shared__ uint32_t s_polls[2];
    if (blockIdx.x % p.shape.stride) return;
    CGStatus<T>* st = a.st;
    if (st->done) return;  // written by an earlier launch
    const uint32_t wg = blockIdx.x / p.shape.stride, wgs = p.shape.wgs;
    const uint32_t gw = p.shape.stride > 1 ? wg : xcd_logical_block(wg, wgs);
    const uint32_t group = p.shape.stride > 1 ? 0u : wg % kNumXcd;
    const uint32_t gsize = p.shape.stride > 1 ? wgs : (wgs - group + kNumXcd - 1) / kNumXcd;
    const uint32_t ngroups = p.shape.stride > 1 ? 1u : (wgs < kNumXcd ? wgs : kNumXcd);
    const uint32_t subs = blockDim.x / (64 * AW);
    const uint32_t sub = threadIdx.x / (64 * AW), tid = threadIdx.x % (64 * AW);
    const int lane = threadIdx.x & (kWave - 1);
    const uint32_t w = tid / kWave;
    const uint32_t L = gw * subs + sub;
    if (threadIdx.x == 0) {
        s_polls[0] = p.polls;
        s_polls[1] = p.sum_polls;
    }
    const bool first_wave = threadIdx.x < uint32_t(kWave);
    const Pairs<T> dh(p.dh, a.m);

    // the lane's row(s) of the matrix
    const uint32_t trows = BLK ? a.m / 2 : a.m;
    const uint64_t t64 = (uint64_t(L) * a.sps + w) * 64 + uint32_t(lane);
    const bool have = L < a.P && w < a.sps && t64 < trows;
    const uint32_t row = have ? uint32_t(t64) : 0u;
    uint32_t jb = 0, je = 0;
    if (have) {
        jb = a.rp[row];
        je = a.rp[row + 1];
    }
    auto column = [&](uint32_t j) {
        return a.cols.ci16 ? a.cols.segb[j >> kSegShift] + uint32_t(a.cols.ci16[j])
                           : a.cols.ci[j];
    };
    auto value = [&](uint32_t j, T (&v)[NV]) {
        if constexpr (BLK) {
            const T *u = a.val + block_upper<T>(j), *l = a.val + block_lower<T>(j);
            v[0] = u[0];
            v[1] = u[1];
            v[2] = l[0];
            v[3] = l[1];
        } else {
            v[0] = a.val[j];
        }
    };
    uint32_t c[W];  // byte offsets of the columns' pairs
    T av[W][NV];
    uint32_t most = 0;  // longest kept row of the wavefront
    constexpr uint32_t kPair = Pairs<T>::kBytes;
#pragma unroll
    for (int u = 0; u < W; ++u) {
        c[u] = 0;
#pragma unroll
        for (int v = 0; v < NV; ++v) av[u][v] = T(0);
        if (jb + uint32_t(u) < je) {
            c[u] = NR * kPair * column(jb + uint32_t(u));
            value(jb + uint32_t(u), av[u]);
        }
        if (__ballot(jb + uint32_t(u) < je)) most = uint32_t(u) + 1u;
    }
    const uint32_t len = je - jb;
    // rows for the launches (persist_longest): no state has been written, and
    // without this workgroup no barrier passes
    if (__syncthreads_or(len > p.longest)) {
        if (threadIdx.x == 0)
            __hip_atomic_fetch_or(p.bar, kPersistFail | kPersistLong, __ATOMIC_RELAXED,
                                  __HIP_MEMORY_SCOPE_AGENT);
        return;
    }

    // the lane's rows of the element-wise steps
    uint32_t r0 = 0, r1 = 0;
    if (L < a.P) block_row_range(a.m, a.chunk, L, r0, r1);
    uint32_t ri[E];
    bool in[E];
    T x[E], r[E], h[E], d[E], dinv[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        ri[e] = r0 + tid + uint32_t(e * kBlock);
        in[e] = ri[e] < r1;
        x[e] = r[e] = h[e] = d[e] = T(0);
        dinv[e] = T(1);  // no preconditioner: h = 1 r
        if (in[e]) {
            x[e] = a.x[ri[e]];
            r[e] = a.r[ri[e]];
            h[e] = a.h[ri[e]];
            d[e] = a.d[ri[e]];
            if (a.dinv) dinv[e] = a.dinv[ri[e]];
        }
    }
    // an SpMV row is the lane's own element-wise row: q stays in a register
    const bool same = !BLK && E == 1 && a.chunk == 64u * a.sps;

    int it = st->iter_a, iter_b = st->iter_b;
    T rho_prev = st->rho_prev, alpha = st->alpha, beta = st->beta, old_rho = st->rho,
      old_err = st->err;
    const T thresh = st->thresh;
    const int max_iter = st->max_iter;
    // Grid barrier behind the stores of every wavefront (the first and the
    // last of a launch).
    uint32_t epoch = 0;
    auto barrier = [&] {
        ++epoch;
        wait_stores();
        __syncthreads();
        if (threadIdx.x == 0) {
            const DeviceWord root{p.bar};
            barrier_arrive(DeviceWord{p.bar + kPersistBarPad * (1u + group)}, root, gsize, epoch);
            s_ok = barrier_wait(root, ngroups, epoch, s_polls[0]) ? 1u : 0u;
        }
        __syncthreads();
        return s_ok != 0;
    };
    // The N sums of a step over the whole grid, in the order of the three
    // launches: each logical workgroup's wavefront sums in order into its
    // slot, then (reduce_partials) virtual thread 64 v + lane, v < 4, adds the
    // slots 64 v + lane + 256 k, each virtual wavefront is combined by the
    // butterfly, and the four in order.  A workgroup's slots are written
    // behind its other stores, so whoever has read all slots may read what
    // the step stored: the wait for the slots is the grid barrier.
    auto grid_sum = [&](auto n, const T (&mine)[2], uint32_t which, uint32_t tag, T (&out)[2]) {
        constexpr int N = decltype(n)::value;
#pragma unroll
        for (int q = 0; q < N; ++q) {
            const T v = group_sum<kWave>(mine[q]);
            if (lane == 0) s_wave[q][sub * AW + w] = v;
        }
        if (threadIdx.x == 0) s_ok = 1;
        wait_stores();
        __syncthreads();
        constexpr uint32_t kWords = sizeof(T) / 4;
        if (threadIdx.x < subs * N) {
            const uint32_t q = threadIdx.x / subs, l = threadIdx.x % subs;
            if (gw * subs + l < a.P) {
                T t = s_wave[q][l * AW];
#pragma unroll
                for (int y = 1; y < AW; ++y) t += s_wave[q][l * AW + y];
                // the wavefronts without rows add +0
                if (AW < kWavesPerBlock) t += T(0);
                Tagged<T>::put(p.slots + kWords * (size_t(which + q) * a.P + gw * subs + l), t,
                               tag);
            }
        }
        const uint32_t nw = blockDim.x / kWave;
        for (uint32_t v = threadIdx.x / kWave; v < 4; v += nw) {
            T s[N];
#pragma unroll
            for (int q = 0; q < N; ++q) s[q] = T(0);
            for (uint32_t k = 64u * v; k < a.P; k += kBlock) {
                const uint32_t i = k + uint32_t(lane);
                T t[N];
                bool good = false;
                for (uint32_t polls = 0;; ++polls) {
                    good = true;
#pragma unroll
                    for (int q = 0; q < N; ++q) {
                        t[q] = T(0);
                        if (i < a.P)
                            good &= Tagged<T>::get(p.slots + kWords * (size_t(which + q) * a.P + i),
                                                   tag, t[q]);
                    }
                    good = __all(good);
                    if (good) break;
                    if (polls >= *static_cast<volatile uint32_t*>(&s_polls[1])) {
                        s_ok = 0;
                        break;
                    }
                }
                if (i < a.P) {
#pragma unroll
                    for (int q = 0; q < N; ++q) s[q] += t[q];
                }
            }
#pragma unroll
            for (int q = 0; q < N; ++q) {
                s[q] = group_sum<kWave>(s[q]);
                if (lane == 0) s_red[q][v] = s[q];
            }
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < N; ++q)
            out[q] = ((s_red[q][0] + s_red[q][1]) + s_red[q][2]) + s_red[q][3];
        if (s_ok) return true;
        if (threadIdx.x == 0)
            __hip_atomic_fetch_or(p.bar, kPersistFail, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return false;
    };
    using N1 = std::integral_constant<int, 1>;
    using N2 = std::integral_constant<int, 2>;

    // the pairs of this state; behind the barrier every workgroup has read the
    // status, so one of them may write it
#pragma unroll
    for (int e = 0; e < E; ++e)
        if (in[e]) dh.store(kPair * ri[e], d[e], h[e]);
    if (!barrier()) return;
    // no polls at all (a test): one sum is missing, whoever else polls first
    if (p.sum_polls == 0 && gw == 0) {
        if (threadIdx.x == 0)
            __hip_atomic_fetch_or(p.bar, kPersistFail, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return;
    }
    // r.h and r.r of the current state, from the previous launch's partials
    for (uint32_t v = threadIdx.x / kWave; v < 4; v += blockDim.x / kWave) {
        T s0 = T(0), s1 = T(0);
        for (uint32_t i = 64u * v + uint32_t(lane); i < a.P; i += kBlock) {
            s0 += a.part_rh[i];
            s1 += a.part_rr[i];
        }
        s0 = group_sum<kWave>(s0);
        s1 = group_sum<kWave>(s1);
        if (lane == 0) {
            s_red[0][v] = s0;
            s_red[1][v] = s1;
        }
    }
    __syncthreads();
    T rho = ((s_red[0][0] + s_red[0][1]) + s_red[0][2]) + s_red[0][3];
    T err = ((s_red[1][0] + s_red[1][1]) + s_red[1][2]) + s_red[1][3];
    uint32_t count = 0;
    for (;;) {
        const bool stop = !(err > thresh) || it >= max_iter;
        if (stop || count == p.n_iter) {
            if (!barrier()) return;  // every workgroup is here, or none writes
            // write the state back: the stopping direction step applies the
            // pending update of x, otherwise it stays pending (alpha, d)
            const bool upd = stop && it > 0;
#pragma unroll
            for (int e = 0; e < E; ++e)
                if (in[e]) {
                    a.x[ri[e]] = upd ? add_rn(x[e], mul_rn(-alpha, d[e])) : x[e];
                    if (count) {
                        a.r[ri[e]] = r[e];
                        a.h[ri[e]] = h[e];
                        a.d[ri[e]] = d[e];
                    }
                }
            if (count && first_wave && uint32_t(lane) < subs &&
                gw * subs + uint32_t(lane) < a.P) {
                const uint32_t l = gw * subs + uint32_t(lane);
                constexpr uint32_t kWords = sizeof(T) / 4;
                T v0, v1;
                Tagged<T>::get(p.slots + kWords * (size_t(a.P) + l), count, v0);
                Tagged<T>::get(p.slots + kWords * (2 * size_t(a.P) + l), count, v1);
                a.part_rh[l] = v0;
                a.part_rr[l] = v1;
            }
            if (gw == 0 && threadIdx.x == 0) {
                st->iter_a = it;
                st->iter_b = iter_b;
                st->rho_prev = rho_prev;
                st->alpha = alpha;
                st->beta = beta;
                st->rho = stop ? rho : old_rho;
                st->err = stop ? err : old_err;
                if (stop) {
                    st->iters = it;
                    st->stop = 1;
                    __hip_atomic_store(&st->done, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
            return;
        }
        // direction
        const bool first = it == 0;
        beta = first ? T(0) : rho / rho_prev;
        old_rho = rho;
        old_err = err;
        iter_b = it;
        auto dir = [&](T dv, T hv) { return first ? hv : add_rn(mul_rn(beta, dv), hv); };
#pragma unroll
        for (int e = 0; e < E; ++e) {
            if (!first) x[e] = add_rn(x[e], mul_rn(-alpha, d[e]));
            d[e] = dir(d[e], h[e]);
        }
        // SpMV: q = A d, each row's products added left to right
        T acc[NR], dr[NR];
#pragma unroll
        for (int q = 0; q < NR; ++q) acc[q] = dr[q] = T(0);
        if (have) {
            T gd[NR], gh[NR];
#pragma unroll
            for (int q = 0; q < NR; ++q)
                dh.load(kPair * (NR * row + uint32_t(q)), gd[q], gh[q]);
            constexpr int G = BLK ? 4 : W;  // gathers in flight
#pragma unroll
            for (int u0 = 0; u0 < W; u0 += G) {
                if (uint32_t(u0) >= most) break;
                T d_[G][NR], h_[G][NR];
#pragma unroll
                for (int u = 0; u < G; ++u)  // past the row's end: row 0's pair, not used
#pragma unroll
                    for (int q = 0; q < NR; ++q)
                        dh.load(c[u0 + u] + kPair * uint32_t(q), d_[u][q], h_[u][q]);
#pragma unroll
                for (int u = 0; u < G; ++u) {
                    const bool on = uint32_t(u0 + u) < len;
                    T xv[NR];
#pragma unroll
                    for (int q = 0; q < NR; ++q) xv[q] = dir(d_[u][q], h_[u][q]);
#pragma unroll
                    for (int q = 0; q < NR; ++q)
#pragma unroll
                        for (int y = 0; y < NR; ++y) {
                            const T t = add_rn(acc[q], mul_rn(av[u0 + u][q * NR + y], xv[y]));
                            acc[q] = on ? t : acc[q];
                        }
                }
            }
            // the rest of a longer row, an entry at a time
            for (uint32_t j = jb + uint32_t(W); j < je; ++j) {
                const uint32_t cj = NR * kPair * column(j);
                T v[NV], xv[NR];
                value(j, v);
#pragma unroll
                for (int q = 0; q < NR; ++q) {
                    T dv, hv;
                    dh.load(cj + kPair * uint32_t(q), dv, hv);
                    xv[q] = dir(dv, hv);
                }
#pragma unroll
                for (int q = 0; q < NR; ++q)
#pragma unroll
                    for (int y = 0; y < NR; ++y) acc[q] = add_rn(acc[q], mul_rn(v[q * NR + y], xv[y]));
            }
#pragma unroll
            for (int q = 0; q < NR; ++q) {
                dr[q] = dir(gd[q], gh[q]);
                if (!same) st_dev(a.q + NR * row + uint32_t(q), acc[q]);
            }
        }
        T pdq[2] = {T(0), T(0)};
        if (have) {
#pragma unroll
            for (int q = 0; q < NR; ++q) pdq[0] += dr[q] * acc[q];
        }
        T red[2];
        if (!grid_sum(N1{}, pdq, 0, count + 1u, red)) return;
        // update
        alpha = rho / red[0];
        T pr[2] = {T(0), T(0)};
        T qv[E];
#pragma unroll
        for (int e = 0; e < E; ++e) {
            qv[e] = acc[0];
            if (!same && in[e]) qv[e] = ld_dev(a.q + ri[e]);
        }
#pragma unroll
        for (int e = 0; e < E; ++e)
            if (in[e]) {
                r[e] = add_rn(r[e], mul_rn(-alpha, qv[e]));
                h[e] = mul_rn(dinv[e], r[e]);
                dh.store(kPair * ri[e], d[e], h[e]);
                pr[0] += r[e] * h[e];
                pr[1] += r[e] * r[e];
            }
        rho_prev = rho;
        ++it;
        ++count;
        if (!grid_sum(N2{}, pr, 1, count, red)) return;
        rho = red[0];
        err = red[1];
    }
}

__global__ void k_persist_reset(uint32_t* bar, uint64_t* slots, uint32_t words) {
    if (threadIdx.x <= kNumXcd && blockIdx.x == 0) bar[kPersistBarPad * threadIdx.x] = 0;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < words;
         i += gridDim.x * blockDim.x)
        slots[i] = 0;
}

template <typename T>
static void (*persist_kernel(int kind))(CGArgs<T>, CGPersist<T>) {
    return kind == kPersistSmall  ? &k_cg_persist<T, false, 2, 1, 512>
           : kind == kPersistRows ? &k_cg_persist<T, false, 4, 1, 512>
                                  : &k_cg_persist<T, true, 4, 2, 512>;
}

template <typename T>
hipError_t cg_persist(const CGArgs<T>& a, const CGPersist<T>& p, hipStream_t s) {
    const PersistShape& h = p.shape;
    if (a.m == 0 || a.P == 0 || h.wgs == 0 || h.kind == 0) return hipErrorInvalidValue;
    const uint32_t grid = (h.wgs - 1) * h.stride + 1;
    k_persist_reset<<<4, kBlock, 0, s>>>(p.bar, p.slots, persist_slot_words<T>(a.P));
    persist_kernel<T>(h.kind)<<<grid, h.threads, 0, s>>>(a, p);
    return hipGetLastError();
}
template hipError_t cg_persist<double>(const CGArgs<double>&, const CGPersist<double>&,
                                       hipStream_t);
template hipError_t cg_persist<float>(const CGArgs<float>&, const CGPersist<float>&, hipStream_t);

// The launch of a system (kind 0: none): as many logical workgroups for the
// SpMV step as for the others, one of the engines with contiguous tiles
// (their twins with other chunk widths or column formats form the same sums),
// and no more workgroups than are resident.
template <typename T>
void cg_persist_plan(const CGArgs<T>& a, int code, uint64_t nnz, uint32_t cus, CGPersist<T>& p) {
    p.shape = PersistShape{};
    const bool blk = code >= 73;
    const bool known = (code >= 65 && code <= 68) || code == 71 || code == 72 ||
                       (blk && code <= 79 && code != 77);
    if (!known || a.Ps != a.P) return;
    p.shape = persist_resident(persist_shape(blk, a.P, a.sps, a.chunk, kNumXcd), cus, kNumXcd);
    p.longest = persist_longest(p.shape, nnz, a.m);
}
template void cg_persist_plan<double>(const CGArgs<double>&, int, uint64_t, uint32_t,
                                      CGPersist<double>&);
template void cg_persist_plan<float>(const CGArgs<float>&, int, uint64_t, uint32_t,
                                     CGPersist<float>&);

}  // namespace nlhip
