// Least-squares normal equations on the device: what a least-squares OpenNL
// context builds row by row (nlBegin/nlEnd(NL_ROW) with NL_LEAST_SQUARES,
// used by LSCM at src/lib/OGF/mesh/commands/mesh_grob_surface_commands.cpp:
// 724-779 and by the transport scripts through voxel_grob_transport_commands
// .cpp:236-279), with the same sums in the same order.
//
// Per row r (entries in order, variable v_e, coefficient a_e):
//   S_r = rhs_r - sum over locked entries of a_e x_{v_e}   (entry order)
//   for every ordered pair of free entries (e1, e2):  M[f(e1)][f(e2)] += a_e1 a_e2
//   for every free entry e:                           b[f(e)] += a_e S_r
// Rows are taken in order.  A dynamic row (OpenNL's NLRowColumn) stores the
// first contribution to an entry and adds the later ones; compression sorts
// each row by column.
//
// Device plan, by variable (rows, occurrences and columns per variable of at
// most kWaveMax): the entries of every free variable f1 are listed (counted,
// scattered, then sorted by entry index in registers), and one wavefront per
// variable walks the rows of those entries in order.  It meets the
// contributions to (f1, f2) in (row, e1, e2) order, the order in which the
// context adds them, and holds one matrix entry per lane; a first pass counts
// the columns, a second one sums and writes them sorted.  Nothing but the
// entry lists is stored between the passes.
// Otherwise (some variable is in more rows, or has more columns, or some row
// is longer): every row emits its pair products keyed by (f1, f2) in (row, e1,
// e2) order; a stable radix sort by key groups the contributions to each entry
// in that order, and one thread per entry adds them left to right; the
// right-hand side sorts the free entries by f (stable, so entry order) and
// one thread per free variable adds a_e S_r in that order.
// Separately rounded products and sums, as the host code.
//
// LSCM of a 1000^2 grid (2 M variables, 24 M entries, 72 M products): the
// sorted plan's 4.6 GB of keys, values and run heads cost 18 ms of kernels and,
// in calls that follow one another, ten times that for memory that is
// cleared before it is handed out again; the call takes 221 ms with it and
// 12.9 ms by variable (6.4 ms of kernels, 4.5 of them in k_ls_wave).
#include <algorithm>

#include <hipcub/hipcub.hpp>

#include "dev_common.h"
#include "nlhip_internal.h"

namespace nlhip {

namespace {

constexpr uint32_t kNone = 0xffffffffu;
constexpr uint32_t kWaveMax = kWave;  // of the plan by variable

__device__ __forceinline__ double sub_rn(double a, double b) { return __dsub_rn(a, b); }

// Input checks: row_ptr monotone and within the entry count, variables in
// range, coefficients, right-hand sides and values of locked variables
// finite.  Bits of *bad: 1 row_ptr, 2 variable, 4 non-finite value.
__global__ void k_ls_check(uint32_t nrows, uint32_t nvars, uint64_t nent, const uint32_t* rp,
                           const uint32_t* var, const double* coef, uint32_t nsys,
                           const double* row_rhs, const uint32_t* free_index,
                           const double* values, uint32_t* bad) {
    const uint32_t stride = gridDim.x * blockDim.x;
    uint32_t flags = 0;
    if (values)
        for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < nvars; v += stride)
            if (free_index[v] == kNone)
                for (uint32_t s = 0; s < nsys; ++s)
                    if (!isfinite(values[size_t(s) * nvars + v])) flags |= 4u;
    for (uint32_t r = blockIdx.x * blockDim.x + threadIdx.x; r < nrows; r += stride) {
        const uint32_t b = rp[r], e = rp[r + 1];
        if (b > e || e > nent) {
            flags |= 1u;
            continue;
        }
        for (uint32_t k = b; k < e; ++k) {
            if (var[k] >= nvars) flags |= 2u;
            if (!isfinite(coef[k])) flags |= 4u;
        }
        if (row_rhs)
            for (uint32_t s = 0; s < nsys; ++s)
                if (!isfinite(row_rhs[size_t(s) * nrows + r])) flags |= 4u;
    }
    if (flags) atomicOr(bad, flags);
}

// Totals over the rows that choose the plan.
struct LSTotals {
    unsigned long long pairs;  // pair products
    uint32_t max_row;          // entries of the longest row
    uint32_t max_occ;          // entries of the commonest variable
};

// Per row: S (nsys values), the number of pair products it emits, and the
// row of each of its entries; the totals.
__global__ void k_ls_rows(uint32_t nrows, const uint32_t* rp, const uint32_t* var,
                          const double* coef, const uint32_t* free_index, const double* values,
                          uint32_t nvars, uint32_t nsys, const double* row_rhs, double* S,
                          uint32_t* row_of, LSTotals* tot) {
    const uint32_t stride = gridDim.x * blockDim.x;
    unsigned long long pairs = 0;
    uint32_t longest = 0;
    for (uint32_t r = blockIdx.x * blockDim.x + threadIdx.x; r < nrows; r += stride) {
        const uint32_t b = rp[r], e = rp[r + 1];
        unsigned long long nf = 0;
        for (uint32_t k = b; k < e; ++k) {
            row_of[k] = r;
            nf += free_index[var[k]] != kNone ? 1u : 0u;
        }
        pairs += nf * nf;
        longest = longest > e - b ? longest : e - b;
        for (uint32_t s = 0; s < nsys; ++s) {
            double acc = row_rhs ? row_rhs[size_t(s) * nrows + r] : 0.0;
            for (uint32_t k = b; k < e; ++k) {
                const uint32_t v = var[k];
                if (free_index[v] == kNone)
                    acc = sub_rn(acc, mul_rn(coef[k], values ? values[size_t(s) * nvars + v] : 0.0));
            }
            S[size_t(s) * nrows + r] = acc;
        }
    }
    for (int o = kWave / 2; o > 0; o >>= 1) {
        pairs += __shfl_xor(pairs, o, kWave);
        const uint32_t l = __shfl_xor(longest, o, kWave);
        longest = longest > l ? longest : l;
    }
    if ((threadIdx.x & (kWave - 1)) == 0 && longest) {
        atomicAdd(&tot->pairs, pairs);
        atomicMax(&tot->max_row, longest);
    }
}

// Pair products of each row (the sorted plan).
__global__ void k_ls_npairs(uint32_t nrows, const uint32_t* rp, const uint32_t* var,
                            const uint32_t* free_index, uint64_t* npairs) {
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t r = blockIdx.x * blockDim.x + threadIdx.x; r < nrows; r += stride) {
        uint64_t nf = 0;
        for (uint32_t k = rp[r]; k < rp[r + 1]; ++k)
            nf += free_index[var[k]] != kNone ? 1u : 0u;
        npairs[r] = nf * nf;
    }
}

// Pair products of row r at pair_off[r]: key f1 << bits | f2, value a1 a2,
// in (e1, e2) order.
__global__ void k_ls_pairs(uint32_t nrows, const uint32_t* rp, const uint32_t* var,
                           const double* coef, const uint32_t* free_index,
                           const uint64_t* pair_off, uint32_t bits, uint64_t* keys,
                           double* vals) {
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t r = blockIdx.x * blockDim.x + threadIdx.x; r < nrows; r += stride) {
        const uint32_t b = rp[r], e = rp[r + 1];
        uint64_t o = pair_off[r];
        for (uint32_t k1 = b; k1 < e; ++k1) {
            const uint32_t f1 = free_index[var[k1]];
            if (f1 == kNone) continue;
            const double a1 = coef[k1];
            for (uint32_t k2 = b; k2 < e; ++k2) {
                const uint32_t f2 = free_index[var[k2]];
                if (f2 == kNone) continue;
                keys[o] = (uint64_t(f1) << bits) | f2;
                vals[o] = mul_rn(a1, coef[k2]);
                ++o;
            }
        }
    }
}

// Free entries keyed by their free index (locked ones by nfree, sorted last),
// valued by the entry index.
__global__ void k_ls_entries(uint64_t nent, const uint32_t* var, const uint32_t* free_index,
                             uint32_t nfree, uint32_t* keys, uint32_t* vals) {
    const uint64_t stride = uint64_t(gridDim.x) * blockDim.x;
    for (uint64_t k = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; k < nent; k += stride) {
        const uint32_t f = free_index[var[k]];
        keys[k] = f == kNone ? nfree : f;
        vals[k] = uint32_t(k);
    }
}

// Entries per free variable, and the most of any.
__global__ void k_ls_count(uint64_t nent, const uint32_t* var, const uint32_t* free_index,
                           uint32_t* count, LSTotals* tot) {
    const uint64_t stride = uint64_t(gridDim.x) * blockDim.x;
    uint32_t most = 0;
    for (uint64_t k = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; k < nent; k += stride) {
        const uint32_t f = free_index[var[k]];
        if (f == kNone) continue;
        const uint32_t c = atomicAdd(&count[f], 1u) + 1u;
        most = most > c ? most : c;
    }
    for (int o = kWave / 2; o > 0; o >>= 1) {
        const uint32_t m = __shfl_xor(most, o, kWave);
        most = most > m ? most : m;
    }
    if ((threadIdx.x & (kWave - 1)) == 0 && most) atomicMax(&tot->max_occ, most);
}

// Entry indices by free variable, in any order within one (k_ls_wave sorts
// them); leaves count at 0.
__global__ void k_ls_scatter(uint64_t nent, const uint32_t* var, const uint32_t* free_index,
                             const uint32_t* occ_off, uint32_t* count, uint32_t* occ) {
    const uint64_t stride = uint64_t(gridDim.x) * blockDim.x;
    for (uint64_t k = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; k < nent; k += stride) {
        const uint32_t f = free_index[var[k]];
        if (f != kNone) occ[occ_off[f] + (atomicSub(&count[f], 1u) - 1u)] = uint32_t(k);
    }
}

__device__ __forceinline__ double lane_f64(double v, int l) {
    const long long b = __double_as_longlong(v);
    const uint32_t lo = lane_word(uint32_t(b), l), hi = lane_word(uint32_t(b >> 32), l);
    return __longlong_as_double((long long)((uint64_t(hi) << 32) | lo));
}

// One wavefront per free variable: the columns of its matrix row (FILL =
// false: counted), their sums and its right-hand sides (FILL).
//
// The variable's occurrences (at most 64, one per lane) are sorted by entry
// index: rank among them by one comparison with every lane.  Their rows are
// then read 64 / W at a time, W lanes per row (W a power of two, no row is
// longer), so lane order is (row, e1, e2) order.  Of those up to 64
// contributions, each distinct column is taken once: the lanes that hold it
// (a ballot) become the bit mask of the lane that owns the column (lane d
// owns the d-th column met), and then every owner adds its contributions in
// bit order, all columns side by side.  For LSCM (72 contributions to 14
// columns of at most 12) that is about a third of the steps of adding them
// one by one.  *over is raised when a variable has more than 64 columns.
template <bool FILL>
__global__ __launch_bounds__(kBlock) void k_ls_wave(
    uint32_t nfree, const uint32_t* __restrict__ occ_off, const uint32_t* __restrict__ occ,
    const uint32_t* __restrict__ row_of, const uint32_t* __restrict__ rp,
    const uint32_t* __restrict__ var, const double* __restrict__ coef,
    const uint32_t* __restrict__ free_index, uint32_t logW, uint32_t* __restrict__ row_count,
    uint32_t* __restrict__ over, const uint32_t* __restrict__ rowptr,
    uint32_t* __restrict__ colind, double* __restrict__ val, const double* __restrict__ S,
    uint32_t nrows, uint32_t nsys, double* __restrict__ rhs) {
    const int lane = threadIdx.x & (kWave - 1);
    const uint32_t w = xcd_logical_block(blockIdx.x, gridDim.x) * kWavesPerBlock +
                       threadIdx.x / kWave;
    const uint32_t stride = gridDim.x * kWavesPerBlock;
    for (uint32_t f = uint32_t(__builtin_amdgcn_readfirstlane(int(w))); f < nfree; f += stride) {
        const uint32_t o0 = occ_off[f], m = occ_off[f + 1] - o0;
        uint32_t k = uint32_t(lane) < m ? occ[o0 + uint32_t(lane)] : kNone;
        uint32_t rank = 0;
        for (uint32_t i = 0; i < m; ++i) rank += lane_word(k, int(i)) < k ? 1u : 0u;
        // push lane l's entry to lane rank (a permutation of the first m lanes;
        // the others keep their place)
        if (uint32_t(lane) >= m) rank = uint32_t(lane);
        k = uint32_t(__builtin_amdgcn_ds_permute(int(rank << 2), int(k)));
        const bool mine = uint32_t(lane) < m;
        const uint32_t r = mine ? row_of[k] : 0u;
        const uint32_t rb = mine ? rp[r] : 0u;
        const uint32_t len = mine ? rp[r + 1] - rb : 0u;
        const double a = FILL && mine ? coef[k] : 0.0;
        uint32_t col = kNone;  // of the matrix entry this lane owns
        double sum = 0.0;
        bool first = true;     // the owned entry has no contribution yet
        uint32_t ncol = 0;
        const uint32_t step = uint32_t(kWave) >> logW;
        for (uint32_t t = 0; t < m; t += step) {
            const uint32_t o = t + (uint32_t(lane) >> logW), q = uint32_t(lane) & ((1u << logW) - 1u);
            const uint32_t b = __shfl(rb, int(o & 63u), kWave);
            const uint32_t n = __shfl(len, int(o & 63u), kWave);
            const double ao = FILL ? __shfl(a, int(o & 63u), kWave) : 0.0;
            const bool in = o < m && q < n;
            const uint32_t f2 = in ? free_index[var[b + q]] : kNone;
            double p = 0.0;
            if (FILL && in) p = mul_rn(ao, coef[b + q]);
            uint64_t left = __ballot(f2 != kNone);
            uint64_t todo = 0;  // contributions of this chunk to the owned entry
            while (left) {
                const uint32_t c = lane_word(f2, __builtin_ctzll(left));
                const uint64_t here = __ballot(f2 == c);
                left &= ~here;
                if (!__ballot(col == c)) {
                    if (ncol == uint32_t(kWave)) {
                        if (lane == 0) atomicOr(over, 1u);
                        return;
                    }
                    if (uint32_t(lane) == ncol) col = c;
                    ++ncol;
                }
                if (FILL && col == c) todo = here;
            }
            if (FILL) {
                while (__ballot(todo != 0)) {
                    const int l = todo ? __builtin_ctzll(todo) : lane;
                    const double v = __shfl(p, l, kWave);
                    if (todo) {
                        sum = first ? v : add_rn(sum, v);
                        first = false;
                        todo &= todo - 1;
                    }
                }
            }
        }
        if (!FILL) {
            if (lane == 0) row_count[f] = ncol;
            continue;
        }
        uint32_t at = 0;
        for (uint32_t i = 0; i < ncol; ++i) at += lane_word(col, int(i)) < col ? 1u : 0u;
        if (uint32_t(lane) < ncol) {
            const uint32_t j = rowptr[f] + at;
            colind[j] = col;
            val[j] = sum;
        }
        for (uint32_t s = 0; s < nsys; ++s) {
            const double t = mine ? mul_rn(a, S[size_t(s) * nrows + r]) : 0.0;
            double acc = 0.0;
            for (uint32_t i = 0; i < m; ++i) acc = add_rn(acc, lane_f64(t, int(i)));
            if (lane == 0) rhs[size_t(s) * nfree + f] = acc;
        }
    }
}

// 1 where a run of equal keys starts.
__global__ void k_ls_heads(uint64_t n, const uint64_t* keys, uint32_t* head) {
    const uint64_t stride = uint64_t(gridDim.x) * blockDim.x;
    for (uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride)
        head[i] = (i == 0 || keys[i] != keys[i - 1]) ? 1u : 0u;
}

__global__ void k_ls_starts(uint64_t n, const uint32_t* head, const uint32_t* seg,
                            uint64_t* start) {
    const uint64_t stride = uint64_t(gridDim.x) * blockDim.x;
    for (uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride)
        if (head[i]) start[seg[i]] = i;
}

// One matrix entry per run: the first contribution, then the others added in
// order; its column, and a count for its row.
__global__ void k_ls_entry_sums(uint32_t nseg, uint64_t n, const uint64_t* start,
                                const uint64_t* keys, const double* vals, uint32_t bits,
                                uint32_t* colind, double* val, uint32_t* row_count) {
    const uint32_t stride = gridDim.x * blockDim.x;
    const uint64_t mask = (uint64_t(1) << bits) - 1u;
    for (uint32_t s = blockIdx.x * blockDim.x + threadIdx.x; s < nseg; s += stride) {
        const uint64_t b = start[s], e = (s + 1 < nseg) ? start[s + 1] : n;
        double v = vals[b];
        for (uint64_t i = b + 1; i < e; ++i) v = add_rn(v, vals[i]);
        const uint64_t key = keys[b];
        colind[s] = uint32_t(key & mask);
        val[s] = v;
        atomicAdd(&row_count[uint32_t(key >> bits)], 1u);
    }
}

// b[s][f] = sum over the free entries of f (entry order) of a_e S[s][row(e)],
// starting from 0.
__global__ void k_ls_rhs(uint32_t nfree, const uint32_t* occ_off, const uint32_t* occ,
                         const double* coef, const uint32_t* row_of, const double* S,
                         uint32_t nrows, uint32_t nsys, double* rhs) {
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t f = blockIdx.x * blockDim.x + threadIdx.x; f < nfree; f += stride) {
        const uint32_t b = occ_off[f], e = occ_off[f + 1];
        for (uint32_t s = 0; s < nsys; ++s) {
            double acc = 0.0;
            for (uint32_t i = b; i < e; ++i) {
                const uint32_t k = occ[i];
                acc = add_rn(acc, mul_rn(coef[k], S[size_t(s) * nrows + row_of[k]]));
            }
            rhs[size_t(s) * nfree + f] = acc;
        }
    }
}

// ---- LSCM rows on the device

// Triangle t's 12 LSCM coefficients (Levy, Petitjean, Ray, Maillot 2002):
// the conformality of the map in the triangle's orthonormal frame (X along
// p1 - p0, Y = N x X), W0 = z2 - z1, W1 = z0 - z2, W2 = z1 - z0, scaled by
// 1/sqrt(|e1 x e2|): real row (Wr, -Wi) then imaginary row (Wi, Wr) over
// (u0, v0, u1, v1, u2, v2).  False for a degenerate triangle.  Every
// operation is the host builder's (workloads.cpp, lscm_coeffs), in its
// order, correctly rounded and unfused, so the coefficients are its bits.
// COEFS = false: the test alone.
template <bool COEFS>
__device__ __forceinline__ bool lscm_coeffs(const double* P, const uint32_t* T, uint32_t t,
                                            double (&out)[12]) {
    const uint32_t* q = T + 3 * size_t(t);
    const double* p0 = P + 3 * size_t(q[0]);
    const double* p1 = P + 3 * size_t(q[1]);
    const double* p2 = P + 3 * size_t(q[2]);
    const double e1[3] = {p1[0] - p0[0], p1[1] - p0[1], p1[2] - p0[2]};
    const double e2[3] = {p2[0] - p0[0], p2[1] - p0[1], p2[2] - p0[2]};
    const double nr[3] = {e1[1] * e2[2] - e1[2] * e2[1], e1[2] * e2[0] - e1[0] * e2[2],
                          e1[0] * e2[1] - e1[1] * e2[0]};
    const double dT = sqrt(nr[0] * nr[0] + nr[1] * nr[1] + nr[2] * nr[2]);
    const double l1 = sqrt(e1[0] * e1[0] + e1[1] * e1[1] + e1[2] * e1[2]);
    if (!(dT > 0.0) || !(l1 > 0.0)) return false;
    if (!COEFS) return true;
    const double X[3] = {e1[0] / l1, e1[1] / l1, e1[2] / l1};
    const double Nn[3] = {nr[0] / dT, nr[1] / dT, nr[2] / dT};
    const double Y[3] = {Nn[1] * X[2] - Nn[2] * X[1], Nn[2] * X[0] - Nn[0] * X[2],
                         Nn[0] * X[1] - Nn[1] * X[0]};
    const double z1x = l1, z1y = 0.0;
    const double z2x = e2[0] * X[0] + e2[1] * X[1] + e2[2] * X[2];
    const double z2y = e2[0] * Y[0] + e2[1] * Y[1] + e2[2] * Y[2];
    const double Wr[3] = {z2x - z1x, -z2x, z1x};
    const double Wi[3] = {z2y - z1y, -z2y, z1y};
    const double sq = sqrt(dT);
    for (int j = 0; j < 3; ++j) {
        const double cr = Wr[j] / sq, ci = Wi[j] / sq;
        out[2 * j] = cr;
        out[2 * j + 1] = -ci;
        out[6 + 2 * j] = ci;
        out[6 + 2 * j + 1] = cr;
    }
    return true;
}

// ok[t] = 0 for a degenerate triangle.
__global__ void k_lscm_valid(uint32_t nt, const double* P, const uint32_t* T, uint32_t* ok) {
    const uint32_t stride = gridDim.x * blockDim.x;
    double c[12];
    for (uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < nt; t += stride)
        ok[t] = lscm_coeffs<false>(P, T, t, c) ? 1u : 0u;
}

// Rows of the valid triangles in triangle order: triangle t at slot s (an
// exclusive count of the valid ones before it) gives rows 2s (real) and
// 2s + 1 (imaginary), 6 entries each.  The valid triangles of a workgroup
// have consecutive slots, so their entries are staged in LDS and written in
// order: with one triangle per thread each store instruction touched 64
// lines (656 us for 2 M triangles; now 64 us).
__global__ __launch_bounds__(kBlock) void k_lscm_rows(uint32_t nt, const double* P,
                                                      const uint32_t* T, const uint32_t* ok,
                                                      const uint32_t* slot, uint32_t* var,
                                                      double* coef) {
    __shared__ double s_coef[12 * kBlock];
    __shared__ uint32_t s_var[6 * kBlock];
    for (uint32_t t0 = blockIdx.x * kBlock; t0 < nt; t0 += gridDim.x * kBlock) {
        const uint32_t t = t0 + threadIdx.x;
        const uint32_t first = slot[t0];
        const uint32_t last = slot[t0 + kBlock < nt ? t0 + kBlock : nt];  // nt + 1 slots
        if (t < nt && ok[t]) {
            double c[12];
            lscm_coeffs<true>(P, T, t, c);
            const uint32_t at = slot[t] - first;
#pragma unroll
            for (int e = 0; e < 12; ++e) s_coef[12 * at + e] = c[e];
#pragma unroll
            for (int e = 0; e < 6; ++e)
                s_var[6 * at + e] = 2u * T[3 * size_t(t) + e / 2] + uint32_t(e & 1);
        }
        __syncthreads();
        const uint32_t n = 12u * (last - first);
        const size_t base = 12 * size_t(first);
        for (uint32_t i = threadIdx.x; i < n; i += kBlock) {
            coef[base + i] = s_coef[i];
            var[base + i] = s_var[6u * (i / 12u) + (i % 6u)];
        }
        __syncthreads();
    }
}

// The variables (2v, 2v + 1) of nv vertices, those of two of them locked at
// (u0, v0) and (u1, v1): free indices in order, and the locked values.
__global__ void k_lscm_free(uint32_t nv, uint32_t pin0, double u0, double v0, uint32_t pin1,
                            double u1, double v1, uint32_t* free_index, double* values) {
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < nv; v += stride) {
        const uint32_t f = 2u * (v - (pin0 < v ? 1u : 0u) - (pin1 < v ? 1u : 0u));
        const bool l0 = v == pin0, l1 = v == pin1;
        free_index[2 * size_t(v)] = l0 || l1 ? kNone : f;
        free_index[2 * size_t(v) + 1] = l0 || l1 ? kNone : f + 1u;
        values[2 * size_t(v)] = l0 ? u0 : (l1 ? u1 : 0.0);
        values[2 * size_t(v) + 1] = l0 ? v0 : (l1 ? v1 : 0.0);
    }
}

__global__ void k_lscm_check(uint32_t nv, uint32_t nt, const double* P, const uint32_t* T,
                             uint32_t* bad) {
    const uint32_t stride = gridDim.x * blockDim.x;
    uint32_t flags = 0;
    for (uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < nt; t += stride)
        for (int k = 0; k < 3; ++k)
            if (T[3 * size_t(t) + k] >= nv) flags |= 2u;
    for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < nv; v += stride)
        for (int k = 0; k < 3; ++k)
            if (!isfinite(P[3 * size_t(v) + k])) flags |= 4u;
    if (flags) atomicOr(bad, flags);
}

// *bad = 1 when a triangle's vertices lie in different charts (chart c owns
// vertices [voff[c], voff[c+1])).
__global__ void k_tri_chart_check(uint32_t nt, const uint32_t* T, const uint32_t* voff,
                                  uint32_t nc, uint32_t* bad) {
    const uint32_t stride = gridDim.x * blockDim.x;
    uint32_t flag = 0;
    for (uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < nt; t += stride) {
        uint32_t chart[3];
        for (int k = 0; k < 3; ++k) {
            const uint32_t v = T[3 * size_t(t) + k];
            uint32_t lo = 0, hi = nc;  // last c with voff[c] <= v
            while (hi - lo > 1) {
                const uint32_t mid = (lo + hi) / 2;
                if (voff[mid] <= v) lo = mid;
                else hi = mid;
            }
            chart[k] = lo;
        }
        flag |= (chart[0] != chart[1] || chart[0] != chart[2]) ? 1u : 0u;
    }
    if (flag) atomicOr(bad, 1u);
}

__global__ void k_row_ptr6(uint32_t nrows, uint32_t* rp) {
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t r = blockIdx.x * blockDim.x + threadIdx.x; r <= nrows; r += stride)
        rp[r] = 6u * r;
}

uint32_t grid_for(uint64_t n) {
    const uint64_t g = (n + kBlock - 1) / kBlock;
    return uint32_t(g < 1 ? 1 : (g > 65536 ? 65536 : g));
}

// The same for kernels that end with an atomic per wavefront on one address:
// 262,144 of them took 1.4 ms (sum) and 2.8 ms (maximum) of k_ls_rows and
// k_ls_count, 8,192 some microseconds.
uint32_t grid_atomic(uint64_t n) { return std::min(grid_for(n), 2048u); }

// A hipCUB call with its temporary storage (kept until the call has run).
template <typename F>
void with_temp(F&& call, hipStream_t s) {
    size_t bytes = 0;
    NLHIP_CHECK(call(nullptr, bytes));
    DevBuf<uint8_t> tmp(bytes);
    NLHIP_CHECK(call(tmp.get(), bytes));
    NLHIP_CHECK(hipStreamSynchronize(s));
}

}  // namespace

void lscm_rows_device(uint32_t nv, const double* P, uint32_t nt, const uint32_t* T,
                      LSRows& rows, hipStream_t s) {
    {
        DevBuf<uint32_t> bad(1);
        NLHIP_CHECK(hipMemsetAsync(bad.get(), 0, 4, s));
        k_lscm_check<<<grid_for(nt > nv ? nt : nv), kBlock, 0, s>>>(nv, nt, P, T, bad.get());
        NLHIP_CHECK(hipGetLastError());
        uint32_t h = 0;
        NLHIP_CHECK(hipMemcpyAsync(&h, bad.get(), 4, hipMemcpyDeviceToHost, s));
        NLHIP_CHECK(hipStreamSynchronize(s));
        if (h & 2u) throw Error(NLHIP_ERR_INVALID, "triangle vertex index out of range");
        if (h & 4u) throw Error(NLHIP_ERR_NONFINITE, "vertex coordinate is NaN or Inf");
    }
    DevBuf<uint32_t> ok(size_t(nt) + 1), slot(size_t(nt) + 1);
    NLHIP_CHECK(hipMemsetAsync(ok.get(), 0, (size_t(nt) + 1) * 4, s));
    if (nt) k_lscm_valid<<<grid_for(nt), kBlock, 0, s>>>(nt, P, T, ok.get());
    NLHIP_CHECK(hipGetLastError());
    with_temp([&](void* t, size_t& b) {
        return hipcub::DeviceScan::ExclusiveSum(t, b, ok.get(), slot.get(), size_t(nt) + 1, s);
    }, s);
    uint32_t nvalid = 0;
    NLHIP_CHECK(hipMemcpyAsync(&nvalid, slot.get() + nt, 4, hipMemcpyDeviceToHost, s));
    NLHIP_CHECK(hipStreamSynchronize(s));
    if (uint64_t(nvalid) * 12 > 0xffffffffull)
        throw Error(NLHIP_ERR_UNSUPPORTED, "more than 2^32 - 1 row coefficients");
    rows.nrows = 2 * nvalid;
    rows.rp.alloc(size_t(rows.nrows) + 1);
    rows.var.alloc(12 * size_t(nvalid ? nvalid : 1));
    rows.coef.alloc(12 * size_t(nvalid ? nvalid : 1));
    k_row_ptr6<<<grid_for(size_t(rows.nrows) + 1), kBlock, 0, s>>>(rows.nrows, rows.rp.get());
    if (nt)
        k_lscm_rows<<<grid_for(nt), kBlock, 0, s>>>(nt, P, T, ok.get(), slot.get(),
                                                    rows.var.get(), rows.coef.get());
    NLHIP_CHECK(hipGetLastError());
    NLHIP_CHECK(hipStreamSynchronize(s));
}

void lscm_free_device(uint32_t nv, const uint32_t pin[2], const double uv[4],
                      uint32_t* free_index, double* values, hipStream_t s) {
    k_lscm_free<<<grid_for(nv), kBlock, 0, s>>>(nv, pin[0], uv[0], uv[1], pin[1], uv[2], uv[3],
                                                free_index, values);
    NLHIP_CHECK(hipGetLastError());
}

void check_triangle_charts(uint32_t nt, const uint32_t* T, const uint32_t* voff, uint32_t nc,
                           hipStream_t s) {
    DevBuf<uint32_t> bad(1);
    NLHIP_CHECK(hipMemsetAsync(bad.get(), 0, 4, s));
    if (nt) k_tri_chart_check<<<grid_for(nt), kBlock, 0, s>>>(nt, T, voff, nc, bad.get());
    NLHIP_CHECK(hipGetLastError());
    uint32_t h = 0;
    NLHIP_CHECK(hipMemcpyAsync(&h, bad.get(), 4, hipMemcpyDeviceToHost, s));
    NLHIP_CHECK(hipStreamSynchronize(s));
    if (h) throw Error(NLHIP_ERR_INVALID, "a triangle spans two charts");
}

// The plan by variable (k_ls_wave); false when a variable has more columns
// than a wavefront has lanes (out.rhs is then still to be written).
static bool ls_assemble_waves(const LSInput& in, LSOutput& out, const LSTotals& tot,
                              const double* S, const uint32_t* row_of, uint32_t* occ_count,
                              const uint32_t* occ_off, hipStream_t s) {
    const uint32_t nfree = in.nfree;
    uint32_t logW = 0;
    while ((1u << logW) < tot.max_row) ++logW;
    const uint32_t grid =
        uint32_t(std::min<uint64_t>((uint64_t(nfree) + kWavesPerBlock - 1) / kWavesPerBlock,
                                    1u << 20));
    DevBuf<uint32_t> occ(in.nent ? in.nent : 1), row_count(size_t(nfree) + 1), over(1);
    DevBuf<uint32_t> rowptr(size_t(nfree) + 1);
    NLHIP_CHECK(hipMemsetAsync(row_count.get() + nfree, 0, 4, s));
    NLHIP_CHECK(hipMemsetAsync(over.get(), 0, 4, s));
    if (in.nent)
        k_ls_scatter<<<grid_for(in.nent), kBlock, 0, s>>>(in.nent, in.var, in.free_index,
                                                          occ_off, occ_count, occ.get());
    k_ls_wave<false><<<grid, kBlock, 0, s>>>(nfree, occ_off, occ.get(), row_of, in.rp, in.var,
                                             in.coef, in.free_index, logW, row_count.get(),
                                             over.get(), nullptr, nullptr, nullptr, S, in.nrows,
                                             in.nsys, nullptr);
    NLHIP_CHECK(hipGetLastError());
    with_temp([&](void* t, size_t& b) {
        return hipcub::DeviceScan::ExclusiveSum(t, b, row_count.get(), rowptr.get(),
                                                size_t(nfree) + 1, s);
    }, s);
    uint32_t nnz = 0, h_over = 0;
    NLHIP_CHECK(hipMemcpyAsync(&nnz, rowptr.get() + nfree, 4, hipMemcpyDeviceToHost, s));
    NLHIP_CHECK(hipMemcpyAsync(&h_over, over.get(), 4, hipMemcpyDeviceToHost, s));
    NLHIP_CHECK(hipStreamSynchronize(s));
    if (h_over) return false;
    out.colind.alloc(nnz);
    out.val.alloc(nnz);
    k_ls_wave<true><<<grid, kBlock, 0, s>>>(nfree, occ_off, occ.get(), row_of, in.rp, in.var,
                                            in.coef, in.free_index, logW, nullptr, over.get(),
                                            rowptr.get(), out.colind.get(), out.val.get(), S,
                                            in.nrows, in.nsys, out.rhs.get());
    NLHIP_CHECK(hipGetLastError());
    NLHIP_CHECK(hipStreamSynchronize(s));  // before the lists go
    out.rowptr = std::move(rowptr);
    out.nnz = nnz;
    return true;
}

void ls_assemble_device(const LSInput& in, LSOutput& out, hipStream_t s) {
    const uint32_t nrows = in.nrows, nvars = in.nvars, nsys = in.nsys, nfree = in.nfree;
    const uint64_t nent = in.nent;
    // checks
    {
        DevBuf<uint32_t> bad(1);
        NLHIP_CHECK(hipMemsetAsync(bad.get(), 0, 4, s));
        k_ls_check<<<grid_for(nrows > nvars ? nrows : nvars), kBlock, 0, s>>>(
            nrows, nvars, nent, in.rp, in.var, in.coef, nsys, in.row_rhs, in.free_index,
            in.values, bad.get());
        NLHIP_CHECK(hipGetLastError());
        uint32_t h = 0;
        NLHIP_CHECK(hipMemcpyAsync(&h, bad.get(), 4, hipMemcpyDeviceToHost, s));
        NLHIP_CHECK(hipStreamSynchronize(s));
        if (h & 1u) throw Error(NLHIP_ERR_INVALID, "row_ptr is not monotone or exceeds the entries");
        if (h & 2u) throw Error(NLHIP_ERR_INVALID, "variable index out of range");
        if (h & 4u) throw Error(NLHIP_ERR_NONFINITE, "coefficient or right-hand side is NaN or Inf");
    }
    // rows: S, row of each entry; entries per variable; the totals
    DevBuf<double> S(size_t(nsys) * (nrows ? nrows : 1));
    DevBuf<uint32_t> row_of(nent ? nent : 1);
    DevBuf<uint32_t> occ_count(size_t(nfree) + 1), occ_off(size_t(nfree) + 1);
    DevBuf<LSTotals> tot(1);
    NLHIP_CHECK(hipMemsetAsync(occ_count.get(), 0, (size_t(nfree) + 1) * 4, s));
    NLHIP_CHECK(hipMemsetAsync(tot.get(), 0, sizeof(LSTotals), s));
    if (nrows)
        k_ls_rows<<<grid_atomic(nrows), kBlock, 0, s>>>(nrows, in.rp, in.var, in.coef,
                                                     in.free_index, in.values, nvars, nsys,
                                                     in.row_rhs, S.get(), row_of.get(),
                                                     tot.get());
    if (nent)
        k_ls_count<<<grid_atomic(nent), kBlock, 0, s>>>(nent, in.var, in.free_index,
                                                     occ_count.get(), tot.get());
    NLHIP_CHECK(hipGetLastError());
    with_temp([&](void* t, size_t& b) {
        return hipcub::DeviceScan::ExclusiveSum(t, b, occ_count.get(), occ_off.get(),
                                                size_t(nfree) + 1, s);
    }, s);
    LSTotals h_tot{};
    NLHIP_CHECK(hipMemcpyAsync(&h_tot, tot.get(), sizeof(h_tot), hipMemcpyDeviceToHost, s));
    NLHIP_CHECK(hipStreamSynchronize(s));
    const uint64_t npair = h_tot.pairs;
    if (npair > 0xffffffffull)
        throw Error(NLHIP_ERR_UNSUPPORTED,
                    "more than 2^32 - 1 coefficient products in one least-squares assembly");
    out.rhs.alloc(size_t(nsys) * nfree);
    if (h_tot.max_row <= kWaveMax && h_tot.max_occ <= kWaveMax &&
        ls_assemble_waves(in, out, h_tot, S.get(), row_of.get(), occ_count.get(), occ_off.get(),
                          s))
        return;
    DevBuf<uint64_t> npairs(size_t(nrows) + 1);
    NLHIP_CHECK(hipMemsetAsync(npairs.get(), 0, (size_t(nrows) + 1) * 8, s));
    if (nrows)
        k_ls_npairs<<<grid_for(nrows), kBlock, 0, s>>>(nrows, in.rp, in.var, in.free_index,
                                                       npairs.get());
    NLHIP_CHECK(hipGetLastError());
    DevBuf<uint64_t> pair_off(size_t(nrows) + 1);
    with_temp([&](void* t, size_t& b) {
        return hipcub::DeviceScan::ExclusiveSum(t, b, npairs.get(), pair_off.get(),
                                                size_t(nrows) + 1, s);
    }, s);
    npairs.release();

    uint32_t bits = 1;
    while (bits < 32 && (uint64_t(1) << bits) < nfree) ++bits;

    // matrix: pair products, stable sort by (f1, f2), one sum per entry
    uint64_t nnz = 0;
    DevBuf<uint32_t> row_count(size_t(nfree) + 1);
    NLHIP_CHECK(hipMemsetAsync(row_count.get(), 0, (size_t(nfree) + 1) * 4, s));
    if (npair) {
        DevBuf<uint64_t> k0(npair), k1(npair);
        DevBuf<double> v0(npair), v1(npair);
        k_ls_pairs<<<grid_for(nrows), kBlock, 0, s>>>(nrows, in.rp, in.var, in.coef,
                                                      in.free_index, pair_off.get(), bits,
                                                      k0.get(), v0.get());
        NLHIP_CHECK(hipGetLastError());
        hipcub::DoubleBuffer<uint64_t> kb(k0.get(), k1.get());
        hipcub::DoubleBuffer<double> vb(v0.get(), v1.get());
        with_temp([&](void* t, size_t& b) {
            return hipcub::DeviceRadixSort::SortPairs(t, b, kb, vb, npair, 0, int(2 * bits), s);
        }, s);
        const uint64_t* keys = kb.Current();
        const double* vals = vb.Current();
        DevBuf<uint32_t> head(npair), seg(npair);
        k_ls_heads<<<grid_for(npair), kBlock, 0, s>>>(npair, keys, head.get());
        NLHIP_CHECK(hipGetLastError());
        with_temp([&](void* t, size_t& b) {
            return hipcub::DeviceScan::ExclusiveSum(t, b, head.get(), seg.get(), npair, s);
        }, s);
        uint32_t last_seg = 0, last_head = 0;
        NLHIP_CHECK(hipMemcpyAsync(&last_seg, seg.get() + npair - 1, 4, hipMemcpyDeviceToHost, s));
        NLHIP_CHECK(hipMemcpyAsync(&last_head, head.get() + npair - 1, 4, hipMemcpyDeviceToHost, s));
        NLHIP_CHECK(hipStreamSynchronize(s));
        nnz = uint64_t(last_seg) + last_head;
        if (nnz > 0xffffffffull)
            throw Error(NLHIP_ERR_UNSUPPORTED, "normal equations with 2^32 or more nonzeros");
        DevBuf<uint64_t> start(nnz);
        k_ls_starts<<<grid_for(npair), kBlock, 0, s>>>(npair, head.get(), seg.get(), start.get());
        NLHIP_CHECK(hipGetLastError());
        NLHIP_CHECK(hipStreamSynchronize(s));
        head.release();
        seg.release();
        out.colind.alloc(nnz);
        out.val.alloc(nnz);
        k_ls_entry_sums<<<grid_for(nnz), kBlock, 0, s>>>(uint32_t(nnz), npair, start.get(), keys,
                                                         vals, bits, out.colind.get(),
                                                         out.val.get(), row_count.get());
        NLHIP_CHECK(hipGetLastError());
        NLHIP_CHECK(hipStreamSynchronize(s));  // before the sort buffers go
    } else {
        out.colind.alloc(1);
        out.val.alloc(1);
    }
    out.rowptr.alloc(size_t(nfree) + 1);
    with_temp([&](void* t, size_t& b) {
        return hipcub::DeviceScan::ExclusiveSum(t, b, row_count.get(), out.rowptr.get(),
                                                size_t(nfree) + 1, s);
    }, s);
    out.nnz = nnz;

    // right-hand sides: free entries sorted by free index (stable)
    DevBuf<uint32_t> ek0(nent ? nent : 1), ek1(nent ? nent : 1), ev0(nent ? nent : 1),
        ev1(nent ? nent : 1);
    const uint32_t* occ = ev0.get();
    if (nent) {
        k_ls_entries<<<grid_for(nent), kBlock, 0, s>>>(nent, in.var, in.free_index, nfree,
                                                       ek0.get(), ev0.get());
        NLHIP_CHECK(hipGetLastError());
        uint32_t ebits = 1;
        while (ebits < 32 && (uint64_t(1) << ebits) <= nfree) ++ebits;
        hipcub::DoubleBuffer<uint32_t> kb(ek0.get(), ek1.get()), vb(ev0.get(), ev1.get());
        with_temp([&](void* t, size_t& b) {
            return hipcub::DeviceRadixSort::SortPairs(t, b, kb, vb, nent, 0, int(ebits), s);
        }, s);
        occ = vb.Current();
    }
    k_ls_rhs<<<grid_for(nfree), kBlock, 0, s>>>(nfree, occ_off.get(), occ, in.coef,
                                                row_of.get(), S.get(), nrows, nsys,
                                                out.rhs.get());
    NLHIP_CHECK(hipGetLastError());
    NLHIP_CHECK(hipStreamSynchronize(s));
}

}  // namespace nlhip
