// SSOR preconditioner objects (nlNewSSORPreconditioner): level schedules of
// the two triangular sweeps, built once on the host from the matrix
// pattern, and the sweeps of one application captured as a graph.  The
// arithmetic is in k_ssor.hip.
#include <algorithm>
#include <cmath>
#include <memory>

#include "nlhip_internal.h"

namespace nlhip {

namespace {

// Levels of at most this many loads (six per row and two per entry it reads)
// run back to back in one workgroup, larger ones are launches of their own: a
// launch takes about 4 us, and the one CU of the chain issues a wavefront's
// loads, which are not coalesced, in some 30 ns each.  us per application with
// limits of 2500, 5000, 9000, 16000, 24000: 300^2 cotangent 2470, 1630, 1630, 1610,
// 1620; 317^2 LSCM 5920, 4200, 3060, 3030, 3050; 27-point stencil on 64^3 4360,
// 4280, 4180, 4200, 4600; 7-point 1500, 1430, 1400, 1470, 1680; Delaunay mesh of
// 20 k vertices numbered at random 170, 172, 174, 179, 221.  With a limit of 4096
// rows instead the last three took 9750, 2950 and 350.
constexpr uint64_t kChainLoads = 9000;

// level(i) = 1 + the deepest level among the rows i reads (j < i for the
// forward sweep, j > i for the backward one); rows counting-sorted by level
// (increasing row index within a level); eoff: the first of the entries that
// each position reads.
void level_schedule(uint32_t n, const std::vector<uint32_t>& rp, const std::vector<uint32_t>& ci,
                    bool upper, std::vector<uint32_t>& rows, std::vector<uint32_t>& off,
                    std::vector<uint32_t>& eoff) {
    std::vector<uint32_t> reads(n);
    std::vector<uint32_t> lev(n, 0);
    uint32_t top = 0;
    for (uint32_t k = 0; k < n; ++k) {
        const uint32_t i = upper ? n - 1 - k : k;
        uint32_t l = 0, m = 0;
        for (uint32_t e = rp[i]; e < rp[i + 1]; ++e) {
            const uint32_t j = ci[e];
            if (upper ? j > i : j < i) {
                l = std::max(l, lev[j] + 1);
                ++m;
            }
        }
        lev[i] = l;
        reads[i] = m;
        top = std::max(top, l);
    }
    off.assign(size_t(top) + 2, 0);
    for (uint32_t i = 0; i < n; ++i) ++off[lev[i] + 1];
    for (size_t l = 1; l < off.size(); ++l) off[l] += off[l - 1];
    rows.resize(n);
    std::vector<uint32_t> next(off.begin(), off.end() - 1);
    for (uint32_t i = 0; i < n; ++i) rows[next[lev[i]]++] = i;
    eoff.assign(size_t(n) + 1, 0);
    for (uint32_t k = 0; k < n; ++k) eoff[k + 1] = eoff[k] + reads[rows[k]];
}

}  // namespace

// One sweep on the device: rows by level and their packed entries.
struct SweepBufs {
    DevBuf<uint32_t> rows, off, eoff, col, dep, lev;
    DevBuf<double> val;
    SsorSweepArgs args() const {
        return SsorSweepArgs{rows.get(), off.get(), eoff.get(), col.get(),
                             dep.get(),  lev.get(), val.get()};
    }
};

class Ssor {
  public:
    struct Step {
        uint32_t l0, l1, k0, k1;  // levels [l0, l1), positions [k0, k1)
        bool grid;                // one level over the whole grid, or a chain
    };
    uint32_t n = 0;
    double omega = 1.5;
    SweepBufs lo, up;
    DevBuf<double> diag, dscale, x, w, y;
    std::vector<Step> lo_steps, up_steps;
    Stream stream;
    Graph graph;
    std::mutex mu;

    SsorArgs args() const {
        SsorArgs a{};
        a.lo = lo.args();
        a.up = up.args();
        a.diag = diag.get();
        a.dscale = dscale.get();
        a.x = x.get();
        a.w = w.get();
        a.y = y.get();
        a.omega = omega;
        a.post = 2.0 - omega;
        a.n = n;
        return a;
    }
};

namespace {

// One launch per level that is too large for one workgroup, one workgroup
// per run of consecutive others.  off: first position of each level, eoff:
// first entry of each position.
std::vector<Ssor::Step> plan(const std::vector<uint32_t>& off, const std::vector<uint32_t>& eoff) {
    std::vector<Ssor::Step> steps;
    const uint32_t nl = uint32_t(off.size() - 1);
    auto large = [&](uint32_t l) {
        const uint64_t rows = off[l + 1] - off[l], entries = eoff[off[l + 1]] - eoff[off[l]];
        return 6 * rows + 2 * entries > kChainLoads;
    };
    uint32_t l = 0;
    while (l < nl) {
        uint32_t e = l + 1;
        const bool grid = large(l);
        while (!grid && e < nl && !large(e)) ++e;
        steps.push_back({l, e, off[l], off[e], grid});
        l = e;
    }
    return steps;
}

}  // namespace

namespace {

// Level schedule of one sweep, its positions' packed entries, and the
// launch plan; uploaded on stream s.
std::vector<Ssor::Step> build_sweep(uint32_t n, const std::vector<uint32_t>& rp,
                                    const std::vector<uint32_t>& ci, const std::vector<double>& va,
                                    bool upper, SweepBufs& B, hipStream_t s) {
    std::vector<uint32_t> rows, off, eoff;
    level_schedule(n, rp, ci, upper, rows, off, eoff);
    std::vector<Ssor::Step> steps = plan(off, eoff);
    // columns for the levels launched over the grid, positions for the others
    bool by_col = false, by_pos = false;
    for (const Ssor::Step& st : steps) (st.grid ? by_col : by_pos) = true;
    std::vector<uint32_t> col, dep, lev(by_pos ? n : 0), at(by_pos ? n : 0);
    std::vector<double> val;
    val.reserve(ci.size() / 2 + 1);
    if (by_col) col.reserve(ci.size() / 2 + 1);
    if (by_pos) {
        dep.reserve(ci.size() / 2 + 1);
        for (uint32_t k = 0; k < n; ++k) at[rows[k]] = k;
        for (size_t l = 0; l + 1 < off.size(); ++l)
            std::fill(lev.begin() + off[l], lev.begin() + off[l + 1], uint32_t(l));
    }
    for (uint32_t k = 0; k < n; ++k) {
        const uint32_t i = rows[k];
        for (uint32_t e = rp[i]; e < rp[i + 1]; ++e)
            if (upper ? ci[e] > i : ci[e] < i) {
                if (by_col) col.push_back(ci[e]);
                if (by_pos) dep.push_back(at[ci[e]]);
                val.push_back(va[e]);
            }
    }
    auto put = [&](auto& dst, const auto& src) {
        if (src.empty()) return;
        dst.alloc(src.size());
        copy_in(dst.get(), src.data(), src.size() * sizeof(src[0]), s);
    };
    put(B.rows, rows);
    put(B.off, off);
    put(B.eoff, eoff);
    put(B.col, col);
    put(B.dep, dep);
    put(B.lev, lev);
    put(B.val, val);
    NLHIP_CHECK(hipStreamSynchronize(s));  // the host arrays go out of scope
    return steps;
}

}  // namespace

Ssor* ssor_create(System& S, double omega) {
    if (!std::isfinite(omega) || omega == 0.0)
        throw Error(NLHIP_ERR_INVALID, "SSOR omega must be finite and nonzero");
    std::lock_guard<std::mutex> lock(S.mu);
    auto P = std::make_unique<Ssor>();
    const uint32_t n = S.n;
    const uint64_t nnz = S.nnz;
    P->n = n;
    P->omega = omega;
    hipStream_t s = P->stream.get();
    // the matrix on the host (a copy: the preconditioner outlives changes to M)
    std::vector<uint32_t> rp(size_t(n) + 1), ci(nnz);
    std::vector<double> va(nnz);
    NLHIP_CHECK(hipMemcpyAsync(rp.data(), S.rowptr.get(), rp.size() * 4, hipMemcpyDeviceToHost, s));
    if (nnz) {
        NLHIP_CHECK(hipMemcpyAsync(ci.data(), S.colind.get(), nnz * 4, hipMemcpyDeviceToHost, s));
        NLHIP_CHECK(hipMemcpyAsync(va.data(), S.val.get(), nnz * 8, hipMemcpyDeviceToHost, s));
    }
    P->diag.alloc(n);
    P->dscale.alloc(n);
    {
        DevBuf<uint32_t> bad(1);
        NLHIP_CHECK(hipMemsetAsync(bad.get(), 0, 4, s));
        NLHIP_CHECK(ssor_diag(n, S.rowptr.get(), S.colind.get(), S.val.get(), omega,
                              P->diag.get(), P->dscale.get(), bad.get(), s));
        uint32_t h = 0;
        NLHIP_CHECK(hipMemcpyAsync(&h, bad.get(), 4, hipMemcpyDeviceToHost, s));
        P->stream.sync();
        if (h) throw Error(NLHIP_ERR_INVALID, "SSOR needs a nonzero, finite diagonal entry in every row");
    }
    P->lo_steps = build_sweep(n, rp, ci, va, false, P->lo, s);
    P->up_steps = build_sweep(n, rp, ci, va, true, P->up, s);
    P->x.alloc(n);
    P->w.alloc(n);
    P->y.alloc(n);
    const SsorArgs a = P->args();
    NLHIP_CHECK(ssor_chain_init());
    P->graph.capture(s, [&] {
        auto sweep = [&](const std::vector<Ssor::Step>& steps, bool upper) {
            for (const Ssor::Step& st : steps) {
                if (st.grid)
                    NLHIP_CHECK(ssor_level(a, upper, st.l0, st.k1 - st.k0, s));
                else
                    NLHIP_CHECK(ssor_chain(a, upper, st.k0, st.k1, s));
            }
        };
        sweep(P->lo_steps, false);
        sweep(P->up_steps, true);
        NLHIP_CHECK(ssor_scale(a, s));
    });
    return P.release();
}

void ssor_destroy(Ssor* P) { delete P; }

uint32_t ssor_n(const Ssor& P) { return P.n; }

void ssor_apply(Ssor& P, const double* x, double* y, hipStream_t s) {
    std::lock_guard<std::mutex> lock(P.mu);
    const size_t bytes = size_t(P.n) * 8;
    NLHIP_CHECK(hipMemcpyAsync(P.x.get(), x, bytes, hipMemcpyDeviceToDevice, s));
    P.graph.launch(s);
    NLHIP_CHECK(hipMemcpyAsync(y, P.y.get(), bytes, hipMemcpyDeviceToDevice, s));
    // the next application (maybe on another stream) reuses x, w, y
    NLHIP_CHECK(hipStreamSynchronize(s));
}

void precond_apply(const Precond& P, uint32_t n, const double* in, double* out, hipStream_t s) {
    if (P.ssor) {
        if (ssor_n(*P.ssor) != n) throw Error(NLHIP_ERR_INVALID, "preconditioner size mismatch");
        ssor_apply(*P.ssor, in, out, s);
    } else if (P.dinv) {
        NLHIP_CHECK(blas_dmul(n, P.dinv, in, out, s));
    } else {
        NLHIP_CHECK(hipMemcpyAsync(out, in, size_t(n) * 8, hipMemcpyDeviceToDevice, s));
    }
}

}  // namespace nlhip
