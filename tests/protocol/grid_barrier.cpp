// Model check of csrc/grid_barrier.h: workgroups as coroutines, every access
// to a barrier word a scheduling point, every schedule (or, with a sample
// count, that many random ones) run.  Each workgroup passes `barriers`
// barriers and then "writes"; between two of them one may give up a wait of
// its own (`quitter`).  At the end either all have written and the bit is
// clear, or none has and the bit is set: the caller goes on from the new state
// or from the old one by that bit alone.
//
//   grid_barrier WORKGROUPS BARRIERS POLLS GROUPS QUITTER(-1: none) SAMPLES(0: all)
// prints the schedules run and how many of them passed; exit status 1 and the
// schedule on a violation.
#include <ucontext.h>

#include <cstdio>
#include <cstdlib>
#include <memory>
#include <random>
#include <vector>

#include "grid_barrier.h"

using namespace nlhip;

namespace {

constexpr size_t kStack = 64 << 10;
ucontext_t g_main;
ucontext_t* g_self = nullptr;

void step() { swapcontext(g_self, &g_main); }

struct ModelWord {
    uint32_t* p;
    uint32_t load() const {
        step();
        return *p;
    }
    uint32_t add(uint32_t v) const {
        step();
        const uint32_t old = *p;
        *p += v;
        return old;
    }
    uint32_t cas(uint32_t expected, uint32_t desired) const {
        step();
        const uint32_t old = *p;
        if (old == expected) *p = desired;
        return old;
    }
    void pause() const {}
};

struct Config {
    int n, barriers;
    uint32_t polls;
    int groups, quitter;
} cfg;

uint32_t g_root, g_group[8];
bool g_done[8];
int g_written;

void workgroup(int w) {
    const int g = w % cfg.groups;
    const uint32_t size = uint32_t((cfg.n - g + cfg.groups - 1) / cfg.groups);
    ModelWord root{&g_root}, group{&g_group[g]};
    for (int e = 1; e <= cfg.barriers; ++e) {
        if (w == cfg.quitter && e == cfg.barriers) {  // a wait between barriers
            step();
            g_root |= kPersistFail;
            return;
        }
        barrier_arrive(group, root, size, uint32_t(e));
        if (!barrier_wait(root, uint32_t(cfg.groups), uint32_t(e), cfg.polls)) return;
    }
    step();
    ++g_written;
}

void entry(int w) {
    workgroup(w);
    g_done[w] = true;
    for (;;) step();
}

struct Run {
    std::vector<std::vector<char>> stacks;
    std::vector<ucontext_t> ctx;
    Run() : stacks(size_t(cfg.n), std::vector<char>(kStack)), ctx(size_t(cfg.n)) {}
    void reset() {
        g_root = 0;
        g_written = 0;
        for (int w = 0; w < 8; ++w) g_group[w] = 0, g_done[w] = false;
        for (int w = 0; w < cfg.n; ++w) {
            getcontext(&ctx[size_t(w)]);
            ctx[size_t(w)].uc_stack.ss_sp = stacks[size_t(w)].data();
            ctx[size_t(w)].uc_stack.ss_size = kStack;
            ctx[size_t(w)].uc_link = nullptr;
            makecontext(&ctx[size_t(w)], reinterpret_cast<void (*)()>(entry), 1, w);
        }
    }
    void resume(int w) {
        g_self = &ctx[size_t(w)];
        swapcontext(&g_main, g_self);
    }
    bool open() const {
        for (int w = 0; w < cfg.n; ++w)
            if (!g_done[w]) return true;
        return false;
    }
    bool ok() const {
        const bool fail = g_root & kPersistFail;
        return fail ? g_written == 0 : g_written == cfg.n;
    }
};

}  // namespace

int main(int argc, char** argv) {
    if (argc != 7) return 2;
    cfg = {std::atoi(argv[1]), std::atoi(argv[2]), uint32_t(std::atoi(argv[3])),
           std::atoi(argv[4]), std::atoi(argv[5])};
    const long samples = std::atol(argv[6]);
    if (cfg.n < 1 || cfg.n > 8 || cfg.groups < 1 || cfg.groups > cfg.n) return 2;
    Run run;
    std::vector<int> path;  // the schedule: workgroup run at each step
    std::mt19937 rng(1);
    long total = 0, passed = 0;
    for (;;) {
        run.reset();
        size_t at = 0;
        while (run.open()) {
            if (samples) {
                int w;
                do w = int(rng() % uint32_t(cfg.n));
                while (g_done[w]);
                path.push_back(w);
                run.resume(w);
                continue;
            }
            if (at == path.size()) {  // new step: the first workgroup still open
                int w = 0;
                while (g_done[w]) ++w;
                path.push_back(w);
            }
            run.resume(path[at++]);
        }
        ++total;
        passed += g_written != 0;
        if (!run.ok()) {
            std::printf("violated after %ld schedules: %d of %d wrote, bit %s; schedule", total,
                        g_written, cfg.n, g_root & kPersistFail ? "set" : "clear");
            for (int w : path) std::printf(" %d", w);
            std::printf("\n");
            return 1;
        }
        if (samples) {
            path.clear();
            if (total == samples) break;
            continue;
        }
        // next schedule in order: the last step that another workgroup could take
        for (;;) {
            if (path.empty()) {
                std::printf("schedules %ld passed %ld\n", total, passed);
                return 0;
            }
            const int last = path.back();
            path.pop_back();
            run.reset();
            for (int w : path) run.resume(w);
            int w = last + 1;
            while (w < cfg.n && g_done[w]) ++w;
            if (w < cfg.n) {
                path.push_back(w);
                break;
            }
        }
    }
    std::printf("schedules %ld passed %ld\n", total, passed);
    return 0;
}
