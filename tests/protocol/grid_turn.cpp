// Turns of csrc/grid_turn.h: who waits, in which order, what a wait that runs
// out leaves behind, and that there is one holder at a time.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <thread>
#include <vector>

#include "grid_turn.h"

using namespace nlhip;
using Wait = GridTurn::Wait;
using std::chrono::milliseconds;

#define CHECK(x)                                                    \
    do {                                                            \
        if (!(x)) {                                                 \
            std::printf("line %d: %s\n", __LINE__, #x);             \
            std::exit(1);                                           \
        }                                                           \
    } while (0)

// Starts a thread that takes the turn, notes its number and gives it back.
struct Asker {
    std::thread t;
    Asker(GridTurn& g, Wait w, milliseconds limit, std::vector<int>& order, std::mutex& m, int id,
          std::atomic<int>& missed)
        : t([&g, w, limit, &order, &m, id, &missed] {
              GridTurn::Hold h = g.take(w, limit);
              std::lock_guard<std::mutex> lock(m);
              if (h) order.push_back(id);
              else ++missed;
          }) {}
};

int main() {
    const milliseconds none(0), shorter(30), longer(20000);
    GridTurn g;
    {
        GridTurn::Hold a = g.take(Wait::Never);
        CHECK(a);
        CHECK(!g.take(Wait::Never) && !g.take(Wait::ForLarge, longer));  // it is not large
        CHECK(!g.take(Wait::Large, shorter));                           // runs out
        a = GridTurn::Hold();
        a = g.take(Wait::ForLarge, none);  // free again, nobody in line
        CHECK(a);
    }
    {
        GridTurn::Hold a = g.take(Wait::Large);
        CHECK(a && !g.take(Wait::Never) && !g.take(Wait::ForLarge, shorter));
    }
    CHECK(g.take(Wait::Never));
    // in the order of asking; one in the middle gives up first
    {
        std::vector<int> order;
        std::mutex m;
        std::atomic<int> missed{0};
        GridTurn::Hold a = g.take(Wait::Large);
        std::vector<Asker> all;
        all.reserve(5);
        const Wait w[5] = {Wait::Large, Wait::ForLarge, Wait::Large, Wait::ForLarge, Wait::Large};
        for (int i = 0; i < 5; ++i) {
            all.emplace_back(g, w[i], i == 1 ? shorter : longer, order, m, i, missed);
            std::this_thread::sleep_for(milliseconds(20));
        }
        std::this_thread::sleep_for(milliseconds(50));
        CHECK(missed == 1 && !g.take(Wait::Never));
        a = GridTurn::Hold();
        for (Asker& x : all) x.t.join();
        CHECK((order == std::vector<int>{0, 2, 3, 4}));
        CHECK(g.take(Wait::Never));
    }
    // one holder at a time
    std::atomic<int> inside{0}, taken{0}, bad{0};
    std::vector<std::thread> all;
    for (int i = 0; i < 8; ++i)
        all.emplace_back([&, i] {
            for (int k = 0; k < 2000; ++k) {
                GridTurn::Hold h = g.take(Wait(i % 3), milliseconds(i % 2 ? 0 : 5));
                if (!h) continue;
                if (inside.fetch_add(1) != 0) ++bad;
                ++taken;
                inside.fetch_sub(1);
            }
        });
    for (std::thread& t : all) t.join();
    CHECK(bad == 0 && taken > 0 && g.take(Wait::Never));
    std::printf("taken %d\n", int(taken));
    return 0;
}
