#pragma once

#include <algorithm>
#include <chrono>
#include <condition_variable>
#include <cstdint>
#include <deque>
#include <mutex>
#include <utility>

namespace nlhip {

// The turn of the one kernel with grid-wide barriers that may run at a time in
// a process: two of them, each partly resident, would wait for one another.
// Turns go in the order of asking, among those that wait:
//   Never     none when it is held or waited for
//   ForLarge  waits where one that needs most of the device is ahead
//   Large     is such a one; waits
class GridTurn {
  public:
    enum class Wait { Never, ForLarge, Large };
    class Hold {  // gives the turn back; false when there is none
      public:
        Hold() = default;
        explicit Hold(GridTurn* t) : t_(t) {}
        Hold(Hold&& o) noexcept : t_(o.t_) { o.t_ = nullptr; }
        Hold& operator=(Hold&& o) noexcept {
            std::swap(t_, o.t_);
            return *this;
        }
        ~Hold() {
            if (t_) t_->give();
        }
        explicit operator bool() const { return t_ != nullptr; }

      private:
        GridTurn* t_ = nullptr;
    };
    Hold take(Wait wait, std::chrono::milliseconds limit = std::chrono::milliseconds(0));

  private:
    void give();
    std::mutex m_;
    std::condition_variable cv_;
    struct Ticket {
        uint64_t id;
        bool large;
    };
    std::deque<Ticket> waiting_;  // in order
    uint64_t next_ = 0;
    bool held_ = false, held_large_ = false;
};

inline GridTurn::Hold GridTurn::take(Wait wait, std::chrono::milliseconds limit) {
    std::unique_lock<std::mutex> lock(m_);
    const bool large = wait == Wait::Large;
    if (held_ || !waiting_.empty()) {
        bool ahead = held_ && held_large_;
        for (const Ticket& t : waiting_) ahead |= t.large;
        if (wait == Wait::Never || (!large && !ahead)) return Hold();
        const uint64_t mine = next_++;
        waiting_.push_back({mine, large});
        const bool got =
            cv_.wait_for(lock, limit, [&] { return !held_ && waiting_.front().id == mine; });
        waiting_.erase(std::find_if(waiting_.begin(), waiting_.end(),
                                    [&](const Ticket& t) { return t.id == mine; }));
        if (!got) {
            cv_.notify_all();  // perhaps it was the front of the line
            return Hold();
        }
    }
    held_ = true;
    held_large_ = large;
    return Hold(this);
}

inline void GridTurn::give() {
    {
        std::lock_guard<std::mutex> lock(m_);
        held_ = false;
    }
    cv_.notify_all();
}

}  // namespace nlhip
