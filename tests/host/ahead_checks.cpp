// Checks of in_turn (host_ahead.h): every result used once, in order, on the calling thread; no more
// results at once than allowed; exceptions and an early end.
#include <atomic>
#include <cstdio>
#include <stdexcept>
#include <thread>
#include <vector>

#include "../../cfd_solver_withcuda_amd/csrc/host_ahead.h"

static std::atomic<int> live{0}, most{0};

struct Made {
    int value = -1;
    bool counted = false;
    Made() = default;
    explicit Made(int v) : value(v), counted(true) {
        const int now = ++live;
        for (int m = most; now > m && !most.compare_exchange_weak(m, now);) {
        }
    }
    Made(Made &&o) noexcept : value(o.value), counted(o.counted) { o.counted = false; }
    Made &operator=(Made &&) = delete;
    ~Made() {
        if (counted) live--;
    }
};

static int fails = 0;
#define CHECK(x)                                                              \
    do {                                                                      \
        if (!(x)) {                                                           \
            std::printf("failed: %s (line %d)\n", #x, __LINE__);              \
            fails++;                                                          \
        }                                                                     \
    } while (0)

int main() {
    const auto me = std::this_thread::get_id();
    for (int n : {0, 1, 5, 64})
        for (int ahead : {0, 1, 3, 15, 100}) {
            live = most = 0;
            std::vector<int> used;
            cfd::in_turn(n, ahead, [](int i) { return Made(i * i); }, [&](int i, Made &m) {
                CHECK(m.value == i * i && std::this_thread::get_id() == me);
                used.push_back(i);
                return true;
            });
            CHECK((int)used.size() == n && live == 0 && most <= ahead + 1);
            for (int i = 0; i < (int)used.size(); i++) CHECK(used[i] == i);
            // an early end
            int last = -1;
            cfd::in_turn(n, ahead, [](int i) { return Made(i); }, [&](int i, Made &) {
                last = i;
                return i < 2;
            });
            CHECK(last == (n > 2 ? 2 : n - 1) && live == 0);
            // an exception: at its own turn
            bool caught = false;
            last = -1;
            try {
                cfd::in_turn(n, ahead, [](int i) -> Made {
                    if (i == 3) throw std::runtime_error("three");
                    return Made(i);
                }, [&](int i, Made &) {
                    last = i;
                    return true;
                });
            } catch (const std::runtime_error &) {
                caught = true;
            }
            CHECK(caught == (n > 3) && last == (n > 3 ? 2 : n - 1) && live == 0);
        }
    std::printf("checked\n");
    return fails ? 1 : 0;
}
