// Work made ahead on other threads and used in order (part of the C-ABI translation units).
#pragma once
#include <deque>
#include <future>

namespace cfd {

// use(i, make(i)) for i = 0 .. n - 1 in turn on this thread, until one returns false. make runs on threads
// of its own, at most `ahead` results early (0: here, when its turn comes), so that no more than ahead + 1
// results exist at once. Exceptions of make come out of the turn that needs them.
template <typename Make, typename Use>
void in_turn(int n, int ahead, Make make, Use use) {
    std::deque<std::future<decltype(make(0))>> early;
    for (int i = 0, next = 0; i < n; i++) {
        // without a thread to be had a result is made when its turn comes
        const auto policy = ahead > 0 ? std::launch::async | std::launch::deferred : std::launch::deferred;
        for (; next < n && next <= i + ahead; next++) early.push_back(std::async(policy, make, next));
        auto made = early.front().get();
        early.pop_front();
        if (!use(i, made)) return;
    }
}

}  // namespace cfd
