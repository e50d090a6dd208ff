// small_place.cpp — SmallPlace (csrc/small_place.h) under threads: no XCD holds more than its CUs, launches that fit begin at once, the
// others in the order they came.
#include "small_place.h"

#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <memory>
#include <set>
#include <thread>
#include <vector>

using sli::SmallPlace;
static void check(bool ok, const char* what) {
    if (!ok) {
        std::printf("failed: %s\n", what);
        std::exit(1);
    }
}
static constexpr unsigned kMask = 0xff;
static std::unique_ptr<SmallPlace> one(SmallPlace::Chip& c, int first = 0) { return std::make_unique<SmallPlace>(c, 32, kMask, 16, 8, first); }
static std::unique_ptr<SmallPlace> all(SmallPlace::Chip& c) { return std::make_unique<SmallPlace>(c, 32, 0u, 0, 8, 0); }
template <class F>
static bool waits(F f, std::thread& t, std::atomic<bool>& done) {
    t = std::thread([&done, f] { f(), done = true; });
    std::this_thread::sleep_for(std::chrono::milliseconds(50));
    return !done;
}

int main() {
    {  // an XCD each while there are empty ones, from where each process begins; then the second halves
        SmallPlace::Chip c;
        std::vector<std::unique_ptr<SmallPlace>> p;
        std::set<int> xcds;
        for (int i = 0; i < 8; ++i) p.push_back(one(c, 5)), xcds.insert(p.back()->xcd);
        check(p[0]->xcd == 5 && p[1]->xcd == 6 && xcds.size() == 8, "XCDs of their own");
        auto beside = all(c);
        check(beside->xcd == -1, "over all XCDs beside them");
        auto b2 = all(c);
        std::atomic<bool> done{false};
        std::thread t;
        check(waits([&] { one(c); }, t, done), "no launch that reaches a full XCD begins");
        b2.reset(), beside.reset();
        t.join();
        check(done, "it begins when the place is given back");
    }
    {  // four over all XCDs fill the chip
        SmallPlace::Chip c;
        std::vector<std::unique_ptr<SmallPlace>> p;
        for (int i = 0; i < 4; ++i) p.push_back(all(c));
        std::atomic<bool> d1{false}, d2{false};
        std::thread t1, t2;
        check(waits([&] { one(c); }, t1, d1), "one waits");
        check(waits([&] { all(c); }, t2, d2), "all waits behind it");
        p.resize(2);
        t1.join(), t2.join();
    }
    {  // many threads of both kinds: never more than there are, and all end
        SmallPlace::Chip c;
        std::atomic<int> used[SmallPlace::kXcds] = {};
        std::atomic<bool> over{false};
        std::vector<std::thread> ts;
        for (int i = 0; i < 40; ++i)
            ts.emplace_back([&, i] {
                for (int k = 0; k < 50; ++k) {
                    const bool o = (i + k) % 3 != 0;
                    auto p = o ? one(c, i % 8) : all(c);
                    for (int x = 0; x < 8; ++x) {
                        const int n = o ? (x == p->xcd ? 16 : 0) : 8;
                        if ((used[x] += n) > 32) over = true;
                    }
                    std::this_thread::yield();
                    for (int x = 0; x < 8; ++x) used[x] -= o ? (x == p->xcd ? 16 : 0) : 8;
                }
            });
        for (auto& t : ts) t.join();
        check(!over, "CUs");
        for (int u : c.used) check(u == 0, "all given back");
    }
    std::puts("ok");
}
