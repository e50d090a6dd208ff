// small_place.h — which CUs the one-launch loops of small models (small_model.h) share between threads.
#pragma once
#include <condition_variable>
#include <mutex>

namespace sli {

// The workgroups of such a launch wait for each other and fill a CU each, so a launch may begin only where all of them get a CU
// beside the launches that run: `one` CUs of a single XCD (xcd, of those in `mask`), or `all` CUs of every XCD (xcd -1). A launch on one
// XCD also sends workgroups to the others, which leave at once; they too need a CU, so no XCD may be full when it begins. Threads are
// served in the order they came; the place is given back when the launch has ended.
struct SmallPlace {
    static constexpr int kXcds = 16;
    struct Chip {  // of a device
        std::mutex mu;
        std::condition_variable cv;
        int used[kXcds] = {};  // CUs by XCC_ID
        unsigned long long next = 0, serving = 0;
    };
    Chip& chip;
    const int one, all;
    int xcd = -1;
    // cus: of an XCD. first: where the search begins (processes do not see each other's launches: each begins elsewhere)
    SmallPlace(Chip& c, int cus, unsigned mask, int one_cus, int all_cus, int first) : chip(c), one(one_cus), all(all_cus) {
        std::unique_lock<std::mutex> lock(chip.mu);
        const unsigned long long mine = chip.next++;
        chip.cv.wait(lock, [&] { return mine == chip.serving && (one ? pick(cus, mask, first) : fits(cus)); });
        take(1);
        ++chip.serving;
        chip.cv.notify_all();
    }
    ~SmallPlace() {
        std::lock_guard<std::mutex> lock(chip.mu);
        take(-1);
        chip.cv.notify_all();
    }
    SmallPlace(const SmallPlace&) = delete;
    SmallPlace& operator=(const SmallPlace&) = delete;

private:
    void take(int sign) {
        for (int x = 0; x < kXcds; ++x) chip.used[x] += xcd < 0 ? sign * all : x == xcd ? sign * one : 0;
    }
    bool fits(int cus) const {
        for (int u : chip.used)
            if (u + all > cus) return false;
        return true;
    }
    bool pick(int cus, unsigned mask, int first) {  // the emptiest XCD
        xcd = -1;
        for (int i = 0; i < kXcds; ++i) {
            const int x = (first + i) % kXcds;
            if (!(mask >> x & 1)) continue;
            if (chip.used[x] >= cus) return xcd = -1, false;
            if (chip.used[x] + one <= cus && (xcd < 0 || chip.used[x] < chip.used[xcd])) xcd = x;
        }
        return xcd >= 0;
    }
};

}  // namespace sli
