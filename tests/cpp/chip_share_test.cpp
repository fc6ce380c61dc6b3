// Checks of the admission of one-launch solves to a GPU: what runs side by side, and in which order.
#include "fem_share.hpp"

#include <atomic>
#include <chrono>
#include <cstdio>
#include <memory>
#include <thread>
#include <vector>

using namespace femgpu;

namespace {

int failures = 0;
void check(bool ok, const char* what) {
    std::printf("%s: %s\n", ok ? "ok" : "FAILED", what);
    failures += !ok;
}

constexpr int kCus = 256;

// A solve asked for on a thread of its own.
struct Solve {
    std::atomic<bool> in{false}, end{false};
    std::thread thread;
    Solve(ChipShare& chip, int workgroups) {
        thread = std::thread([this, &chip, workgroups] {
            ChipShare::Use use(chip, workgroups, kCus);
            in = true;
            while (!end) std::this_thread::yield();
        });
    }
    ~Solve() { leave(); }
    bool admitted(int ms) {
        for (int i = 0; i < ms && !in; ++i) std::this_thread::sleep_for(std::chrono::milliseconds(1));
        return in;
    }
    void leave() {
        end = true;
        if (thread.joinable()) thread.join();
    }
};

constexpr int kSoon = 5000, kNever = 50;  // ms

}  // namespace

int main() {
    ChipShare chip;
    {
        Solve large(chip, 225);
        check(large.admitted(kSoon), "a large solve");
        Solve small(chip, 4), next(chip, 24);  // 29 + 1 + 3 CUs of an XCD's 32
        const bool a = small.admitted(kNever), b = next.admitted(kNever);
        check(a != b, "one of two small ones beside it, the other would need a 33rd CU of an XCD");
        large.leave();
        check(small.admitted(kSoon) && next.admitted(kSoon), "both once it has ended");
    }
    {
        Solve first(chip, 256);
        check(first.admitted(kSoon), "a solve of the whole chip");
        Solve second(chip, 256);
        check(!second.admitted(kNever), "not two of them");
        Solve small(chip, 1);
        check(!small.admitted(kNever), "a later one does not pass the one that waits");
        first.leave();
        check(second.admitted(kSoon) && !small.admitted(kNever), "first come, first served");
        second.leave();
        check(small.admitted(kSoon), "then the small one");
    }
    {
        Solve beyond(chip, 300);
        check(beyond.admitted(kSoon), "more than the chip: alone");
    }
    {
        ChipShare::Use use(chip, 256, kCus), moved;
        moved = std::move(use);
        Solve other(chip, 1);
        check(!other.admitted(kNever), "held by what it was moved to");
        moved.release();
        moved.release();
        check(other.admitted(kSoon), "released early, once");
    }
    {
        std::atomic<int> used{0}, most{0};
        std::vector<std::thread> threads;
        for (int t = 0; t < 8; ++t)
            threads.emplace_back([&, t] {
                for (int i = 0; i < 500; ++i) {
                    const int cus = 1 + (t * 7 + i) % 20;
                    ChipShare::Use use(chip, 8 * cus, kCus);
                    const int now = used += cus;
                    for (int m = most; m < now && !most.compare_exchange_weak(m, now);) {}
                    used -= cus;
                }
            });
        for (auto& t : threads) t.join();
        check(most <= 32, "never more than an XCD's CUs");
    }
    std::printf("%d failed\n", failures);
    return failures != 0;
}
