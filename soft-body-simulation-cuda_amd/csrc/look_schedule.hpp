// When the host looks at an iterative solve that it has queued on the GPU.
// Plain C++17 (no HIP): the CPU test suite compiles it alone.
//
// A look leaves the GPU idle for about 30 us, an iteration launched after the
// solve has stopped costs it about 5.  Without a count to go by the host looks
// after 16 iterations and then after every quarter of what it has launched.  A
// solver that has just solved a system of the same size, to its stop test,
// expects about that count again and waits for nine tenths of it; but another
// right-hand side or start may need far fewer, so the first look comes after
// 128 iterations at the latest and a wait is never longer than what has been
// launched before it: a solve of c iterations launches at most
// max(128, 2 c) + 16.  (A system of 12 iterations after one of 3,000 on the
// same handle took 20.0 ms with a first look at 2,700, 0.3 ms alone.)
#pragma once

#include <algorithm>

namespace sbs {

class LookSchedule {
public:
    // A solve of this system begins (n unknowns, nz triplets, with or without a start).
    void begin(int n, long long nz, bool guess) {
        if (n != n_ || nz != nz_ || guess != guess_) learned_ = 0;
        n_ = n;
        nz_ = nz;
        guess_ = guess;
    }
    // Iterations to launch before the next look, `launched` so far.
    int next(int launched) const {
        const int expected = learned_ - learned_ / 10;
        if (launched == 0) return std::clamp(expected, kFewest, kFirstMost);
        const int wait = std::max(kFewest, launched / 4);
        return expected > launched + wait ? std::max(kFewest, std::min(expected - launched, launched)) : wait;
    }
    // It ended after `iterations`, by its stop test or (not `stopped`) by the limit.
    void end(int iterations, bool stopped) { learned_ = stopped ? iterations : 0; }

private:
    static constexpr int kFewest = 16, kFirstMost = 128;
    int n_ = 0;
    long long nz_ = 0;
    bool guess_ = false;
    int learned_ = 0;
};

}  // namespace sbs
