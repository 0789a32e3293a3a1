// Reads solves "n nz guess iterations limit" and prints, per solve, the launched
// iterations and the looks.  A solve of `iterations` stops at the first look
// that has launched more than that many (the launch after the last iteration
// sees the stop test), or at the limit.
#include <cstdio>

#include "look_schedule.hpp"

int main() {
    sbs::LookSchedule s;
    int n, guess, its, limit;
    long long nz;
    while (std::scanf("%d %lld %d %d %d", &n, &nz, &guess, &its, &limit) == 5) {
        s.begin(n, nz, guess != 0);
        int k = 0, looks = 0;
        bool done = false;
        while (k < limit && !done) {
            k += std::min(s.next(k), limit - k);
            ++looks;
            done = k > its;
        }
        s.end(done ? its : limit, done);
        std::printf("%d %d\n", k, looks);
    }
}
