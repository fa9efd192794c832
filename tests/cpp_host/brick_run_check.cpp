// runs of a brick's entries (csrc/brick_run.hpp): every entry of a brick is in one run, also where
// the brick ends at the largest particle number
#include <climits>
#include <cstdio>

#include "brick_run.hpp"

int main() {
    const int len = 4096, item = 1024;
    const int ends[] = {0, 1, 4095, 4096, 4097, 9000, INT_MAX - 4096, INT_MAX - 255, INT_MAX - 1, INT_MAX};
    const int counts[] = {0, 1, 255, 1024, 4095, 4096, 4097, 8192, 20001};
    for (int end : ends)
        for (int n : counts) {
            if (n > end) continue;
            const int start = end - n;
            long long next = start;
            for (int k = 0; k * item < n; ++k) {
                if (k % (len / item) != 0) continue;  // taken by the group's first item
                const lf2mi::BrickRun r = lf2mi::brick_run(start, end, k * item, len);
                if (r.p0 != next || r.n < 1 || r.n > len) {
                    std::printf("start %d end %d k %d: %d + %d\n", start, end, k, r.p0, r.n);
                    return 1;
                }
                next = (long long)r.p0 + r.n;
            }
            if (next != end) {
                std::printf("start %d end %d: ends at %lld\n", start, end, next);
                return 1;
            }
        }
    return 0;
}
