// The stretch of a brick's particles that one workgroup takes.  Particles are numbered in 32 bits up to
// the largest int, so ends are never formed as start + length: a run is its first entry and its
// length, and loops count from 0.  No HIP in here: checked on the host.
#pragma once

namespace lf2mi {

struct BrickRun {
    int p0, n;
};

// up to `len` entries from the `at`-th of a brick whose entries are [start, end); at <= end - start
constexpr BrickRun brick_run(int start, int end, int at, int len) {
    const int left = end - start - at;
    return BrickRun{start + at, left < len ? left : len};
}

}  // namespace lf2mi
