// Brick index of particles that keep their own order (the FP64 container, the differentiable
// run): the particles of every 8^3-cell brick as a list of particle numbers, and the LDS
// windows of the deposits that walk those lists.
//
// A particle's atomics into the field cost 8 to 48 global transactions (FP64: 40 G atomics/s
// on particles in lattice order, 23 on random ones); summed in an LDS window per brick first
// (1500 G FP64 LDS atomics/s on random nodes, against 200 for FP32 ones), only the window's
// nodes go to the field, in rows (100 G atomics/s).  The index costs 12 bytes per particle.
//
// Building it: brick_count_kernel counts the cells in particle order (brick_rank: the
// particle's place among its brick's, one global atomic per brick and wave), one or two scan
// kernels turn the counts into starts (and clear them for the next time), and
// brick_list_kernel writes each particle's number at start + place.  Counted in particle order
// a list consists of runs of consecutive particles, which the kernels that walk it read in
// whole lines; places given by a kernel that walks the old lists break the runs up from step
// to step (256^3 FP64 particles in brick order: the gather went from 0.73 to 1.3 ms in 400
// steps).  Bricks at the upper faces are partial when 8 does not
// divide N.
#pragma once

#include "common.hpp"

namespace lf2mi {

static constexpr int BRK = 8;          // brick edge (cells)
static constexpr int BRK_ITEM = 1024;  // particles of one item

struct BrickIndex {
    int N, NB, lgN;       // lgN: log2 N when N is a power of two, else -1
    int nbk;
    const int *start;     // [nbk + 1] first list entry of each brick
    const int *istart;    // [nbk + 1] first item of each brick (an item: up to BRK_ITEM entries)
    const int *item;      // item -> brick
    const int *list;      // particle numbers, brick by brick
};

// writable side, with the scratch of the build
struct BrickBuild {
    int *start, *istart, *item, *list;
    int *count;           // [nbk], zero between builds
    int *rank;            // [np] place of a particle in its brick
    int *bsum;            // [2 * blocks] totals of the scan's blocks
};

__device__ __forceinline__ void brick_decode(int cell, int N, int lgN, int &x, int &y, int &z) {
    if (lgN >= 0) {
        x = cell & (N - 1);
        y = (cell >> lgN) & (N - 1);
        z = cell >> (2 * lgN);
    } else {
        x = cell % N;
        y = (cell / N) % N;
        z = cell / (N * N);
    }
}
__device__ __forceinline__ int brick_of(int x, int y, int z, int NB) {
    return (x / BRK) + NB * ((y / BRK) + NB * (z / BRK));
}

// place of a particle among those of its brick so far: lanes of a wave with the same brick
// share one atomic, and the groups' atomics go out together after the groups are found (one
// round trip per wave instead of one per group: counting 16.8 M particles in lattice order,
// 8 bricks to a wave, took 358 us that way).  Every lane of the wave calls it.
__device__ __forceinline__ int brick_rank(int *__restrict__ count, int brick, bool active) {
    unsigned long long todo = __ballot(active);
    const int lane = __lane_id();
    int first = lane, place = 0, size = 0;
    while (todo) {
        const int leader = __ffsll((long long)todo) - 1;
        const int key = __builtin_amdgcn_readlane(brick, leader);
        const unsigned long long grp = __ballot(active && brick == key);
        if (active && brick == key) {
            first = leader;
            place = __popcll(grp & ((1ull << lane) - 1ull));
            size = __popcll(grp);
        }
        todo &= ~grp;
    }
    int base = 0;
    if (active && lane == first) base = atomicAdd(&count[brick], size);
    return __shfl(base, first) + place;
}

// inclusive scan over a wave
__device__ __forceinline__ int wave_scan(int v) {
    const int lane = __lane_id();
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(v, o);
        if (lane >= o) v += y;
    }
    return v;
}
// exclusive scans of two values over a workgroup of WG threads; totals in ta, tb
template <int WG>
__device__ __forceinline__ void block_scan2(int &a, int &b, int &ta, int &tb, int *sh) {
    const int lane = __lane_id(), wave = threadIdx.x >> 6;
    const int ia = wave_scan(a), ib = wave_scan(b);
    if (lane == 63) {
        sh[wave] = ia;
        sh[WG / 64 + wave] = ib;
    }
    __syncthreads();
    int pa = 0, pb = 0;
    ta = tb = 0;
#pragma unroll
    for (int w = 0; w < WG / 64; ++w) {
        const int va = sh[w], vb = sh[WG / 64 + w];
        if (w < wave) {
            pa += va;
            pb += vb;
        }
        ta += va;
        tb += vb;
    }
    __syncthreads();
    a = pa + ia - a;
    b = pb + ib - b;
}

// ---- scans of the brick counts
// A block takes BS_CHUNK bricks.  With one block the second kernel does everything; otherwise
// the first kernel leaves each block's totals and every block of the second sums those before
// its own (at most 4096 blocks).  The second kernel writes starts, item starts and the
// item -> brick table (threads over the block's items, whose brick a binary search in LDS
// finds: a brick of thousands of items is written by the whole block) and clears the counts.
static constexpr int BS_WG = 256, BS_PER = 4, BS_CHUNK = BS_WG * BS_PER;

static __global__ __launch_bounds__(BS_WG) void brick_sums_kernel(const int *__restrict__ count, int n,
                                                                  int *__restrict__ bsum) {
    __shared__ int sh[2 * BS_WG / 64];
    const int base = blockIdx.x * BS_CHUNK + threadIdx.x * BS_PER;
    int a = 0, b = 0, ta, tb;
#pragma unroll
    for (int k = 0; k < BS_PER; ++k) {
        const int c = base + k < n ? count[base + k] : 0;
        a += c;
        b += (c + BRK_ITEM - 1) / BRK_ITEM;
    }
    block_scan2<BS_WG>(a, b, ta, tb, sh);
    if (threadIdx.x == 0) {
        bsum[2 * blockIdx.x] = ta;
        bsum[2 * blockIdx.x + 1] = tb;
    }
}

static __global__ __launch_bounds__(BS_WG) void brick_starts_kernel(int *__restrict__ count, int n,
                                                                    const int *__restrict__ bsum,
                                                                    int *__restrict__ start, int *__restrict__ istart,
                                                                    int *__restrict__ item) {
    __shared__ int sh[2 * BS_WG / 64];
    __shared__ int si[BS_CHUNK + 1];
    const int base = blockIdx.x * BS_CHUNK + threadIdx.x * BS_PER;
    int c[BS_PER], a = 0, b = 0, ta, tb;
#pragma unroll
    for (int k = 0; k < BS_PER; ++k) {
        c[k] = base + k < n ? count[base + k] : 0;
        a += c[k];
        b += (c[k] + BRK_ITEM - 1) / BRK_ITEM;
    }
    int oa = 0, ob = 0;  // totals of the blocks before this one
    if (blockIdx.x > 0) {
        int pa = 0, pb = 0;
        for (int k = threadIdx.x; k < (int)blockIdx.x; k += BS_WG) {
            pa += bsum[2 * k];
            pb += bsum[2 * k + 1];
        }
        block_scan2<BS_WG>(pa, pb, oa, ob, sh);
    }
    block_scan2<BS_WG>(a, b, ta, tb, sh);
    a += oa;
    b += ob;
#pragma unroll
    for (int k = 0; k < BS_PER; ++k) {
        const int i = base + k;
        si[threadIdx.x * BS_PER + k] = b;
        if (i < n) {
            start[i] = a;
            istart[i] = b;
            count[i] = 0;
        }
        a += c[k];
        b += (c[k] + BRK_ITEM - 1) / BRK_ITEM;
    }
    if (threadIdx.x == 0) {
        si[BS_CHUNK] = ob + tb;
        if (blockIdx.x + 1 == gridDim.x) {
            start[n] = oa + ta;
            istart[n] = ob + tb;
        }
    }
    __syncthreads();
    for (int i = ob + (int)threadIdx.x; i < ob + tb; i += BS_WG) {
        int lo = 0, hi = BS_CHUNK;  // the last brick whose first item is <= i
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (si[mid] <= i) lo = mid;
            else hi = mid;
        }
        // bricks without items share the next brick's start: the last of them is the owner
        item[i] = blockIdx.x * BS_CHUNK + lo;
    }
}

inline int brick_blocks(int64_t nbk) { return (int)((nbk + BS_CHUNK - 1) / BS_CHUNK); }

// starts, items and (cleared) counts of `n` bricks
inline int brick_scan(int *count, int n, int *bsum, int *start, int *istart, int *item, hipStream_t st) {
    const int nb = brick_blocks(n);
    if (nb > 1) {
        brick_sums_kernel<<<nb, BS_WG, 0, st>>>(count, n, bsum);
        LF2MI_LAUNCHED();
    }
    brick_starts_kernel<<<nb, BS_WG, 0, st>>>(count, n, bsum, start, istart, item);
    LF2MI_LAUNCHED();
    return LF2MI_OK;
}

static __global__ __launch_bounds__(256) void brick_count_kernel(int64_t np, const int32_t *__restrict__ cell, int N,
                                                                 int NB, int lgN, int *__restrict__ count,
                                                                 int *__restrict__ rank) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const bool in = i < np;
    int x = 0, y = 0, z = 0;
    if (in) brick_decode(cell[i], N, lgN, x, y, z);
    const int r = brick_rank(count, brick_of(x, y, z, NB), in);
    if (in) rank[i] = r;
}

static __global__ __launch_bounds__(256) void brick_list_kernel(int64_t np, const int32_t *__restrict__ cell, int N,
                                                                int NB, int lgN, const int *__restrict__ start,
                                                                const int *__restrict__ rank, int *__restrict__ list) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= np) return;
    int x, y, z;
    brick_decode(cell[i], N, lgN, x, y, z);
    list[start[brick_of(x, y, z, NB)] + rank[i]] = (int)i;
}

// the index of the particles whose cells are in `cell` and whose places are in B.rank already
inline int brick_build_ranked(const int32_t *cell, int64_t np, int N, const BrickBuild &B, hipStream_t st) {
    const int NB = (N + BRK - 1) / BRK, lgN = is_pow2(N) ? __builtin_ctz((unsigned)N) : -1;
    if (int rc = brick_scan(B.count, NB * NB * NB, B.bsum, B.start, B.istart, B.item, st)) return rc;
    brick_list_kernel<<<blocks_for(np, 256), 256, 0, st>>>(np, cell, N, NB, lgN, B.start, B.rank, B.list);
    LF2MI_LAUNCHED();
    return LF2MI_OK;
}
inline int brick_build(const int32_t *cell, int64_t np, int N, const BrickBuild &B, hipStream_t st) {
    const int NB = (N + BRK - 1) / BRK, lgN = is_pow2(N) ? __builtin_ctz((unsigned)N) : -1;
    brick_count_kernel<<<blocks_for(np, 256), 256, 0, st>>>(np, cell, N, NB, lgN, B.count, B.rank);
    LF2MI_LAUNCHED();
    return brick_build_ranked(cell, np, N, B, st);
}

inline BrickIndex brick_view(const BrickBuild &B, int N) {
    BrickIndex V;
    V.N = N;
    V.NB = (N + BRK - 1) / BRK;
    V.lgN = is_pow2(N) ? __builtin_ctz((unsigned)N) : -1;
    V.nbk = V.NB * V.NB * V.NB;
    V.start = B.start;
    V.istart = B.istart;
    V.item = B.item;
    V.list = B.list;
    return V;
}
// items there can be, and workgroups of a kernel that takes one item each
inline int64_t brick_items(int64_t nbk, int64_t np) { return nbk + np / BRK_ITEM + 1; }

// a group of MERGE consecutive items of one brick: the workgroup of the first takes them all.
// Uniform over the workgroup; false when there is nothing to do.
struct BrickRange {
    int b, p0, p1, ox, oy, oz;
};
template <int MERGE>
__device__ __forceinline__ bool brick_range(const BrickIndex &V, int it, BrickRange &r) {
    if (it >= V.istart[V.nbk]) return false;
    r.b = V.item[it];
    const int k = it - V.istart[r.b];
    if (k % MERGE != 0) return false;
    r.p0 = V.start[r.b] + k * BRK_ITEM;
    r.p1 = min(r.p0 + MERGE * BRK_ITEM, V.start[r.b + 1]);
    r.ox = (r.b % V.NB) * BRK;
    r.oy = ((r.b / V.NB) % V.NB) * BRK;
    r.oz = (r.b / (V.NB * V.NB)) * BRK;
    return true;
}

__device__ __forceinline__ int brick_wrap(int v, int N) { return v < 0 ? v + N : (v >= N ? v - N : v); }

// FP64 add into an LDS window (ds_add_f64)
__device__ __forceinline__ void lds_add(double *p, double v) { unsafeAtomicAdd(p, v); }

}  // namespace lf2mi
