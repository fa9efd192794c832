// Brick index of particles that keep their own order (the FP64 container, the differentiable
// run): the particles of every 8^3-cell brick as a list of particle numbers, and the LDS
// windows of the deposits that walk those lists.
//
// A particle's atomics into the field cost 8 to 48 global transactions (FP64: 40 G atomics/s
// on particles in lattice order, 23 on random ones); summed in an LDS window per brick first
// (1500 G FP64 LDS atomics/s on random nodes, against 200 for FP32 ones), only the window's
// nodes go to the field, in rows (100 G atomics/s).  The index costs 8 bytes per particle (list and
// rank) and about 16 per brick, an order of the particles beside it 4 (their places) to 12.
//
// Building it: brick_count_kernel counts the cells in particle order and leaves each particle's
// place among its brick's (one global atomic per brick and workgroup), one or two scan
// kernels turn the counts into starts (and clear them for the next time), and
// brick_list_kernel writes each particle's number at start + place.  Counted in particle order
// a list consists of runs of consecutive particles, which the kernels that walk it read in
// whole lines; places given by a kernel that walks the old lists break the runs up from step
// to step (256^3 FP64 particles in brick order: the gather went from 0.73 to 1.3 ms in 400
// steps).  Bricks at the upper faces are partial when 8 does not
// divide N.
#pragma once

#include "brick_run.hpp"
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

// the arrays of a scan of the brick counts (brick_scan)
struct BrickScan {
    int *count;                  // cleared
    int *bsum;                   // scratch, 3 per block
    int *start, *istart, *item;
    int *cursor;                 // copy of the starts, or null
    int2 *group;                 // (brick, k): particles [k group_p, (k + 1) group_p) of a brick with
    int *ngroup;                 // dense_min or more, and their number; null without
    int dense_min, group_p;
    // runs of sparse bricks along x: (first particle, past the last, first brick, bricks), at
    // most chunk_w bricks of a row with 1 to sparse_max - 1 particles each; null without
    int4 *chunk;
    int *nchunk;                 // their number, and a counter of claims (cleared)
    int NB, sparse_max, chunk_w;
};

// writable side, with the scratch of the build
struct BrickBuild {
    int *start, *istart, *item, *list;
    int *count;           // [nbk], zero between builds
    int *rank;            // [np] place of a particle in its brick
    int *bsum;            // [3 * blocks] totals of the scan's blocks
    BrickScan scan() const {
        BrickScan S{};
        S.count = count;
        S.bsum = bsum;
        S.start = start;
        S.istart = istart;
        S.item = item;
        return S;
    }
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

// the groups of lanes of a wave with the same brick: a lane's group's first lane, its place in the
// group and the group's size.  Every lane of the wave calls it.
__device__ __forceinline__ void brick_groups(int brick, bool active, int &first, int &place, int &size) {
    unsigned long long todo = __ballot(active);
    const int lane = __lane_id();
    first = lane;
    place = size = 0;
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
}

// place of a particle among those of its brick so far: lanes of a wave with the same brick
// share one atomic, and the groups' atomics go out together after the groups are found (one
// round trip per wave instead of one per group: counting 16.8 M particles in lattice order,
// 8 bricks to a wave, took 358 us that way).  Every lane of the wave calls it.
__device__ __forceinline__ int brick_rank(int *__restrict__ count, int brick, bool active) {
    int first, place, size;
    brick_groups(brick, active, first, place, size);
    int base = 0;
    if (active && (int)__lane_id() == first) base = atomicAdd(&count[brick], size);
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
// exclusive scans of K values over a workgroup of WG threads; totals in tot
template <int WG, int K>
__device__ __forceinline__ void block_scan(int (&v)[K], int (&tot)[K], int *sh) {
    const int lane = __lane_id(), wave = threadIdx.x >> 6;
    int incl[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        incl[k] = wave_scan(v[k]);
        if (lane == 63) sh[k * (WG / 64) + wave] = incl[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) {
        int before = 0, t = 0;
#pragma unroll
        for (int w = 0; w < WG / 64; ++w) {
            const int x = sh[k * (WG / 64) + w];
            if (w < wave) before += x;
            t += x;
        }
        tot[k] = t;
        v[k] = before + incl[k] - v[k];
    }
    __syncthreads();
}

// ---- scans of the brick counts
// A block takes BS_CHUNK bricks.  With one block the second kernel does everything; otherwise
// the first kernel leaves each block's totals and every block of the second sums those before
// its own (at most 4096 blocks).  The second kernel writes starts, item starts and the
// item -> brick table (threads over the block's items, whose brick a binary search in LDS
// finds: a brick of thousands of items is written by the whole block, where one thread per
// brick took 106 us at 512^3 with dense blobs) and clears the counts.  A container that
// scatters its particles also gets a copy of the starts to claim places from and a list of the
// dense bricks' groups, and chunks of sparse bricks.  (Five launches, a list kernel for each of
// the two and four fills before: 51 us a step at 256^3, 190 us at 512^3 with dense blobs.)
static constexpr int BS_WG = 256, BS_PER = 4, BS_CHUNK = BS_WG * BS_PER;

__device__ __forceinline__ void brick_sizes(const BrickScan &S, int c, int (&v)[3]) {
    v[0] = c;
    v[1] = (c + BRK_ITEM - 1) / BRK_ITEM;
    v[2] = S.group && c >= S.dense_min ? (c + S.group_p - 1) / S.group_p : 0;
}

static __global__ __launch_bounds__(BS_WG) void brick_sums_kernel(BrickScan S, int n) {
    __shared__ int sh[3 * BS_WG / 64];
    const int base = blockIdx.x * BS_CHUNK + threadIdx.x * BS_PER;
    int a[3] = {0, 0, 0}, tot[3];
#pragma unroll
    for (int k = 0; k < BS_PER; ++k) {
        int v[3];
        brick_sizes(S, base + k < n ? S.count[base + k] : 0, v);
        for (int q = 0; q < 3; ++q) a[q] += v[q];
    }
    block_scan<BS_WG>(a, tot, sh);
    if (S.chunk && blockIdx.x == 0 && threadIdx.x == 0) S.nchunk[0] = 0;
    if (threadIdx.x < 3) S.bsum[3 * blockIdx.x + threadIdx.x] = threadIdx.x == 0 ? tot[0] : (threadIdx.x == 1 ? tot[1] : tot[2]);
}

// inclusive maxima over a workgroup: on entry the largest of the thread's own values, on exit
// the largest of all threads before it (0 for none)
template <int WG> __device__ __forceinline__ int block_max_before(int v, int *sh) {
    const int lane = __lane_id(), wave = threadIdx.x >> 6;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(v, o);
        if (lane >= o) v = max(v, y);
    }
    if (lane == 63) sh[wave] = v;
    __syncthreads();
    int before = 0;
    for (int w = 0; w < wave; ++w) before = max(before, sh[w]);
    const int up = __shfl_up(v, 1);
    __syncthreads();
    return lane > 0 ? max(before, up) : before;
}

static __global__ __launch_bounds__(BS_WG) void brick_starts_kernel(BrickScan S, int n) {
    __shared__ int sh[4 * BS_WG / 64];
    __shared__ int si[BS_CHUNK + 1];          // item starts
    __shared__ int ss[BS_CHUNK + 1];          // starts
    __shared__ unsigned char tk[BS_CHUNK];    // 1: a sparse brick, 2: one at the start of a row
    __shared__ int cbase;
    const int base = blockIdx.x * BS_CHUNK + threadIdx.x * BS_PER, l0 = threadIdx.x * BS_PER;
    int c[BS_PER], a[4] = {0, 0, 0, 0}, tot[4];
    int first[BS_PER], last = 0;  // first brick of the run a brick belongs to, 1-based
#pragma unroll
    for (int k = 0; k < BS_PER; ++k) {
        int v[3];
        c[k] = base + k < n ? S.count[base + k] : 0;
        brick_sizes(S, c[k], v);
        for (int q = 0; q < 3; ++q) a[q] += v[q];
        if (S.chunk) {
            const bool take = c[k] > 0 && c[k] < S.sparse_max, row = (base + k) % S.NB == 0;
            tk[l0 + k] = take ? (row ? 2 : 1) : 0;
            // a run begins after a brick that is not sparse, and with a row or the block
            if (!take) last = l0 + k + 2;
            else if (row || l0 + k == 0) last = l0 + k + 1;
            first[k] = last;
        }
    }
    unsigned heads = 0u;  // bricks that begin a chunk
    if (S.chunk) {
        const int before = block_max_before<BS_WG>(last, sh);
#pragma unroll
        for (int k = 0; k < BS_PER; ++k)
            if (c[k] > 0 && c[k] < S.sparse_max) {
                const int pos = l0 + k + 1 - max(first[k], before);
                if (pos % S.chunk_w == 0) heads |= 1u << k;
            }
        a[3] = __popc(heads);
    }
    int off[3] = {0, 0, 0};  // totals of the blocks before this one
    if (blockIdx.x > 0) {
        int p[3] = {0, 0, 0};
        for (int k = threadIdx.x; k < (int)blockIdx.x; k += BS_WG)
            for (int q = 0; q < 3; ++q) p[q] += S.bsum[3 * k + q];
        block_scan<BS_WG>(p, off, sh);
    }
    block_scan<BS_WG>(a, tot, sh);
    for (int q = 0; q < 3; ++q) a[q] += off[q];
#pragma unroll
    for (int k = 0; k < BS_PER; ++k) {
        const int i = base + k;
        si[l0 + k] = a[1];
        ss[l0 + k] = a[0];
        int v[3];
        brick_sizes(S, c[k], v);
        if (i < n) {
            S.start[i] = a[0];
            S.istart[i] = a[1];
            S.count[i] = 0;
            if (S.cursor) S.cursor[i] = a[0];
            for (int g = 0; g < v[2]; ++g) S.group[a[2] + g] = make_int2(i, g);
        }
        for (int q = 0; q < 3; ++q) a[q] += v[q];
    }
    if (threadIdx.x == 0) {
        si[BS_CHUNK] = off[1] + tot[1];
        ss[BS_CHUNK] = off[0] + tot[0];
        if (S.chunk) {
            if (gridDim.x == 1) S.nchunk[0] = tot[3];
            cbase = gridDim.x == 1 ? 0 : (tot[3] ? atomicAdd(&S.nchunk[0], tot[3]) : 0);
        }
        if (blockIdx.x + 1 == gridDim.x) {
            S.start[n] = off[0] + tot[0];
            S.istart[n] = off[1] + tot[1];
            if (S.group) S.ngroup[0] = off[2] + tot[2];
            if (S.chunk) S.nchunk[1] = 0;
        }
    }
    __syncthreads();
    if (S.chunk) {
        int at = cbase + a[3];
#pragma unroll
        for (int k = 0; k < BS_PER; ++k) {
            if (!((heads >> k) & 1u)) continue;
            int e = l0 + k + 1;
            while (e < BS_CHUNK && e < l0 + k + S.chunk_w && tk[e] == 1) ++e;
            S.chunk[at++] = make_int4(ss[l0 + k], ss[e], base + k, e - (l0 + k));
        }
    }
    for (int i = off[1] + (int)threadIdx.x; i < off[1] + tot[1]; i += BS_WG) {
        int lo = 0, hi = BS_CHUNK;  // the last brick whose first item is <= i
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (si[mid] <= i) lo = mid;
            else hi = mid;
        }
        // bricks without items share the next brick's start: the last of them is the owner
        S.item[i] = blockIdx.x * BS_CHUNK + lo;
    }
}

inline int brick_blocks(int64_t nbk) { return (int)((nbk + BS_CHUNK - 1) / BS_CHUNK); }

inline int brick_scan(const BrickScan &S, int n, hipStream_t st) {
    const int nb = brick_blocks(n);
    if (nb > 1) {
        brick_sums_kernel<<<nb, BS_WG, 0, st>>>(S, n);
        LF2MI_LAUNCHED();
    }
    brick_starts_kernel<<<nb, BS_WG, 0, st>>>(S, n);
    LF2MI_LAUNCHED();
    return LF2MI_OK;
}

// Counts and ranks of PER particles per thread.  The groups of a workgroup's waves meet in an LDS hash
// table of their bricks (twice as many slots as there can be bricks), and a brick takes one global
// atomic per workgroup: with one per wave the counters of crowded bricks, a few lines, were the bound
// (2 M clustered particles on 64^3: 82 us).
template <int PER>
static __global__ __launch_bounds__(256) void brick_count_kernel(int64_t np, const int32_t *__restrict__ cell, int N,
                                                                 int NB, int lgN, int *__restrict__ count,
                                                                 int *__restrict__ rank) {
    constexpr int HT = 512 * PER, HASH = PER == 4 ? 21 : 23;  // slots, and the shift to the key's top bits
    static_assert(HT == 1 << (32 - HASH), "table size");
    __shared__ int hkey[HT];
    __shared__ int hval[HT];  // the bricks' particles so far, then their base in the brick
    for (int i = threadIdx.x; i < HT; i += 256) {
        hkey[i] = -1;
        hval[i] = 0;
    }
    const int64_t i0 = (int64_t)blockIdx.x * (256 * PER) + threadIdx.x;
    int brick[PER], ent[PER], place[PER];
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const int64_t i = i0 + 256 * k;
        brick[k] = -1;
        if (i < np) {
            int x, y, z;
            brick_decode(cell[i], N, lgN, x, y, z);
            brick[k] = brick_of(x, y, z, NB);
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        int first, size, e = 0, base = 0;
        brick_groups(brick[k], brick[k] >= 0, first, place[k], size);
        if (brick[k] >= 0 && (int)__lane_id() == first) {
            e = (int)(((unsigned)brick[k] * 2654435761u) >> HASH);
            for (;;) {
                const int old = atomicCAS(&hkey[e], -1, brick[k]);
                if (old == -1 || old == brick[k]) break;
                e = (e + 1) & (HT - 1);
            }
            base = atomicAdd(&hval[e], size);
        }
        ent[k] = __shfl(e, first);
        place[k] += __shfl(base, first);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < HT; i += 256)
        if (hkey[i] >= 0) hval[i] = atomicAdd(&count[hkey[i]], hval[i]);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const int64_t i = i0 + 256 * k;
        if (i < np) rank[i] = hval[ent[k]] + place[k];
    }
}
// four particles per thread where that still gives every CU four workgroups
inline void brick_count(int64_t np, const int32_t *cell, int N, int NB, int lgN, const BrickBuild &B, hipStream_t st) {
    if (np < 1024 * 1024) brick_count_kernel<1><<<blocks_for(np, 256), 256, 0, st>>>(np, cell, N, NB, lgN, B.count, B.rank);
    else brick_count_kernel<4><<<blocks_for(np, 1024), 256, 0, st>>>(np, cell, N, NB, lgN, B.count, B.rank);
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
    if (int rc = brick_scan(B.scan(), NB * NB * NB, st)) return rc;
    brick_list_kernel<<<blocks_for(np, 256), 256, 0, st>>>(np, cell, N, NB, lgN, B.start, B.rank, B.list);
    LF2MI_LAUNCHED();
    return LF2MI_OK;
}
inline int brick_build(const int32_t *cell, int64_t np, int N, const BrickBuild &B, hipStream_t st) {
    const int NB = (N + BRK - 1) / BRK, lgN = is_pow2(N) ? __builtin_ctz((unsigned)N) : -1;
    brick_count(np, cell, N, NB, lgN, B, st);
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

// a group of `merge` (a power of two) consecutive items of one brick: the workgroup of the first takes them all.
// Uniform over the workgroup; false when there is nothing to do.
struct BrickRange {
    int b, p0, n, ox, oy, oz;  // list entries p0 + [0, n)
};
__device__ __forceinline__ bool brick_range(const BrickIndex &V, int it, int merge, BrickRange &r) {
    if (it >= V.istart[V.nbk]) return false;
    r.b = V.item[it];
    const int k = it - V.istart[r.b];
    if ((k & (merge - 1)) != 0) return false;
    const BrickRun e = brick_run(V.start[r.b], V.start[r.b + 1], k * BRK_ITEM, merge * BRK_ITEM);
    r.p0 = e.p0;
    r.n = e.n;
    r.ox = (r.b % V.NB) * BRK;
    r.oy = ((r.b / V.NB) % V.NB) * BRK;
    r.oz = (r.b / (V.NB * V.NB)) * BRK;
    return true;
}

__device__ __forceinline__ int brick_wrap(int v, int N) { return v < 0 ? v + N : (v >= N ? v - N : v); }

// FP64 add into an LDS window (ds_add_f64)
__device__ __forceinline__ void lds_add(double *p, double v) { unsafeAtomicAdd(p, v); }

}  // namespace lf2mi
