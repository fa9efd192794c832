// Particle container, CIC deposits and the fused gather + kick + drift of the lf2mi
// library (Particles<part_simple,...> and particles/projections.hpp on one gfx950 device).
//
// F32 representation: per particle an int32 cell index x + N(y + N z) and an FP32 offset
// in cell units in [0,1) per axis (position = (cell + offset)/N, formed in FP64 when the
// particle moves), FP32 velocity, optional FP32 mass and int64 ID, in SoA arrays.
// Particles are bucketed by bricks of B^3 cells (B = 8 when N allows); a bucket is the
// unit of locality that the reference gets from its per-cell std::forward_list
// (particles/LATfield2_Particles.hpp:97-103,333).  Deposits and gathers work on "items":
// chunks of at most ITEM_P particles of one bucket, each staged through an LDS window
// of the brick's nodes.  After a drift the container is re-bucketed with a counting sort
// (histogram -> scan -> scatter into the second buffer).
//
// F64 representation: absolute FP64 positions and velocities, put into brick order at upload and
// every few drifts, with a brick index beside them (bricks.hpp): deposits sum a brick's particles
// in an FP64 LDS window, the gather reads a brick's window of phi.  Where few particles fall into
// a brick, or the index finds no room, both go particle by particle in upload order: FP64 atomics
// into the field, phi straight from HBM.  Downloads come in upload order either way.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <new>
#include <type_traits>
#include <vector>

#include "bricks.hpp"
#include "common.hpp"

namespace lf2mi {

static constexpr int ITEM_P = 1024;     // particles per item
static constexpr int DEP_WG = 256;      // deposit / gather workgroup size
static constexpr int MAXB = 8;          // largest brick edge

// ---------------------------------------------------------------- RNG (counter based)
__host__ __device__ inline uint64_t mix64(uint64_t z) {
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}
// uniform double in [0,1) from (seed, index, stream)
__host__ __device__ inline double urand(uint64_t seed, uint64_t idx, uint32_t stream) {
    const uint64_t h = mix64(seed ^ mix64(idx * 16ull + stream));
    return (double)(h >> 11) * 0x1.0p-53;
}
__device__ inline double grand(uint64_t seed, uint64_t idx, uint32_t stream) {
    // Box-Muller on two uniforms of the same counter
    double u1 = urand(seed, idx, stream);
    const double u2 = urand(seed, idx, stream + 8);
    if (u1 < 0x1.0p-60) u1 = 0x1.0p-60;
    return sqrt(-2.0 * log(u1)) * cospi(2.0 * u2);
}

// ---------------------------------------------------------------- exact FP64 helpers
// Rounded add / multiply that the compiler may not fuse into an FMA: the drift must
// round exactly like the reference's `pos += dtau * vel` (one product, one sum).
__device__ __forceinline__ double add_rn(double a, double b) {
#pragma clang fp contract(off)
    return a + b;
}
__device__ __forceinline__ double sub_rn(double a, double b) {
#pragma clang fp contract(off)
    return a - b;
}
__device__ __forceinline__ double mul_rn(double a, double b) {
#pragma clang fp contract(off)
    return a * b;
}

// ---------------------------------------------------------------- wave helpers
__device__ __forceinline__ int lane_id() { return __lane_id(); }

// wave-aggregated atomic increment: lanes with the same key share one atomic; returns
// each lane's slot (base + rank among the lanes with its key)
__device__ __forceinline__ int agg_inc(int *counters, int key, bool active) {
    unsigned long long todo = __ballot(active);
    int slot = 0;
    const int lane = lane_id();
    while (todo) {
        const int leader = __ffsll((long long)todo) - 1;
        const int lkey = __shfl(key, leader);
        const unsigned long long grp = __ballot(active && key == lkey);
        int base = 0;
        if (lane == leader) base = atomicAdd(&counters[lkey], __popcll(grp));
        base = __shfl(base, leader);
        if (active && key == lkey) slot = base + __popcll(grp & ((1ull << lane) - 1ull));
        todo &= ~grp;
    }
    return slot;
}

// ---------------------------------------------------------------- geometry helpers
struct Geo {
    int N, B, NB;
    int64_t nbk;
    int lgN, lgB;  // log2 of N and B when they are powers of two, else -1
};
// cell index x + N(y + N z) -> coordinates; shifts when N is a power of two
__device__ __forceinline__ void decode_cell(int cell, const Geo &g, int &x, int &y, int &z) {
    if (g.lgN >= 0) {
        const int m = g.N - 1;
        x = cell & m;
        y = (cell >> g.lgN) & m;
        z = cell >> (2 * g.lgN);
    } else {
        x = cell % g.N;
        y = (cell / g.N) % g.N;
        z = cell / (g.N * g.N);
    }
}
__device__ __forceinline__ int bucket_of(int cell, const Geo &g) {
    int x, y, z;
    decode_cell(cell, g, x, y, z);
    if (g.lgB >= 0) return (x >> g.lgB) + g.NB * ((y >> g.lgB) + g.NB * (z >> g.lgB));
    return (x / g.B) + g.NB * ((y / g.B) + g.NB * (z / g.B));
}
__device__ __forceinline__ int wrapi(int v, int N) { return v < 0 ? v + N : (v >= N ? v - N : v); }

// ---------------------------------------------------------------- F32 SoA buffer
struct Soa32 {
    int32_t *cell;
    float *off[3];
    float *vel[3];
    float *mass;   // may be null
    int64_t *id;   // may be null
    unsigned long long *pl;  // payload: plw 8-byte words per particle (user structs), may be null
};

// ---------------------------------------------------------------- binning (FP64 -> cell, offset)
// Particles::getPartCoord: (int)floor(pos*N) % N (particles/LATfield2_Particles.hpp:464-467).
// The offset is pos*N - floor(pos*N) rounded to FP32 and kept below 1.
__device__ __forceinline__ bool bin_one(const double p[3], int N, int &cell, float off[3]) {
    int c[3];
    bool ok = true;
    for (int d = 0; d < 3; ++d) {
        const double t = p[d] * (double)N;
        const double fl = floor(t);
        c[d] = (int)fl % N;
        if (c[d] < 0) ok = false;
        float o = (float)(t - fl);
        if (!(o < 1.0f)) o = 0x1.fffffep-1f;
        off[d] = o;
    }
    cell = ok ? c[0] + N * (c[1] + N * c[2]) : -1;
    return ok;
}

// staged FP64 input: AoS pos/vel (host layout), optional mass/id
__global__ void bin_upload_kernel(int64_t np, const double *__restrict__ pos, const double *__restrict__ vel,
                                  const double *__restrict__ mass, const int64_t *__restrict__ id,
                                  const unsigned long long *__restrict__ pl, int plw, Soa32 dst, Geo g,
                                  int *__restrict__ counts) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool in = i < np;
    int cell = -1;
    if (in) {
        const double p[3] = {pos[3 * i], pos[3 * i + 1], pos[3 * i + 2]};
        float off[3];
        bin_one(p, g.N, cell, off);
        dst.cell[i] = cell;
        for (int d = 0; d < 3; ++d) {
            dst.off[d][i] = off[d];
            dst.vel[d][i] = (float)vel[3 * i + d];
        }
        if (dst.mass) dst.mass[i] = mass ? (float)mass[i] : 1.0f;
        if (dst.id) dst.id[i] = id ? id[i] : i;
        for (int w = 0; w < plw; ++w) dst.pl[i * plw + w] = pl[i * plw + w];
    }
    const bool act = in && cell >= 0;
    agg_inc(counts, act ? bucket_of(cell, g) : 0, act);
}

// ---------------------------------------------------------------- synthetic ICs (F32 and F64)
struct IcArgs {
    int kind;  // 0 lattice, 1 uniform, 2 blobs
    int64_t np;
    int ng;
    double sigma_pos;  // box units
    double sigma_v;
    uint64_t seed;
    int nblobs;
    int64_t nclustered;
    const double *centres;   // 3 * nblobs
    const int64_t *bstart;   // nblobs + 1 prefix of blob occupancies
};

__device__ __forceinline__ void ic_pos(const IcArgs &A, int64_t i, double p[3]) {
    if (A.kind == 0) {
        const int64_t ng = A.ng;
        const int64_t ix = i % ng, iy = (i / ng) % ng, iz = i / (ng * ng);
        const double base[3] = {(double)ix / ng, (double)iy / ng, (double)iz / ng};
        for (int d = 0; d < 3; ++d) p[d] = base[d] + A.sigma_pos * grand(A.seed, i, d);
    } else if (A.kind == 1 || i >= A.nclustered) {
        for (int d = 0; d < 3; ++d) p[d] = urand(A.seed, i, 4 + d);
    } else {
        // blob of particle i: largest b with bstart[b] <= i
        int lo = 0, hi = A.nblobs;
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (A.bstart[mid] <= i) lo = mid;
            else hi = mid;
        }
        for (int d = 0; d < 3; ++d) p[d] = A.centres[3 * lo + d] + A.sigma_pos * grand(A.seed, i, d);
    }
    for (int d = 0; d < 3; ++d) {
        p[d] -= floor(p[d]);  // periodic wrap into [0, 1)
        if (p[d] >= 1.0) p[d] = 0.0;
    }
}
__device__ __forceinline__ void ic_vel(const IcArgs &A, int64_t i, double v[3]) {
    for (int d = 0; d < 3; ++d) v[d] = A.sigma_v * grand(A.seed, i, 12 + d);
}

__global__ void ic_f32_kernel(IcArgs A, Soa32 dst, Geo g, int *__restrict__ counts) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool in = i < A.np;
    int cell = -1;
    if (in) {
        double p[3], v[3];
        ic_pos(A, i, p);
        ic_vel(A, i, v);
        float off[3];
        bin_one(p, g.N, cell, off);
        dst.cell[i] = cell;
        for (int d = 0; d < 3; ++d) {
            dst.off[d][i] = off[d];
            dst.vel[d][i] = (float)v[d];
        }
        if (dst.mass) dst.mass[i] = 1.0f;
        if (dst.id) dst.id[i] = i;
    }
    const bool act = in && cell >= 0;
    agg_inc(counts, act ? bucket_of(cell, g) : 0, act);
}

struct Soa64 {
    int32_t *cell;
    double *pos[3];
    double *vel[3];
    double *mass;
    int64_t *id;
    unsigned long long *pl;  // payload, as in Soa32
};

// cell of an FP64 position (Particles::getPartCoord)
__device__ __forceinline__ int cell64(const double p[3], int N) {
    int c[3];
    for (int d = 0; d < 3; ++d) c[d] = (int)floor(p[d] * (double)N) % N;
    return c[0] + N * (c[1] + N * c[2]);
}

// Where the F64 container keeps a brick index its particles lie in brick order as they were
// uploaded (place `start of the brick + rank` for each), so that the lists of later steps,
// whose particles have moved little, still read memory nearly in order: with particles left
// in lattice order a brick's list touches 64 8-particle runs per array, and after a few
// hundred steps single particles of them (256^3 step: gather 1.1 -> 1.8 ms).  `slot` maps the
// upload order to the place.  (256^3 step in brick order, lists in particle order: gather
// 0.44 ms, 2.0 GB moved at 4.5 TB/s.)
// The place comes from the cell that was counted (`cell`, in upload order), never from a second
// evaluation of the position: one that differed in a bit would put a particle on another's place.
struct Order64 {
    const int *start, *rank, *cell;  // null: upload order
    int *slot;
    int N, NB, lgN;
};
__device__ __forceinline__ int64_t order64(const Order64 &O, int64_t i) {
    if (!O.start) return i;
    int x, y, z;
    brick_decode(O.cell[i], O.N, O.lgN, x, y, z);
    const int j = O.start[brick_of(x, y, z, O.NB)] + O.rank[i];
    O.slot[i] = j;
    return j;
}

// One array (or one word of the payload: `stride` words per particle) into list order through
// `tmp`, and back in place.  The container's pointers stay, so that a captured step can be
// replayed any number of times.
template <typename T>
__global__ void reorder_gather_kernel(int64_t np, const T *__restrict__ src, int stride, const int *__restrict__ list,
                                      T *__restrict__ tmp) {
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j < np) tmp[j] = src[(int64_t)list[j] * stride];
}
template <typename T>
__global__ void reorder_store_kernel(int64_t np, const T *__restrict__ tmp, T *__restrict__ dst, int stride) {
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j < np) dst[j * stride] = tmp[j];
}
// the places after a reorder: inverse of the list, then the uploaded particles' places
// through it (and the list becomes the identity)
__global__ void reorder_inverse_kernel(int64_t np, const int *__restrict__ list, int *__restrict__ place) {
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j < np) place[list[j]] = (int)j;
}
__global__ void reorder_slot_kernel(int64_t np, const int *__restrict__ place, int *__restrict__ slot,
                                    int *__restrict__ list) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= np) return;
    slot[i] = place[slot[i]];
    list[i] = (int)i;
}

// the cells of staged positions (pos: AoS)
__global__ void cells64_kernel(int64_t np, const double *__restrict__ pos, int N, int *__restrict__ cell) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= np) return;
    const double p[3] = {pos[3 * i], pos[3 * i + 1], pos[3 * i + 2]};
    cell[i] = cell64(p, N);
}

__global__ void iota_kernel(int *__restrict__ p, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = (int)i;
}

// synthetic particles in their own order
__global__ void ic_f64_kernel(IcArgs A, Soa64 dst, int N) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= A.np) return;
    double p[3], v[3];
    ic_pos(A, i, p);
    ic_vel(A, i, v);
    for (int d = 0; d < 3; ++d) {
        dst.pos[d][i] = p[d];
        dst.vel[d][i] = v[d];
    }
    dst.cell[i] = cell64(p, N);
    if (dst.mass) dst.mass[i] = 1.0;
    if (dst.id) dst.id[i] = i;
}

// In brick order: the positions are evaluated once, into the velocities' arrays, with their cells;
// counted and scanned, they go to their places, and then the velocities to theirs.
__global__ void ic_stage64_kernel(IcArgs A, Soa64 dst, int N, int *__restrict__ cell) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= A.np) return;
    double p[3];
    ic_pos(A, i, p);
    for (int d = 0; d < 3; ++d) dst.vel[d][i] = p[d];
    cell[i] = cell64(p, N);
}
__global__ void ic_place64_kernel(int64_t np, Soa64 dst, Order64 O) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= np) return;
    const int64_t j = order64(O, i);
    for (int d = 0; d < 3; ++d) dst.pos[d][j] = dst.vel[d][i];
    dst.cell[j] = O.cell[i];
    if (dst.mass) dst.mass[j] = 1.0;
    if (dst.id) dst.id[j] = i;
}
__global__ void ic_vel64_kernel(IcArgs A, Soa64 dst, const int *__restrict__ slot) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= A.np) return;
    double v[3];
    ic_vel(A, i, v);
    const int64_t j = slot[i];
    for (int d = 0; d < 3; ++d) dst.vel[d][j] = v[d];
}

__global__ void upload_f64_kernel(int64_t np, const double *__restrict__ pos, const double *__restrict__ vel,
                                  const double *__restrict__ mass, const int64_t *__restrict__ id,
                                  const unsigned long long *__restrict__ pl, int plw, Soa64 dst, int N, Order64 O) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= np) return;
    const double p[3] = {pos[3 * i], pos[3 * i + 1], pos[3 * i + 2]};
    const int cell = O.cell ? O.cell[i] : cell64(p, N);
    const int64_t j = order64(O, i);
    for (int d = 0; d < 3; ++d) {
        dst.pos[d][j] = p[d];
        dst.vel[d][j] = vel[3 * i + d];
    }
    dst.cell[j] = cell;
    if (dst.mass) dst.mass[j] = mass ? mass[i] : 1.0;
    if (dst.id) dst.id[j] = id ? id[i] : i;
    for (int w = 0; w < plw; ++w) dst.pl[j * plw + w] = pl[i * plw + w];
}

// ---------------------------------------------------------------- drift
// Drift in FP64 cell units and re-anchoring: X = (c + u) + fl(dt v) N, then the sequential
// periodic wrap of Particles.hpp:2028-2032 and re-binning to (cell, FP32 offset o).  Returns the
// new cell.  The kick (which counts the new buckets) and the scatter (which moves the particles
// there) both evaluate it from the stored state, so every operation is pinned: the two agree in
// every bit.  Both kernels are bound by the particles' bytes; moved by the kick, the new
// positions were written once more, 16 of 112 bytes per particle and step (a step of 256^3
// particles on 256^3: 746 -> 703 us).
__device__ __forceinline__ int drift_cell(int N, double dt, int cx, int cy, int cz, const float u[3], const float v[3],
                                          float o[3]) {
    int c3[3] = {cx, cy, cz};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        double X = add_rn((double)c3[d], (double)u[d]);
        X = add_rn(X, mul_rn(mul_rn(dt, (double)v[d]), (double)N));
        if (X < 0.0) X = add_rn(X, (double)N);
        if (X >= (double)N) X = sub_rn(X, (double)N);
        // beyond the reference's range (|dt v| >= box) wrap fully so the cell stays valid
        if (X < 0.0 || X >= (double)N) X = __builtin_fma(-(double)N, floor(X / (double)N), X);
        const double fl = floor(X);
        int cn = (int)fl;
        if (cn >= N) cn = N - 1;
        if (cn < 0) cn = 0;
        float on = (float)sub_rn(X, fl);
        if (!(on < 1.0f)) on = 0x1.fffffep-1f;
        c3[d] = cn;
        o[d] = on;
    }
    return c3[0] + N * (c3[1] + N * c3[2]);
}

// ---------------------------------------------------------------- scatter (counting sort)
// Counting-sort scatter, PER particles per thread (1024 or 256 per block): every load is in
// flight before the slots are claimed.  Slots: per wave, lanes with equal new buckets form
// groups (leader loop) whose leader adds the group size to the bucket's entry in an LDS hash
// table (one CAS to insert the key); after a barrier one global atomic per distinct bucket of
// the block reserves the range, and after a second barrier every particle stores at
// start[b] + base + rank.  A re-bucketing block sees a few buckets (the source is bucket
// ordered); a block of an unordered source (initial sort) at most one per particle, for which the
// table of twice as many slots has room.  Four per thread, or one where that fills less than
// the chip (sort_into_other).
template <bool DRIFT, int PER>
__global__ __launch_bounds__(256) void scatter_kernel(int64_t np, Soa32 src, Soa32 dst, Geo g,
                                                      int *__restrict__ cursor, int plw, double dt) {
    constexpr int HT = 512 * PER;
    constexpr int HASH = PER == 4 ? 21 : 23;  // the key's top bits
    static_assert(HT == 1 << (32 - HASH), "table size");
    __shared__ int hkey[HT];
    __shared__ int hval[HT];  // group counts, then the bucket's reserved base
    for (int i = threadIdx.x; i < HT; i += 256) {
        hkey[i] = -1;
        hval[i] = 0;
    }
    const int64_t i0 = (int64_t)blockIdx.x * (256 * PER) + threadIdx.x;
    int cell[PER];
    float o[PER][3], v[PER][3], m[PER];
    int64_t id[PER];
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const int64_t i = i0 + k * 256;
        cell[k] = i < np ? src.cell[i] : -1;
        m[k] = 0.f;
        id[k] = 0;
        if (cell[k] >= 0) {
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                o[k][d] = src.off[d][i];
                v[k][d] = src.vel[d][i];
            }
            if (src.mass) m[k] = src.mass[i];
            if (src.id) id[k] = src.id[i];
        }
    }
    if constexpr (DRIFT) {
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            if (cell[k] < 0) continue;
            int cx, cy, cz;
            decode_cell(cell[k], g, cx, cy, cz);
            const float u[3] = {o[k][0], o[k][1], o[k][2]};
            cell[k] = drift_cell(g.N, dt, cx, cy, cz, u, v[k], o[k]);
        }
    }
    __syncthreads();
    const int lane = lane_id();
    int bk[PER], ent[PER], rank[PER];
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const bool act = cell[k] >= 0;
        bk[k] = act ? bucket_of(cell[k], g) : 0;
        ent[k] = 0;
        rank[k] = 0;
        unsigned long long todo = __ballot(act);
        while (todo) {
            const int leader = __ffsll((long long)todo) - 1;
            const int lkey = __shfl(bk[k], leader);
            const unsigned long long grp = __ballot(act && bk[k] == lkey);
            int e = 0, r0 = 0;
            if (lane == leader) {
                e = (int)(((unsigned)lkey * 2654435761u) >> HASH) & (HT - 1);
                for (;;) {
                    const int old = atomicCAS(&hkey[e], -1, lkey);
                    if (old == -1 || old == lkey) break;
                    e = (e + 1) & (HT - 1);
                }
                r0 = atomicAdd(&hval[e], __popcll(grp));
            }
            e = __shfl(e, leader);
            r0 = __shfl(r0, leader);
            if (act && bk[k] == lkey) {
                ent[k] = e;
                rank[k] = r0 + __popcll(grp & ((1ull << lane) - 1ull));
            }
            todo &= ~grp;
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < HT; i += 256) {
        const int key = hkey[i];
        if (key >= 0) hval[i] = atomicAdd(&cursor[key], hval[i]);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        if (cell[k] < 0) continue;
        const int64_t j = (int64_t)hval[ent[k]] + rank[k];
        dst.cell[j] = cell[k];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            dst.off[d][j] = o[k][d];
            dst.vel[d][j] = v[k][d];
        }
        if (src.mass) dst.mass[j] = m[k];
        if (src.id) dst.id[j] = id[k];
        const int64_t i = i0 + k * 256;
        for (int w = 0; w < plw; ++w) dst.pl[j * plw + w] = src.pl[i * plw + w];
    }
}

// ---------------------------------------------------------------- items
// A bucket of c particles owns ceil(c / ITEM_P) consecutive items (brick_starts_kernel).
static_assert(ITEM_P == BRK_ITEM, "items of the shared scan");
struct ItemRange {
    int b;        // bucket
    int p0, p1;   // particle range
    int ox, oy, oz;  // brick origin (cells)
};
__device__ __forceinline__ bool item_range(int item, const int *__restrict__ start, const int *__restrict__ istart,
                                           const int *__restrict__ item_bucket, const Geo &g, ItemRange &r) {
    if (item >= istart[g.nbk]) return false;
    const int b = item_bucket[item];
    const int k = item - istart[b];
    r.b = b;
    r.p0 = start[b] + k * ITEM_P;
    r.p1 = min(r.p0 + ITEM_P, start[b + 1]);
    r.ox = (b % g.NB) * g.B;
    r.oy = ((b / g.NB) % g.NB) * g.B;
    r.oz = (int)(b / ((int64_t)g.NB * g.NB)) * g.B;
    return true;
}

// ---------------------------------------------------------------- deposit (F32)
// The reference accumulates, per cell, the contributions of the cell's particles to the
// nodes around it (localCube[8] / vi[36] / tii[24] + tij[54], particles/projections.hpp:
// 140-179, :1034-1122, :1421-1521) and then adds them to the field.  Here a brick's particles
// are summed in a window of its nodes in LDS first: tiles of bricks that store their nodes
// once (deposit_tiles_kernel, deposit_tiles_c_kernel), or one brick per workgroup and atomics
// into the field (deposit_brick32_kernel, dense_body).
// A particle has two non-zero weights per axis on the vertex grid (nodes 0, 1) and on the link
// grid (nodes -1, 0 or 0, 1 of the nodes at n + 1/2, the branch at the link midpoint of
// projections.hpp:1058-1071, whose third weight is zero), and one on a nearest-grid-point axis:
// 8 terms per component, or 4 (CIC-NGP vector) or 2 (CIC-NGP T_ij).  C: components; a window
// spans nodes [LO, B] per axis, LO = -1 when a component of the kind sits on links.
template <int KIND> struct KindC;
template <> struct KindC<0> { static constexpr int C = 1, LO = 0; };
template <> struct KindC<1> { static constexpr int C = 3, LO = -1; };
template <> struct KindC<2> { static constexpr int C = 6, LO = -1; };
// the CIC-NGP hybrids (vertex and nearest-grid-point axes only)
template <> struct KindC<3> { static constexpr int C = 3, LO = 0; };
template <> struct KindC<4> { static constexpr int C = 6, LO = 0; };

// component c of kind KIND: stagger mask (bit d: link grid along axis d), nearest-grid-point
// mask (bit d: the single node of the particle's cell along axis d, weight 1) and velocity
// factors; an axis in neither mask takes the vertex weights
template <int KIND, int COMP> struct Comp;
template <> struct Comp<0, 0> { static constexpr int MASK = 0, NGP = 0, VA = -1, VB = -1; };
template <> struct Comp<1, 0> { static constexpr int MASK = 1, NGP = 0, VA = 0, VB = -1; };
template <> struct Comp<1, 1> { static constexpr int MASK = 2, NGP = 0, VA = 1, VB = -1; };
template <> struct Comp<1, 2> { static constexpr int MASK = 4, NGP = 0, VA = 2, VB = -1; };
template <> struct Comp<2, 0> { static constexpr int MASK = 0, NGP = 0, VA = 0, VB = 0; };  // (0,0)
template <> struct Comp<2, 1> { static constexpr int MASK = 3, NGP = 0, VA = 0, VB = 1; };  // (0,1)
template <> struct Comp<2, 2> { static constexpr int MASK = 5, NGP = 0, VA = 0, VB = 2; };  // (0,2)
template <> struct Comp<2, 3> { static constexpr int MASK = 0, NGP = 0, VA = 1, VB = 1; };  // (1,1)
template <> struct Comp<2, 4> { static constexpr int MASK = 6, NGP = 0, VA = 1, VB = 2; };  // (1,2)
template <> struct Comp<2, 5> { static constexpr int MASK = 0, NGP = 0, VA = 2, VB = 2; };  // (2,2)
// vectorProjectionCICNGP_project (projections.hpp:422-549): component i is NGP along i
template <> struct Comp<3, 0> { static constexpr int MASK = 0, NGP = 1, VA = 0, VB = -1; };
template <> struct Comp<3, 1> { static constexpr int MASK = 0, NGP = 2, VA = 1, VB = -1; };
template <> struct Comp<3, 2> { static constexpr int MASK = 0, NGP = 4, VA = 2, VB = -1; };
// symtensorProjectionCICNGP_project (projections.hpp:709-847): T_ii on the vertices, T_ij
// NGP along i and j and CIC along the third axis
template <> struct Comp<4, 0> { static constexpr int MASK = 0, NGP = 0, VA = 0, VB = 0; };  // (0,0)
template <> struct Comp<4, 1> { static constexpr int MASK = 0, NGP = 3, VA = 0, VB = 1; };  // (0,1)
template <> struct Comp<4, 2> { static constexpr int MASK = 0, NGP = 5, VA = 0, VB = 2; };  // (0,2)
template <> struct Comp<4, 3> { static constexpr int MASK = 0, NGP = 0, VA = 1, VB = 1; };  // (1,1)
template <> struct Comp<4, 4> { static constexpr int MASK = 0, NGP = 6, VA = 1, VB = 2; };  // (1,2)
template <> struct Comp<4, 5> { static constexpr int MASK = 0, NGP = 0, VA = 2, VB = 2; };  // (2,2)

struct DepArgs {
    Soa32 s;
    const int *start;
    const int *istart;
    const int *item_bucket;
    Geo g;
    float mass_nv;           // global mass * N^3 (mass / res^3)
    float *field;            // native accumulation target
    unsigned long long *fx;  // fixed-point target (KIND 0 only)
    double fxs[6];           // fixed-point scale per component (scalar: 2^32 / mass_nv, so the
                             // fixed point counts dimensionless weights)
    int h;
    int tgt;
};

// each particle's term of a fixed-point deposit is quantised on its own, so the integer sums do
// not depend on order
__device__ __forceinline__ unsigned long long fx_term(float q, float w, double fxscale) {
    return (unsigned long long)llrint((double)(q * w) * fxscale);
}

static constexpr int DEP_MERGE = 8;  // items one deposit workgroup takes, at most

// The items a workgroup of a window kernel takes, `most` or fewer: a window is zeroed, filled and
// flushed once for all of them, but the crowded bricks of few particles have to be shared out, or a few
// workgroups work on while the chip waits (clustered particles, 8 items each against this: FP32 vector
// unfolded, 1 M on 64^3 74 -> 29 us, VecVec 2 M on 128^3 176 -> 126; FP64 vector 0.5 M on 128^3 70 -> 50).
static constexpr int64_t MERGE_GROUPS = 2048;
static int merge_items(int64_t np, int most) {
    int m = most;
    while (m > 1 && np < MERGE_GROUPS * m * ITEM_P) m /= 2;
    return m;
}

// ---------------------------------------------------------------- scalar deposit, periodic target
// Three kernels, when the target is periodic, the brick edge 8, the number of bricks per row a
// multiple of TILE_B and the mass global (the PM step's deposit).
// A brick's nodes are [0,8)^3 relative to its origin; its particles also reach the first
// node layer of the bricks above it along x, y and z.
//  * deposit_tiles_kernel: one workgroup per tile of TILE_B bricks along x, one wave per
//    brick.  A brick with fewer than `dense_min` particles sums their terms in the wave's LDS
//    window of 9^3 nodes (a denser brick leaves it empty).  Within the tile each brick's
//    x = 8 plane is added into the next brick's x = 0 plane on chip; the tile's own nodes are
//    then written once, TILE_X consecutive x per row (stored, or added to the field).  The layer
//    that belongs to the bricks above in y or z goes to two shell buffers and the tile's last
//    x = 8 plane to a seam buffer, one value per node.  No global atomics, no sort.
//  * the work list of brick_starts_kernel + dense_body: the bricks with dense_min or more particles,
//    in groups of up to DEP_MERGE items (a work list shared out statically among persistent
//    workgroups); each particle's 8 terms go straight into a 9^3 LDS window (no sort: a
//    wave's 64 particles of a crowded brick rarely share a cell), added to the field with one
//    global atomic per non-zero node after the tiles kernel's stores.
//  * fold_node: every node in the lowest y or z layer of a brick, or in the first x plane of a
//    tile, adds the shell and seam values meant for it, one thread per node, x fastest.  The
//    first FOLD_BLOCKS workgroups of the dense kernel's launch do it with global atomics
//    while the others deposit the dense bricks (deposit_dense_fold_kernel): one is memory
//    bound, the other LDS bound.
// Window sums are exact 64-bit fixed point: per term a power-of-two scale 2^(51 - e) of a
// bound n q < 2^e (ACC float: n = dense_min for the tiles, whose x = 0 planes then take at
// most twice that, the group's count for the dense kernel), or the term quantised on its own
// (ACC fixed point, order independent).
static constexpr int TILE_B = 8;           // bricks per tile (one wave each)
static constexpr int TILE_X = 8 * TILE_B;  // nodes per tile row

// a particle's term for node weight w: float accumulation takes q w times the window scale
// in FP64 (qsc = q * scale, one FMA against 1.5 2^52: |term| < 2^51 leaves the rounded integer in the low
// mantissa bits of the sum, two's complement once the constant's bits are taken off); the fixed point
// quantises fl(q w) to the global scale on its own
template <typename ACC>
__device__ __forceinline__ unsigned long long dep_term(float q, float w, double qsc, double fxs) {
    if constexpr (sizeof(ACC) == 8) {
        return fx_term(q, w, fxs);
    } else {
        const double t = fma((double)w, qsc, 0x1.8p52);
        return (unsigned long long)(__double_as_longlong(t) - 0x4338000000000000ll);
    }
}

// scale of a window whose bound is n particles of value q (float accumulation)
__device__ __forceinline__ double bound_scale(int n, float q) {
    const double bound = (double)n * (double)fabsf(q);
    if (!(bound > 0.0) || !(bound < 1e300)) return 1.0;
    int e;
    frexp(bound, &e);
    return ldexp(1.0, 51 - e);
}

// Shell and seam buffers (row = by + NB bz, X global, tile = X / TILE_X):
//   ysh[row][z in 0..8][X]: nodes with y = 8 of the row's bricks (they belong to row by + 1);
//   zsh[row][y in 0..7][X]: nodes with z = 8, y < 8 (row bz + 1);
//   xsh[row][tile][y + 9 z]: the x = 8 plane of the tile's last brick, addressed by the tile
//   whose first plane it is (the next one, periodically).
template <typename ACC>
__global__ __launch_bounds__(64 * TILE_B) void deposit_tiles_kernel(DepArgs A, int dense_min, int set,
                                                                    ACC *__restrict__ ysh, ACC *__restrict__ zsh,
                                                                    ACC *__restrict__ xsh) {
    constexpr int B = 8, NWE = 9, NW3 = NWE * NWE * NWE, PL = NWE * NWE, SP = 4;
    constexpr bool FX = sizeof(ACC) == 8;
    static_assert(TILE_X == 64, "one lane per x of the tile");
    __shared__ unsigned long long win[TILE_B][NW3];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int NB = A.g.NB, N = A.g.N, G = N + 2 * A.h;
    const int ntile = NB / TILE_B;
    const int tile = blockIdx.x % ntile, row = blockIdx.x / ntile;
    const int by = row % NB, bz = row / NB;
    const int64_t brick = (int64_t)row * NB + tile * TILE_B + wave;  // bricks are numbered x fastest
    unsigned long long *w = win[wave];
    for (int i = lane; i < NW3; i += 64) w[i] = 0ull;
    const float q = A.mass_nv;
    const double sc = FX ? 1.0 : bound_scale(dense_min, q), qsc = (double)q * sc, inv = 1.0 / sc;
    const int a = A.start[brick], n = A.start[brick + 1] - a;
    if (n < dense_min) {
        for (int j0 = 0; j0 < n; j0 += 64 * SP) {
            int c[SP];
            float ux[SP], uy[SP], uz[SP];
#pragma unroll
            for (int k = 0; k < SP; ++k) {
                const int j = j0 + lane + 64 * k;
                c[k] = -1;
                if (j < n) {
                    c[k] = A.s.cell[a + j];
                    ux[k] = A.s.off[0][a + j];
                    uy[k] = A.s.off[1][a + j];
                    uz[k] = A.s.off[2][a + j];
                }
            }
#pragma unroll
            for (int k = 0; k < SP; ++k) {
                if (c[k] < 0) continue;
                int x, y, z;
                decode_cell(c[k], A.g, x, y, z);
                const int base = (x & (B - 1)) + NWE * ((y & (B - 1)) + NWE * (z & (B - 1)));
                const float wx[2] = {1.0f - ux[k], ux[k]}, wy[2] = {1.0f - uy[k], uy[k]},
                            wz[2] = {1.0f - uz[k], uz[k]};
#pragma unroll
                for (int cz = 0; cz < 2; ++cz)
#pragma unroll
                    for (int cy = 0; cy < 2; ++cy)
#pragma unroll
                        for (int cx = 0; cx < 2; ++cx)
                            atomicAdd(&w[base + cx + NWE * (cy + NWE * cz)],
                                      dep_term<ACC>(q, wx[cx] * wy[cy] * wz[cz], qsc, A.fxs[0]));
            }
        }
    }
    __syncthreads();
    // the previous brick's x = 8 plane joins this brick's x = 0 plane
    if (wave > 0)
        for (int yz = lane; yz < PL; yz += 64) w[NWE * yz] += win[wave - 1][B + NWE * yz];
    __syncthreads();
    auto cvt = [&](unsigned long long v) -> ACC {
        if constexpr (FX) return v;
        else return (float)((double)(long long)v * inv);
    };
    const int X0 = tile * TILE_X;
    // own nodes: lane = x within the tile, wave = y, rows z = 0 .. 7
    {
        const int64_t i0 = site_index(N, A.h, X0 + lane, by * B + wave, bz * B);
        const unsigned long long *src = &win[lane / B][(lane % B) + NWE * wave];
#pragma unroll
        for (int z = 0; z < B; ++z) {
            const unsigned long long v = src[NWE * NWE * z];
            const int64_t idx = i0 + (int64_t)z * G * G;
            if constexpr (FX) {
                if (set) A.fx[idx] = v;
                else if (v) A.fx[idx] += v;
            } else {
                const float f = cvt(v);
                if (set) A.field[idx] = f;
                else if (v) A.field[idx] += f;
            }
        }
    }
    // y = 8 layer (rows z = 0 .. 8), then z = 8 layer (rows y = 0 .. 7): row r = wave + 8 j
    for (int r = wave; r < NWE + B; r += TILE_B) {
        const int y = r < NWE ? B : r - NWE, z = r < NWE ? r : B;
        const ACC v = cvt(win[lane / B][(lane % B) + NWE * (y + NWE * z)]);
        if (r < NWE) ysh[((int64_t)row * NWE + z) * N + X0 + lane] = v;
        else zsh[((int64_t)row * B + y) * N + X0 + lane] = v;
    }
    // the tile's last x = 8 plane, for the next tile's first plane
    const int nt = tile + 1 == ntile ? 0 : tile + 1;
    for (int yz = threadIdx.x; yz < PL; yz += 64 * TILE_B)
        xsh[((int64_t)row * ntile + nt) * PL + yz] = cvt(win[TILE_B - 1][B + NWE * yz]);
}

// one thread per node that receives shell or seam values, x fastest: the lowest y layer of
// each brick (N x NB x N nodes), then the lowest z layer without it (N x 7 NB x NB), then the
// first x plane of each tile without both (ntile x 7 NB x 7 NB, x slowest)
// (with global atomics, so that the dense deposit may run at the same time)
template <typename ACC>
__device__ __forceinline__ void fold_node(const DepArgs &A, const ACC *__restrict__ ysh, const ACC *__restrict__ zsh,
                                          const ACC *__restrict__ xsh, unsigned t) {
    constexpr int B = 8, NWE = 9, PL = NWE * NWE;
    constexpr bool FX = sizeof(ACC) == 8;
    const unsigned N = A.g.N, NB = A.g.NB, ntile = NB / TILE_B;
    const unsigned ny = N * NB * N, nz = N * (N - NB) * NB, nx = ntile * (N - NB) * (N - NB);
    if (t >= ny + nz + nx) return;
    // divisions by N and NB as shifts when N is a power of two (wave-uniform branch)
    const int lg = A.g.lgN;
    auto divN = [&](unsigned v) { return lg >= 0 ? v >> lg : v / N; };
    auto divNB = [&](unsigned v) { return lg >= 0 ? v >> (lg - 3) : v / NB; };
    unsigned X, Y, Z;
    if (t < ny) {
        const unsigned r = divN(t);
        X = t - r * N;
        Z = divNB(r);
        Y = (r - Z * NB) * B;
    } else if (t < ny + nz) {
        // r = yy + 7 NB zb: yy = 7 yb + k, k in 0..6
        const unsigned u = t - ny, r = divN(u);
        X = u - r * N;
        const unsigned zb = divNB(r) / (B - 1), yy = r - zb * (N - NB), yb = yy / (B - 1);
        Y = yb * B + 1 + (yy - yb * (B - 1));
        Z = zb * B;
    } else {
        const unsigned u = t - ny - nz, m = N - NB;
        const unsigned r = divNB(u) / (B - 1), yy = u - r * m;  // r = zz + m tile
        const unsigned tl = divNB(r) / (B - 1), zz = r - tl * m;
        const unsigned yb = yy / (B - 1), zb = zz / (B - 1);
        X = tl * TILE_X;
        Y = yb * B + 1 + (yy - yb * (B - 1));
        Z = zb * B + 1 + (zz - zb * (B - 1));
    }
    const unsigned by = Y / B, bz = Z / B, ly = Y % B, lz = Z % B;
    const unsigned bym = by == 0 ? NB - 1 : by - 1, bzm = bz == 0 ? NB - 1 : bz - 1;
    ACC v = ACC(0);
    if (ly == 0) {
        v += ysh[((int64_t)(bym + NB * bz) * NWE + lz) * N + X];
        if (lz == 0) v += ysh[((int64_t)(bym + NB * bzm) * NWE + B) * N + X];
    }
    if (lz == 0) v += zsh[((int64_t)(by + NB * bzm) * B + ly) * N + X];
    if (X % TILE_X == 0) {
        const unsigned tl = X / TILE_X;
        v += xsh[((int64_t)(by + NB * bz) * ntile + tl) * PL + ly + NWE * lz];
        if (ly == 0) v += xsh[((int64_t)(bym + NB * bz) * ntile + tl) * PL + B + NWE * lz];
        if (lz == 0) v += xsh[((int64_t)(by + NB * bzm) * ntile + tl) * PL + ly + NWE * B];
        if (ly == 0 && lz == 0) v += xsh[((int64_t)(bym + NB * bzm) * ntile + tl) * PL + B + NWE * B];
    }
    if (v == ACC(0)) return;
    const int64_t idx = site_index((int)N, A.h, (int)X, (int)Y, (int)Z);
    if constexpr (FX) atomicAdd(&A.fx[idx], v);
    else atomicAdd(&A.field[idx], v);
}

// number of nodes fold_node serves
__host__ __device__ inline unsigned fold_nodes(unsigned N, unsigned NB) {
    return N * NB * N + N * (N - NB) * NB + (NB / TILE_B) * (N - NB) * (N - NB);
}


static constexpr int DENSE_PER = 4;  // particles per thread and round

// persistent: workgroup w takes entries w, w + grid, ... of the work list (full groups are
// alike, so a static share balances); each round's loads are issued before the previous
// round's terms are added
template <typename ACC>
__device__ __forceinline__ void dense_body(const DepArgs &A, const int2 *__restrict__ groups,
                                           const int *__restrict__ ngroups, int bid, int nbid) {
    constexpr int B = 8, NWE = B + 1, NW3 = NWE * NWE * NWE;
    constexpr bool FX = sizeof(ACC) == 8;
    constexpr int GP = DEP_MERGE * ITEM_P;
    constexpr int RP = DENSE_PER * DEP_WG;  // particles per round
    __shared__ unsigned long long nodes[NW3];
    const int N = A.g.N, NB = A.g.NB;
    const float q = A.mass_nv;
    const int total = ngroups[0];
    for (int gi = bid; gi < total; gi += nbid) {
        for (int i = threadIdx.x; i < NW3; i += DEP_WG) nodes[i] = 0ull;
        const int2 gr = groups[gi];
        const int b = gr.x;
        const int bstart = A.start[b], bend = A.start[b + 1];
        const int p0g = bstart + gr.y * GP, end = min(bend, p0g + GP);
        const int ox = (b % NB) * B, oy = ((b / NB) % NB) * B, oz = (int)(b / ((int64_t)NB * NB)) * B;
        const double sc = FX ? 1.0 : bound_scale(end - p0g, q), qsc = (double)q * sc;
        int c[DENSE_PER];
        float ux[DENSE_PER], uy[DENSE_PER], uz[DENSE_PER];
        auto fetch = [&](int p0) {
#pragma unroll
            for (int k = 0; k < DENSE_PER; ++k) {
                const int p = p0 + threadIdx.x + k * DEP_WG;
                c[k] = -1;
                if (p < end) {
                    c[k] = A.s.cell[p];
                    ux[k] = A.s.off[0][p];
                    uy[k] = A.s.off[1][p];
                    uz[k] = A.s.off[2][p];
                }
            }
        };
        fetch(p0g);
        __syncthreads();  // the window is cleared
        for (int p0 = p0g; p0 < end; p0 += RP) {
            int cc[DENSE_PER];
            float vx[DENSE_PER], vy[DENSE_PER], vz[DENSE_PER];
#pragma unroll
            for (int k = 0; k < DENSE_PER; ++k) {
                cc[k] = c[k];
                vx[k] = ux[k];
                vy[k] = uy[k];
                vz[k] = uz[k];
            }
            if (p0 + RP < end) fetch(p0 + RP);
#pragma unroll
            for (int k = 0; k < DENSE_PER; ++k) {
                if (cc[k] < 0) continue;
                int x, y, z;
                decode_cell(cc[k], A.g, x, y, z);
                const int base = (x & (B - 1)) + NWE * ((y & (B - 1)) + NWE * (z & (B - 1)));
                const float wx[2] = {1.0f - vx[k], vx[k]}, wy[2] = {1.0f - vy[k], vy[k]},
                            wz[2] = {1.0f - vz[k], vz[k]};
#pragma unroll
                for (int cz = 0; cz < 2; ++cz)
#pragma unroll
                    for (int cy = 0; cy < 2; ++cy)
#pragma unroll
                        for (int cx = 0; cx < 2; ++cx)
                            atomicAdd(&nodes[base + cx + NWE * (cy + NWE * cz)],
                                      dep_term<ACC>(q, wx[cx] * wy[cy] * wz[cz], qsc, A.fxs[0]));
            }
        }
        __syncthreads();
        const double inv = 1.0 / sc;
        for (int i = threadIdx.x; i < NW3; i += DEP_WG) {
            const unsigned long long w = nodes[i];
            if (w == 0ull) continue;
            const int ax = i % NWE, ay = (i / NWE) % NWE, az = i / (NWE * NWE);
            const int64_t idx = site_index(N, A.h, wrapi(ox + ax, N), wrapi(oy + ay, N), wrapi(oz + az, N));
            if constexpr (FX) atomicAdd(&A.fx[idx], w);
            else atomicAdd(&A.field[idx], (float)((double)(long long)w * inv));
        }
        __syncthreads();  // the window is reused
    }
}

// ghost sites of a cubic field of ghost width h <= TILE_GHOSTS, numbered: z slabs, y slabs (z
// inside), x slabs (in 32 bits for N <= 1024)
static constexpr int TILE_GHOSTS = 16;
__device__ __forceinline__ unsigned ghost_count(int N, int h) {
    const unsigned G = N + 2 * h;
    return 2u * h * (G * G + N * G + (unsigned)N * N);
}
__device__ __forceinline__ int64_t ghost_index(int N, int h, unsigned t) {
    const unsigned G = N + 2 * h, cz = 2u * h * G * G, cy = 2u * h * N * G;
    auto out = [&](unsigned k) { return (int)k < h ? (int)k - h : N + (int)k - h; };
    if (t < cz) return site_index(N, h, (int)(t % G) - h, (int)(t / G % G) - h, out(t / (G * G)));
    t -= cz;
    if (t < cy) return site_index(N, h, (int)(t % G) - h, out(t / G % (2u * h)), (int)(t / (G * 2u * h)));
    t -= cy;
    return site_index(N, h, out(t % (2u * h)), (int)(t / (2u * h) % N), (int)(t / (2u * h * N)));
}

// the first `fold_blocks` workgroups add the shells with atomics, the others run the dense
// deposit: the two overlap (one memory bound, the other LDS bound)
template <typename ACC>
__global__ __launch_bounds__(DEP_WG) void deposit_dense_fold_kernel(DepArgs A, const int2 *__restrict__ groups,
                                                                    const int *__restrict__ ngroups,
                                                                    const ACC *__restrict__ ysh,
                                                                    const ACC *__restrict__ zsh,
                                                                    const ACC *__restrict__ xsh, int fold_blocks,
                                                                    int ghosts) {
    static_assert(DEP_WG == 256, "workgroup size of both parts");
    // without dense bricks (an even spread of particles) every workgroup folds
    const bool all_fold = ngroups[0] == 0;
    if ((int)blockIdx.x < fold_blocks || all_fold) {
        const unsigned n = fold_nodes(A.g.N, A.g.NB);
        const unsigned stride = (unsigned)(all_fold ? (int)gridDim.x : fold_blocks) * DEP_WG;
        for (unsigned t = blockIdx.x * DEP_WG + threadIdx.x; t < n; t += stride)
            fold_node<ACC>(A, ysh, zsh, xsh, t);
        if constexpr (sizeof(ACC) == 4) {
            // a target whose interior the tiles stored gets its ghosts cleared here
            const unsigned ng = ghosts ? ghost_count(A.g.N, A.h) : 0u;
            for (unsigned t = blockIdx.x * DEP_WG + threadIdx.x; t < ng; t += stride)
                A.field[ghost_index(A.g.N, A.h, t)] = 0.0f;
        }
        return;
    }
    dense_body<ACC>(A, groups, ngroups, (int)blockIdx.x - fold_blocks, (int)gridDim.x - fold_blocks);
}

// ---------------------------------------------------------------- multi-component tiles
// The vector, VecVec and CIC-NGP kinds, and the scalar kind with per-particle masses, into
// a periodic target: the scheme of deposit_tiles_kernel with the components in passes.
// One wave per brick, TC_TB bricks along x per workgroup.  The brick's first 64 TC_P
// particles stay in registers across the passes (the rest are read again in each pass),
// and each pass
//   1. sums one component into the wave's LDS window (64-bit fixed point with integer LDS
//      atomics, the scale from the tile's maxima of |q| and |v|, as in deposit_tiles_kernel);
//   2. adds the x halo planes of the windows into the neighbouring waves' windows;
//   3. keeps the bricks' own nodes of that component in registers (each thread owns a
//      column of 8 nodes along z), which are stored (set) or added (without atomics) with
//      all components of a site together after the last pass, so that every line of the
//      interleaved field is written once;
//   4. writes the window nodes outside the bricks in y or z (shell rows of the tile's
//      consecutive x) and the tile's outer x halo planes (seams) to a buffer, which
//      fold_rows_kernel and fold_edges_kernel then add to the nodes they land on.
// A component's window spans nodes [LO, HI] per axis relative to the brick.  On a link axis
// the particle's two nonzero link weights sit on nodes x - 1, x or on x, x + 1
// (projections.hpp:1058-1071, whose third weight is zero), so LO = -1 and HI = 8; a vertex
// axis spans [0, 8], a nearest-grid-point axis [0, 7].
// Bricks with dense_min or more particles are left out (their windows stay zero) and are
// deposited afterwards by deposit_brick32_kernel over a work list of their groups.
// (measured at 1024^3 with about 512 particles per brick: 4 bricks per tile and 2 particles
// per lane in registers, at most 128 VGPRs, against 8 bricks per tile or 8 particles per
// lane: within 5 %, the bricks' own nodes written once per line being what counted)
static constexpr int TC_P = 2;       // particles per lane kept in registers across the passes
static constexpr int TC_WMAX = 900;  // largest window: two link axes, 10 x 10 x 9 nodes
static constexpr int TC_TB = 4;      // bricks per tile (one wave each)

// halo layers below and above the brick along axis d, and the window edge
__host__ __device__ constexpr int tc_nl(int mask, int d) { return (mask >> d) & 1; }
__host__ __device__ constexpr int tc_nh(int ngp, int d) { return ((ngp >> d) & 1) ? 0 : 1; }
__host__ __device__ constexpr int tc_w(int mask, int ngp, int d) { return 8 + tc_nl(mask, d) + tc_nh(ngp, d); }
// shell rows of a component per brick row: the y halo layers over the window's z range,
// then the z halo layers over y = 0 .. 7
__host__ __device__ constexpr int tc_rows(int mask, int ngp) {
    return (tc_nl(mask, 1) + tc_nh(ngp, 1)) * tc_w(mask, ngp, 2) + (tc_nl(mask, 2) + tc_nh(ngp, 2)) * 8;
}
// seam values per tile: its x halo planes (y and z over the window)
__host__ __device__ constexpr int tc_seam(int mask, int ngp) {
    return (tc_nl(mask, 0) + tc_nh(ngp, 0)) * tc_w(mask, ngp, 1) * tc_w(mask, ngp, 2);
}
// Comp<KIND, c>::MASK and ::NGP as tables for the host
static constexpr int TC_MASK[5][6] = {{0}, {1, 2, 4}, {0, 3, 5, 0, 6, 0}, {0, 0, 0}, {0, 0, 0, 0, 0, 0}};
static constexpr int TC_NGP[5][6] = {{0}, {0, 0, 0}, {0, 0, 0, 0, 0, 0}, {1, 2, 4}, {0, 3, 5, 0, 6, 0}};
template <int KIND, int COMP> constexpr bool tc_table_matches() {
    return TC_MASK[KIND][COMP] == Comp<KIND, COMP>::MASK && TC_NGP[KIND][COMP] == Comp<KIND, COMP>::NGP;
}
static_assert(tc_table_matches<0, 0>() && tc_table_matches<1, 0>() && tc_table_matches<1, 1>() &&
                  tc_table_matches<1, 2>() && tc_table_matches<2, 0>() && tc_table_matches<2, 1>() &&
                  tc_table_matches<2, 2>() && tc_table_matches<2, 3>() && tc_table_matches<2, 4>() &&
                  tc_table_matches<2, 5>() && tc_table_matches<3, 0>() && tc_table_matches<3, 1>() &&
                  tc_table_matches<3, 2>() && tc_table_matches<4, 0>() && tc_table_matches<4, 1>() &&
                  tc_table_matches<4, 2>() && tc_table_matches<4, 3>() && tc_table_matches<4, 4>() &&
                  tc_table_matches<4, 5>(),
              "host tables of the component masks");

struct TcArgs {
    int64_t shell_off[6];  // first value of component c's shell rows in the buffer
    int64_t seam_off[6];   // first value of its seams
};

// the particles a lane keeps: cell in the brick (x + 8 (y + 8 z), -1 for none), offsets,
// velocity (vector kinds) and q = m N^3
struct TcRegs {
    static constexpr int P = TC_P > 0 ? TC_P : 1;
    int lc[P];
    float u[3][P], v[3][P], q[P];
};

template <int KIND, bool PM>
__device__ __forceinline__ void tc_load(const DepArgs &A, int p, int &lc, float &u0, float &u1, float &u2, float &v0,
                                        float &v1, float &v2, float &q) {
    int x, y, z;
    decode_cell(A.s.cell[p], A.g, x, y, z);
    lc = (x & 7) | ((y & 7) << 3) | ((z & 7) << 6);
    u0 = A.s.off[0][p];
    u1 = A.s.off[1][p];
    u2 = A.s.off[2][p];
    q = PM ? A.s.mass[p] * A.mass_nv : A.mass_nv;
    if constexpr (KIND > 0) {
        v0 = A.s.vel[0][p];
        v1 = A.s.vel[1][p];
        v2 = A.s.vel[2][p];
    } else {
        v0 = v1 = v2 = 0.0f;
    }
}

// weights of one axis on nodes b, b + 1 (b moves to x - 1 below a link's midpoint)
template <int MASK, int NGP, int D>
__device__ __forceinline__ void tc_weights(float u, int &b, float (&wt)[2]) {
    if constexpr ((MASK >> D) & 1) {
        const float t = u - 0.5f;
        if (t < 0.0f) {
            const float a = -t;
            b -= 1;
            wt[0] = a;
            wt[1] = 1.0f - a;
        } else {
            wt[0] = 1.0f - t;
            wt[1] = t;
        }
    } else if constexpr ((NGP >> D) & 1) {
        wt[0] = 1.0f;
        wt[1] = 0.0f;
    } else {
        wt[0] = 1.0f - u;
        wt[1] = u;
    }
}

// the window scale of a component: 2^(51 - e) with 2 n max|q| max|v_a| max|v_b| < 2^e, so
// that a node's sum, with the x halo of the neighbouring brick added, stays below 2^52 and
// each term below 2^51 (the FMA conversion of dep_term)
template <int KIND, int COMP>
__device__ __forceinline__ double tc_scale(int n, float mq, const float (&mv)[3]) {
    constexpr int VA = Comp<KIND, COMP>::VA, VB = Comp<KIND, COMP>::VB;
    double bound = 2.0 * (double)n * (double)mq;
    if constexpr (VA >= 0) bound *= (double)mv[VA];
    if constexpr (VB >= 0) bound *= (double)mv[VB];
    if (!(bound > 0.0) || !(bound < 1e300)) return 1.0;
    int e;
    frexp(bound, &e);
    return ldexp(1.0, 51 - e);
}

template <int KIND, int COMP, bool PM, int TB>
__device__ __forceinline__ void tc_pass(const DepArgs &A, const TcArgs &T, float *__restrict__ shell,
                                        unsigned long long (*win)[TC_WMAX], const TcRegs &R, int a, int n, double sc,
                                        float (&own)[KindC<KIND>::C][8], int tile, int row, int ntile) {
    constexpr int MASK = Comp<KIND, COMP>::MASK, NGP = Comp<KIND, COMP>::NGP;
    constexpr int VA = Comp<KIND, COMP>::VA, VB = Comp<KIND, COMP>::VB;
    constexpr int TX = 8 * TB;  // nodes per tile row
    constexpr int LX = -tc_nl(MASK, 0), LY = -tc_nl(MASK, 1), LZ = -tc_nl(MASK, 2);
    constexpr int WX = tc_w(MASK, NGP, 0), WY = tc_w(MASK, NGP, 1), WZ = tc_w(MASK, NGP, 2);
    constexpr int W3 = WX * WY * WZ, PL = WY * WZ;
    constexpr int SX = tc_nh(NGP, 0) ? 2 : 1, SY = tc_nh(NGP, 1) ? 2 : 1, SZ = tc_nh(NGP, 2) ? 2 : 1;
    static_assert(W3 <= TC_WMAX, "the window fits");
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int N = A.g.N;
    unsigned long long *w = win[wave];
    __syncthreads();  // the previous pass is done reading every window
    for (int i = lane; i < W3; i += 64) w[i] = 0ull;
    auto add = [&](int c, float x, float y, float z, float q, float v0, float v1, float v2) {
        float qc = q;
        if constexpr (VA >= 0) qc *= VA == 0 ? v0 : (VA == 1 ? v1 : v2);
        if constexpr (VB >= 0) qc *= VB == 0 ? v0 : (VB == 1 ? v1 : v2);
        const double qsc = (double)qc * sc;
        int bx = c & 7, byy = (c >> 3) & 7, bzz = c >> 6;
        float wx[2], wy[2], wz[2];
        tc_weights<MASK, NGP, 0>(x, bx, wx);
        tc_weights<MASK, NGP, 1>(y, byy, wy);
        tc_weights<MASK, NGP, 2>(z, bzz, wz);
        const int base = (bx - LX) + WX * ((byy - LY) + WY * (bzz - LZ));
#pragma unroll
        for (int kz = 0; kz < SZ; ++kz)
#pragma unroll
            for (int ky = 0; ky < SY; ++ky)
#pragma unroll
                for (int kx = 0; kx < SX; ++kx)
                    atomicAdd(&w[base + kx + WX * (ky + WY * kz)], dep_term<float>(qc, wx[kx] * wy[ky] * wz[kz], qsc, 0.0));
    };
#pragma unroll
    for (int k = 0; k < TC_P; ++k)
        if (R.lc[k] >= 0) add(R.lc[k], R.u[0][k], R.u[1][k], R.u[2][k], R.q[k], R.v[0][k], R.v[1][k], R.v[2][k]);
    // the particles past the registers, two per lane and round
    for (int j0 = 64 * TC_P; j0 < n; j0 += 64 * 2) {
        int c[2];
        float u0[2], u1[2], u2[2], v0[2], v1[2], v2[2], q[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int j = j0 + lane + 64 * k;
            c[k] = -1;
            if (j < n) tc_load<KIND, PM>(A, a + j, c[k], u0[k], u1[k], u2[k], v0[k], v1[k], v2[k], q[k]);
        }
#pragma unroll
        for (int k = 0; k < 2; ++k)
            if (c[k] >= 0) add(c[k], u0[k], u1[k], u2[k], q[k], v0[k], v1[k], v2[k]);
    }
    __syncthreads();
    // x halo planes between the tile's waves: the previous brick's x = 8 plane joins this
    // brick's x = 0 plane, the next brick's x = -1 plane this brick's x = 7 plane (each wave
    // writes only its own x = 0 and x = 7 planes and reads only halo planes)
    if constexpr (tc_nh(NGP, 0))
        if (wave > 0)
            for (int yz = lane; yz < PL; yz += 64) w[(0 - LX) + WX * yz] += win[wave - 1][(8 - LX) + WX * yz];
    if constexpr (tc_nl(MASK, 0))
        if (wave < TB - 1)
            for (int yz = lane; yz < PL; yz += 64) w[(7 - LX) + WX * yz] += win[wave + 1][(-1 - LX) + WX * yz];
    __syncthreads();
    const double inv = 1.0 / sc;
    auto cvt = [&](unsigned long long v) -> float { return (float)((double)(long long)v * inv); };
    const int X0 = tile * TX;
    const int tx = threadIdx.x % TX, ty = threadIdx.x / TX;  // this thread's x in the tile, and y
    // own nodes (x = tx, y = ty, z = 0 .. 7): kept until every component is done
    {
        const unsigned long long *src = &win[tx >> 3][((tx & 7) - LX) + WX * (ty - LY)];
#pragma unroll
        for (int z = 0; z < 8; ++z) own[COMP][z] = cvt(src[WX * WY * (z - LZ)]);
    }
    // shell rows: y halo layers (z over the window), then z halo layers (y = 0 .. 7)
    constexpr int RY = (tc_nl(MASK, 1) + tc_nh(NGP, 1)) * WZ, RR = tc_rows(MASK, NGP);
    float *sh = shell + T.shell_off[COMP] + (int64_t)row * RR * N + X0 + tx;
    for (int r = ty; r < RR; r += 8) {
        int y, z;
        if (r < RY) {
            const int hy = r / WZ;
            z = LZ + (r - hy * WZ);
            y = (tc_nl(MASK, 1) && hy == 0) ? -1 : 8;
        } else {
            const int s = r - RY, hz = s >> 3;
            y = s & 7;
            z = (tc_nl(MASK, 2) && hz == 0) ? -1 : 8;
        }
        sh[(int64_t)r * N] = cvt(win[tx >> 3][((tx & 7) - LX) + WX * ((y - LY) + WY * (z - LZ))]);
    }
    // seams: the x = -1 plane of the tile's first brick, the x = 8 plane of its last
    constexpr int NS = tc_nl(MASK, 0) + tc_nh(NGP, 0);
    if constexpr (NS > 0) {
        float *se = shell + T.seam_off[COMP] + ((int64_t)row * ntile + tile) * (NS * PL);
        for (int i = threadIdx.x; i < NS * PL; i += 64 * TB) {
            const int side = i / PL, yz = i - side * PL;
            const bool lower = tc_nl(MASK, 0) && side == 0;
            se[i] = cvt(lower ? win[0][(-1 - LX) + WX * yz] : win[TB - 1][(8 - LX) + WX * yz]);
        }
    }
}

// grid: one workgroup per tile (TB bricks along x) of every row of bricks
template <int KIND, bool PM, int TB>
__global__ __launch_bounds__(64 * TB, 4) void deposit_tiles_c_kernel(DepArgs A, int dense_min, int set, TcArgs T,
                                                                  float *__restrict__ shell) {
    constexpr int C = KindC<KIND>::C, TX = 8 * TB;
    __shared__ unsigned long long win[TB][TC_WMAX];
    __shared__ float smax[TB][4];
    __shared__ int sn[TB];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int NB = A.g.NB, N = A.g.N, G = N + 2 * A.h, ntile = NB / TB;
    const int tile = blockIdx.x % ntile, row = blockIdx.x / ntile;
    const int64_t brick = (int64_t)row * NB + tile * TB + wave;  // bricks are numbered x fastest
    const int a = A.start[brick];
    int n = A.start[brick + 1] - a;
    if (n >= dense_min) n = 0;  // deposit_brick32_kernel's
    TcRegs R;
    float m[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int k = 0; k < TC_P; ++k) {
        const int j = lane + 64 * k;
        R.lc[k] = -1;
        if (j < n) {
            tc_load<KIND, PM>(A, a + j, R.lc[k], R.u[0][k], R.u[1][k], R.u[2][k], R.v[0][k], R.v[1][k], R.v[2][k],
                              R.q[k]);
            m[0] = fmaxf(m[0], fabsf(R.q[k]));
            m[1] = fmaxf(m[1], fabsf(R.v[0][k]));
            m[2] = fmaxf(m[2], fabsf(R.v[1][k]));
            m[3] = fmaxf(m[3], fabsf(R.v[2][k]));
        }
    }
    for (int j = 64 * TC_P + lane; j < n; j += 64) {
        int c;
        float u0, u1, u2, v0, v1, v2, q;
        tc_load<KIND, PM>(A, a + j, c, u0, u1, u2, v0, v1, v2, q);
        m[0] = fmaxf(m[0], fabsf(q));
        m[1] = fmaxf(m[1], fabsf(v0));
        m[2] = fmaxf(m[2], fabsf(v1));
        m[3] = fmaxf(m[3], fabsf(v2));
    }
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) m[k] = fmaxf(m[k], __shfl_xor(m[k], o));
    if (lane == 0) {
        smax[wave][0] = m[0];
        smax[wave][1] = m[1];
        smax[wave][2] = m[2];
        smax[wave][3] = m[3];
        sn[wave] = n;
    }
    __syncthreads();
    float mq = 0.0f, mv[3] = {0.0f, 0.0f, 0.0f};
    int nm = 0;
#pragma unroll
    for (int b = 0; b < TB; ++b) {
        mq = fmaxf(mq, smax[b][0]);
        mv[0] = fmaxf(mv[0], smax[b][1]);
        mv[1] = fmaxf(mv[1], smax[b][2]);
        mv[2] = fmaxf(mv[2], smax[b][3]);
        nm = max(nm, sn[b]);
    }
    float own[C][8];
#define LF2MI_TC_PASS(I) \
    tc_pass<KIND, I, PM, TB>(A, T, shell, win, R, a, n, tc_scale<KIND, I>(nm, mq, mv), own, tile, row, ntile);
    LF2MI_TC_PASS(0)
    if constexpr (C > 1) {
        LF2MI_TC_PASS(1)
        LF2MI_TC_PASS(2)
    }
    if constexpr (C > 3) {
        LF2MI_TC_PASS(3)
        LF2MI_TC_PASS(4)
        LF2MI_TC_PASS(5)
    }
#undef LF2MI_TC_PASS
    // the own nodes, all components of a site together (whole lines of the interleaved field)
    const int tx = threadIdx.x % TX, ty = threadIdx.x / TX;
    const int by = row % NB, bz = row / NB;
    const int64_t i0 = site_index(N, A.h, tile * TX + tx, by * 8 + ty, bz * 8);
#pragma unroll
    for (int z = 0; z < 8; ++z) {
        float *f = A.field + (i0 + (int64_t)z * G * G) * C;
        if (set) {
#pragma unroll
            for (int c = 0; c < C; ++c) f[c] = own[c][z];
        } else {
            float o[C];
#pragma unroll
            for (int c = 0; c < C; ++c) o[c] = f[c];
#pragma unroll
            for (int c = 0; c < C; ++c) f[c] = o[c] + own[c][z];
        }
    }
}

// What the fold kernels need of each component's shells and seams.  The fold visits each
// node that receives shell or seam values once, sums every component's contributions and
// adds them to the field without atomics (nothing else writes the field meanwhile).  A node
// receives from the windows of neighbouring bricks: in y, a brick row's y = 8 layer lands on
// the next row's y = 0 layer and its y = -1 layer on the previous row's y = 7 layer (link
// axes), likewise in z; in x, a tile's outer planes land on the neighbouring tiles' edge
// nodes.  Receiving layers (union over the components): sy = y layers in the brick (0: a
// component has an upper y halo, 7: a lower one), cy the other y layers, likewise z, and sx
// the x positions in the tile (0 and TX - 1).
struct TcFold {
    int64_t shell_off[6], seam_off[6];  // as in TcArgs
    int rows[6], ns[6];                 // shell rows per brick row, seam planes per tile
    int lo[6][3], hi[6][3], w[6][3];    // window per axis
    int C, TX, ntile;
    int ny, nz, nx;                     // receiving layers
    int sy[2], sz[2], sx[2], cy[8], cz[8];
};

// the y and z shell rows of component c that land on the row (Y, Z): their offsets in the
// buffer (the value for x = X at offset + X)
__device__ __forceinline__ int tc_row_sources(const TcFold &F, int N, int NB, int c, int Y, int Z, int64_t (&off)[8]) {
    const int by = Y >> 3, ly = Y & 7, bz = Z >> 3, lz = Z & 7;
    const int LY = F.lo[c][1], HY = F.hi[c][1], LZ = F.lo[c][2], HZ = F.hi[c][2];
    const int WZ = F.w[c][2], RR = F.rows[c], RY = (F.w[c][1] - 8) * WZ;
    int n = 0;
    for (int dz = -1; dz <= 1; ++dz) {
        const int zp = lz - 8 * dz;
        if (zp < LZ || zp > HZ) continue;
        const int bzs = dz < 0 ? (bz == 0 ? NB - 1 : bz - 1) : (dz > 0 ? (bz + 1 == NB ? 0 : bz + 1) : bz);
        for (int dy = -1; dy <= 1; ++dy) {
            const int yp = ly - 8 * dy;
            if (yp < LY || yp > HY || (dy == 0 && dz == 0)) continue;
            const int bys = dy < 0 ? (by == 0 ? NB - 1 : by - 1) : (dy > 0 ? (by + 1 == NB ? 0 : by + 1) : by);
            const int64_t srow = bys + (int64_t)NB * bzs;
            const int r = dy != 0 ? (yp == 8 ? -LY : 0) * WZ + (zp - LZ) : RY + (zp == 8 ? -LZ : 0) * 8 + yp;
            off[n++] = F.shell_off[c] + (srow * RR + r) * N;
        }
    }
    return n;
}

// the seam values of component c that land on node (X, Y, Z): from the previous tile's upper
// plane on the tile's first x, from the next tile's lower plane on its last x
__device__ __forceinline__ float tc_seam_sum(const TcFold &F, const float *__restrict__ shell, int NB, int c, int X,
                                             int Y, int Z) {
    const int tile = X / F.TX, lxt = X - tile * F.TX;
    int st, side;
    if (lxt == 0 && F.hi[c][0] == 8) {
        st = tile == 0 ? F.ntile - 1 : tile - 1;
        side = -F.lo[c][0];
    } else if (lxt == F.TX - 1 && F.lo[c][0] == -1) {
        st = tile + 1 == F.ntile ? 0 : tile + 1;
        side = 0;
    } else {
        return 0.0f;
    }
    const int by = Y >> 3, ly = Y & 7, bz = Z >> 3, lz = Z & 7;
    const int LY = F.lo[c][1], HY = F.hi[c][1], LZ = F.lo[c][2], HZ = F.hi[c][2], WY = F.w[c][1];
    const int PL = WY * F.w[c][2];
    float s = 0.0f;
    for (int dz = -1; dz <= 1; ++dz) {
        const int zp = lz - 8 * dz;
        if (zp < LZ || zp > HZ) continue;
        const int bzs = dz < 0 ? (bz == 0 ? NB - 1 : bz - 1) : (dz > 0 ? (bz + 1 == NB ? 0 : bz + 1) : bz);
        for (int dy = -1; dy <= 1; ++dy) {
            const int yp = ly - 8 * dy;
            if (yp < LY || yp > HY) continue;
            const int bys = dy < 0 ? (by == 0 ? NB - 1 : by - 1) : (dy > 0 ? (by + 1 == NB ? 0 : by + 1) : by);
            const int64_t srow = bys + (int64_t)NB * bzs;
            s += shell[F.seam_off[c] + ((srow * F.ntile + st) * F.ns[c] + side) * PL + (yp - LY) + WY * (zp - LZ)];
        }
    }
    return s;
}

// the receiving nodes of whole rows along x: the sy layers (every z), then the cy layers
// with the sz layers; one workgroup per row.  The row's shell sources are found once and
// summed for every x (coalesced); then the row's tile-edge nodes add their seam values, one
// thread each (after the barrier, which orders the two updates of those nodes).
template <int C>
__global__ __launch_bounds__(256) void fold_rows_kernel(float *__restrict__ field, int N, int h, int NB, TcFold F,
                                                        const float *__restrict__ shell) {
    __shared__ int64_t soff[C][8];
    __shared__ int scnt[C];
    int64_t b = blockIdx.x;
    const int64_t rowsY = (int64_t)F.ny * NB * N;
    int Y, Z;
    if (b < rowsY) {
        const int yi = (int)(b % (F.ny * NB));
        Z = (int)(b / (F.ny * NB));
        Y = (yi / F.ny) * 8 + F.sy[yi % F.ny];
    } else {
        b -= rowsY;
        const int my = (8 - F.ny) * NB;
        const int yi = (int)(b % my), zi = (int)(b / my);
        Y = (yi / (8 - F.ny)) * 8 + F.cy[yi % (8 - F.ny)];
        Z = (zi / F.nz) * 8 + F.sz[zi % F.nz];
    }
    if ((int)threadIdx.x < C) {
        int64_t off[8];
        const int c = threadIdx.x, n = tc_row_sources(F, N, NB, c, Y, Z, off);
        for (int k = 0; k < n; ++k) soff[c][k] = off[k];
        scnt[c] = n;
    }
    __syncthreads();
    float *f0 = field + site_index(N, h, 0, Y, Z) * C;
    for (int X = threadIdx.x; X < N; X += 256) {
        float v[C];
        bool any = false;
#pragma unroll
        for (int c = 0; c < C; ++c) {
            float s = 0.0f;
            for (int k = 0; k < scnt[c]; ++k) s += shell[soff[c][k] + X];
            v[c] = s;
            any |= s != 0.0f;
        }
        if (!any) continue;
        float *f = f0 + (int64_t)X * C;
#pragma unroll
        for (int c = 0; c < C; ++c) f[c] += v[c];
    }
    __syncthreads();
    for (int e = threadIdx.x; e < F.nx * F.ntile; e += 256) {
        const int X = (e / F.nx) * F.TX + F.sx[e % F.nx];
        float v[C];
        bool any = false;
#pragma unroll
        for (int c = 0; c < C; ++c) {
            v[c] = tc_seam_sum(F, shell, NB, c, X, Y, Z);
            any |= v[c] != 0.0f;
        }
        if (!any) continue;
        float *f = f0 + (int64_t)X * C;
#pragma unroll
        for (int c = 0; c < C; ++c) f[c] += v[c];
    }
}

// the remaining receiving nodes: tile edges (sx) in the cy layers and cz layers
template <int C>
__global__ __launch_bounds__(256) void fold_edges_kernel(float *__restrict__ field, int N, int h, int NB, TcFold F,
                                                         const float *__restrict__ shell, int64_t total) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= total) return;
    const int nxt = F.nx * F.ntile, my = (8 - F.ny) * NB;
    const int xi = (int)(t % nxt);
    const int64_t r = t / nxt;
    const int yi = (int)(r % my), zi = (int)(r / my);
    const int X = (xi / F.nx) * F.TX + F.sx[xi % F.nx];
    const int Y = (yi / (8 - F.ny)) * 8 + F.cy[yi % (8 - F.ny)];
    const int Z = (zi / (8 - F.nz)) * 8 + F.cz[zi % (8 - F.nz)];
    // no shell row lands on these y and z layers: the seams only
    float v[C];
    bool any = false;
#pragma unroll
    for (int c = 0; c < C; ++c) {
        v[c] = tc_seam_sum(F, shell, NB, c, X, Y, Z);
        any |= v[c] != 0.0f;
    }
    if (!any) return;
    float *f = field + site_index(N, h, X, Y, Z) * C;
#pragma unroll
    for (int c = 0; c < C; ++c) f[c] += v[c];
}

// maxima over the particles of |q| (out[0]) and |v_d| (out[1 + d]) as the bits of
// non-negative floats: the bound of the vector and tensor fixed-point deposits
// (grid-stride, one atomic per workgroup and quantity: the four addresses see few atomics)
static constexpr int DMAX_BLOCKS = 1024;
__global__ __launch_bounds__(256) void dep_max_kernel(int64_t np, Soa32 s, float mass_nv,
                                                      unsigned int *__restrict__ out) {
    __shared__ float wm[4][4];
    float m[4] = {0.f, 0.f, 0.f, 0.f};
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < np; i += stride) {
        m[0] = fmaxf(m[0], fabsf(s.mass ? s.mass[i] * mass_nv : mass_nv));
        m[1] = fmaxf(m[1], fabsf(s.vel[0][i]));
        m[2] = fmaxf(m[2], fabsf(s.vel[1][i]));
        m[3] = fmaxf(m[3], fabsf(s.vel[2][i]));
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) m[k] = fmaxf(m[k], __shfl_xor(m[k], o));
    }
    const int wave = threadIdx.x >> 6;
    if (lane_id() == 0)
        for (int k = 0; k < 4; ++k) wm[wave][k] = m[k];
    __syncthreads();
    if (threadIdx.x < 4) {
        float v = 0.f;
        for (int w = 0; w < 4; ++w) v = fmaxf(v, wm[w][threadIdx.x]);
        atomicMax(&out[threadIdx.x], __float_as_uint(v));
    }
}

struct FxScales {
    double inv[6];
};

// field += fixed-point sums (SET: = them), which are cleared for the next deposit on the way
// (clear; the tiles deposit stores every sum, and leaves that out).  Clearing both before every
// deposit took two more launches and passes (a step at 128^3 162 -> 147 us; added to a field,
// 128^3 43 -> 32, 256^3 229 -> 198, its vector kind 741 -> 423, 512^3 1720 -> 1490).
// scale(i): the units of value i; FX_PER loads of a thread in flight together.
static constexpr int FX_PER = 4;
template <bool SET, class Scale>
__device__ __forceinline__ void fixed_take(unsigned long long *__restrict__ fx, float *__restrict__ f, int64_t n, int clear,
                                           Scale &&scale) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i0 < n; i0 += FX_PER * stride) {
        long long q[FX_PER];
        float old[FX_PER];
#pragma unroll
        for (int k = 0; k < FX_PER; ++k) {
            const int64_t i = i0 + k * stride;
            q[k] = i < n ? (long long)fx[i] : 0;
            old[k] = !SET && i < n ? f[i] : 0.0f;
        }
#pragma unroll
        for (int k = 0; k < FX_PER; ++k) {
            const int64_t i = i0 + k * stride;
            if (i >= n) break;
            if (clear && q[k]) fx[i] = 0ull;
            if (SET) f[i] = (float)((double)q[k] * scale(i));
            else if (q[k]) f[i] = old[k] + (float)((double)q[k] * scale(i));
        }
    }
}
// component c of site i at fx[i C + c], in units of 1 / S.inv[c]
template <bool SET>
__global__ void fixed_to_field_c_kernel(unsigned long long *__restrict__ fx, float *__restrict__ f, int64_t n, int C,
                                        int clear, FxScales S) {
    fixed_take<SET>(fx, f, n, clear, [&](int64_t i) { return S.inv[i % C]; });
}
__global__ void fill_u64_kernel(unsigned long long *__restrict__ p, int64_t n) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) p[i] = 0ull;
}

template <bool SET>
__global__ void fixed_to_field_kernel(unsigned long long *__restrict__ fx, float *__restrict__ f, int64_t n, int clear,
                                      double scale) {
    fixed_take<SET>(fx, f, n, clear, [scale](int64_t) { return scale; });
}

// ---------------------------------------------------------------- gather + kick + drift (F32)
struct GkdArgs {
    Soa32 s;
    const int *start;
    const int *istart;
    const int *item_bucket;
    Geo g;
    const float *phi;
    int h;
    float dt_kick;
    double dt_drift;
    int *next_counts;       // histogram of the new buckets
    unsigned int *vmax2;    // bits of max |v|^2 (non-negative float)
    int chunked;            // bricks below GKD_DIRECT_MAX are left to gkd_chunk_kernel
    int drift;              // 0: a kick only; positions, cells and buckets stay
};

// kick with the gathered acceleration, store the velocity; returns the cell after the drift
__device__ __forceinline__ int kick_store(const GkdArgs &A, int p, int cx, int cy, int cz, const float u[3],
                                          const float vin[3], const float a[3], float &vmax) {
    float v[3], o[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        v[d] = vin[d] + A.dt_kick * a[d];
        if (A.phi) A.s.vel[d][p] = v[d];  // a drift alone leaves it (1.5M particles: 29 -> 21 us)
    }
    vmax = fmaxf(vmax, v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
    return A.drift ? drift_cell(A.g.N, A.dt_drift, cx, cy, cz, u, v, o) : 0;
}

// CIC interpolation of F = -grad phi (centred differences, N/2 per unit of phi) at a
// particle with offsets u in the cell whose stencil coordinates per axis are
// xs = {x-1, x, x+1, x+2} (likewise ys, zs): the 32 values around the cell from P(x, y, z)
template <typename PHI>
__device__ __forceinline__ void cic_force(const PHI &P, const int xs[4], const int ys[4], const int zs[4], float hn,
                                          const float u[3], float a[3]) {
    float core[2][2][2], xw[2][2][2], yw[2][2][2], zw[2][2][2];
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                core[k][j][i] = P(xs[1 + i], ys[1 + j], zs[1 + k]);
                xw[k][j][i] = P(xs[i ? 3 : 0], ys[1 + j], zs[1 + k]);  // i selects x-1 / x+2
                yw[k][j][i] = P(xs[1 + i], ys[j ? 3 : 0], zs[1 + k]);  // j selects y-1 / y+2
                zw[k][j][i] = P(xs[1 + i], ys[1 + j], zs[k ? 3 : 0]);  // k selects z-1 / z+2
            }
    a[0] = a[1] = a[2] = 0.0f;
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const float w = (i ? u[0] : 1.0f - u[0]) * (j ? u[1] : 1.0f - u[1]) * (k ? u[2] : 1.0f - u[2]);
                // neighbours of node (i,j,k) along each axis, from the core or the wings
                const float xp = i ? xw[k][j][1] : core[k][j][1], xm = i ? core[k][j][0] : xw[k][j][0];
                const float yp = j ? yw[k][1][i] : core[k][1][i], ym = j ? core[k][0][i] : yw[k][0][i];
                const float zp = k ? zw[1][j][i] : core[1][j][i], zm = k ? core[0][j][i] : zw[0][j][i];
                a[0] += w * (-(xp - xm) * hn);
                a[1] += w * (-(yp - ym) * hn);
                a[2] += w * (-(zp - zm) * hn);
            }
}

// the stencil straight from phi in HBM (periodic wrap)
__device__ __forceinline__ void gather_direct(const GkdArgs &A, int cx, int cy, int cz, const float u[3], float a[3]) {
    const int N = A.g.N, h = A.h;
    const int xs[4] = {wrapi(cx - 1, N), cx, wrapi(cx + 1, N), wrapi(cx + 2, N)};
    const int ys[4] = {wrapi(cy - 1, N), cy, wrapi(cy + 1, N), wrapi(cy + 2, N)};
    const int zs[4] = {wrapi(cz - 1, N), cz, wrapi(cz + 1, N), wrapi(cz + 2, N)};
    const float *phi = A.phi;
    cic_force([=](int x, int y, int z) { return phi[site_index(N, h, x, y, z)]; }, xs, ys, zs, 0.5f * (float)N, u, a);
}

// bricks with fewer particles go to the chunks of gkd_chunk_kernel (whose window serves
// several bricks); items below it that belong to fuller bricks (a brick's last item)
// gather phi straight from HBM instead of staging a window and force table for a few
// particles
static constexpr int GKD_DIRECT_MAX = 192;
static constexpr int GKD_MERGE = 4;
// particles per thread and round of a dense brick, their loads issued together: a brick of 8^3
// particles is one round, begun while the window loads (256^3: 249 us with one, 234 with two,
// 239 with four; 512^3 clustered 1328, 1255, 1278)
static constexpr int GKD_PER = 2;

// histogram of the new buckets of one item's particles (bucket b): particles that stay in
// the brick are counted with one LDS atomic per wave, moves to the 26 neighbouring bricks
// in a 27-entry LDS table, farther moves straight in HBM; the table is flushed once per
// item (gkd_hist_flush), so a dense brick's many items do not serialise on its counter
__device__ __forceinline__ void gkd_hist_add(const GkdArgs &A, int b, int *h27, bool act, int newcell) {
    const int nb = act ? bucket_of(newcell, A.g) : b;
    const bool stay = act && nb == b;
    const unsigned long long st = __ballot(stay);
    if (lane_id() == 0 && st) atomicAdd(&h27[13], __popcll(st));
    if (!act || stay) return;
    const int NB = A.g.NB;
    const int bx = nb % NB, by = (nb / NB) % NB, bz = nb / (NB * NB);
    const int rx = b % NB, ry = (b / NB) % NB, rz = b / (NB * NB);
    auto delta = [NB](int d) {
        if (d == NB - 1 && d > 1) return -1;
        if (d == 1 - NB && d < -1) return 1;
        return d;
    };
    const int dx = delta(bx - rx), dy = delta(by - ry), dz = delta(bz - rz);
    if (dx >= -1 && dx <= 1 && dy >= -1 && dy <= 1 && dz >= -1 && dz <= 1)
        atomicAdd(&h27[13 + dx + 3 * dy + 9 * dz], 1);
    else
        atomicAdd(&A.next_counts[nb], 1);
}

// after a barrier: one HBM atomic per non-empty neighbour entry
__device__ __forceinline__ void gkd_hist_flush(const GkdArgs &A, int b, const int *h27) {
    const int t = threadIdx.x;
    if (t >= 27 || h27[t] == 0) return;
    const int NB = A.g.NB;
    const int dx = t % 3 - 1, dy = (t / 3) % 3 - 1, dz = t / 9 - 1;
    const int bx = (b % NB + dx + NB) % NB, by = ((b / NB) % NB + dy + NB) % NB, bz = (b / (NB * NB) + dz + NB) % NB;
    atomicAdd(&A.next_counts[bx + NB * (by + NB * bz)], h27[t]);
}

template <int BC> __device__ __forceinline__ void gkd_dense(const GkdArgs &A, int it) {
    constexpr int PW = MAXB + 3;  // phi window [o-1, o+B+1]
    constexpr int FW = MAXB + 1;  // force nodes [o, o+B]
    __shared__ float phw[PW * PW * PW];
    __shared__ float frc[3][FW * FW * FW];
    __shared__ unsigned int red;
    __shared__ int h27[27];
    ItemRange r;
    if (!item_range(it, A.start, A.istart, A.item_bucket, A.g, r)) return;
    if (A.chunked && A.start[r.b + 1] - A.start[r.b] < GKD_DIRECT_MAX) return;
    if (A.phi) {
        // one workgroup per GKD_MERGE consecutive items of a brick: one phi window and force
        // table serve them all (the group's other items exit)
        const int bs = A.start[r.b], be = A.start[r.b + 1];
        if (((r.p0 - bs) / ITEM_P) % GKD_MERGE != 0) return;
        r.p1 = min(be, r.p0 + GKD_MERGE * ITEM_P);
    }
    const int N = A.g.N, B = BC ? BC : A.g.B;
    if (threadIdx.x == 0) red = 0u;
    if (threadIdx.x < 27) h27[threadIdx.x] = 0;
    __syncthreads();
    float vmax = 0.0f;
    if (!A.phi || r.p1 - r.p0 < GKD_DIRECT_MAX) {
        // sparse item (no window) or drift only (no potential: a = 0)
        for (int base = r.p0; base < r.p1; base += DEP_WG) {
            const int p = base + threadIdx.x;
            const bool act = p < r.p1;
            int newcell = 0;
            if (act) {
                int cx, cy, cz;
                decode_cell(A.s.cell[p], A.g, cx, cy, cz);
                const float u[3] = {A.s.off[0][p], A.s.off[1][p], A.s.off[2][p]};
                const float vin[3] = {A.s.vel[0][p], A.s.vel[1][p], A.s.vel[2][p]};
                float a[3] = {0.f, 0.f, 0.f};
                if (A.phi) gather_direct(A, cx, cy, cz, u, a);
                newcell = kick_store(A, p, cx, cy, cz, u, vin, a, vmax);
            }
            if (A.drift) gkd_hist_add(A, r.b, h27, act, newcell);
        }
    } else {
        const int pw = B + 3, fw = B + 1;
        // the first round's particles in flight while the window loads
        int cell[GKD_PER];
        float u[GKD_PER][3], vin[GKD_PER][3];
        auto fetch = [&](int base) {
#pragma unroll
            for (int k = 0; k < GKD_PER; ++k) {
                const int p = base + threadIdx.x + k * DEP_WG;
                cell[k] = 0;
                if (p < r.p1) {
                    cell[k] = A.s.cell[p];
                    u[k][0] = A.s.off[0][p]; u[k][1] = A.s.off[1][p]; u[k][2] = A.s.off[2][p];
                    vin[k][0] = A.s.vel[0][p]; vin[k][1] = A.s.vel[1][p]; vin[k][2] = A.s.vel[2][p];
                }
            }
        };
        fetch(r.p0);
        {
            // every window load issued before the LDS stores
            constexpr int WK = ((MAXB + 3) * (MAXB + 3) * (MAXB + 3) + DEP_WG - 1) / DEP_WG;
            const int nwin = pw * pw * pw;
            float wv[WK];
#pragma unroll
            for (int k = 0; k < WK; ++k) {
                const int i = threadIdx.x + k * DEP_WG;
                wv[k] = 0.0f;
                if (i < nwin) {
                    const int gx = wrapi(r.ox - 1 + i % pw, N);
                    const int gy = wrapi(r.oy - 1 + (i / pw) % pw, N);
                    const int gz = wrapi(r.oz - 1 + i / (pw * pw), N);
                    wv[k] = A.phi[site_index(N, A.h, gx, gy, gz)];
                }
            }
#pragma unroll
            for (int k = 0; k < WK; ++k) {
                const int i = threadIdx.x + k * DEP_WG;
                if (i < nwin) phw[i] = wv[k];
            }
        }
        __syncthreads();
        const float hn = 0.5f * (float)N;
        for (int i = threadIdx.x; i < fw * fw * fw; i += DEP_WG) {
            const int x = i % fw + 1, y = (i / fw) % fw + 1, z = i / (fw * fw) + 1;
            const int c = x + pw * (y + pw * z);
            frc[0][i] = -(phw[c + 1] - phw[c - 1]) * hn;
            frc[1][i] = -(phw[c + pw] - phw[c - pw]) * hn;
            frc[2][i] = -(phw[c + pw * pw] - phw[c - pw * pw]) * hn;
        }
        __syncthreads();
        for (int base = r.p0; base < r.p1; base += GKD_PER * DEP_WG) {
            if (base != r.p0) fetch(base);
#pragma unroll
            for (int k = 0; k < GKD_PER; ++k) {
                if (base + k * DEP_WG >= r.p1) break;  // uniform: the histogram needs whole waves
                const int p = base + threadIdx.x + k * DEP_WG;
                const bool act = p < r.p1;
                int newcell = 0;
                if (act) {
                    int cx, cy, cz;
                    decode_cell(cell[k], A.g, cx, cy, cz);
                    const int lx = cx - r.ox, ly = cy - r.oy, lz = cz - r.oz;
                    float a[3] = {0.f, 0.f, 0.f};
#pragma unroll
                    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
                        for (int j = 0; j < 2; ++j)
#pragma unroll
                            for (int i = 0; i < 2; ++i) {
                                const float w = (i ? u[k][0] : 1.0f - u[k][0]) * (j ? u[k][1] : 1.0f - u[k][1]) *
                                                (kk ? u[k][2] : 1.0f - u[k][2]);
                                const int n = (lx + i) + fw * ((ly + j) + fw * (lz + kk));
                                a[0] += w * frc[0][n];
                                a[1] += w * frc[1][n];
                                a[2] += w * frc[2][n];
                            }
                    newcell = kick_store(A, p, cx, cy, cz, u[k], vin[k], a, vmax);
                }
                if (A.drift) gkd_hist_add(A, r.b, h27, act, newcell);
            }
        }
    }
    if (A.vmax2) atomicMax(&red, __float_as_uint(vmax));
    __syncthreads();
    gkd_hist_flush(A, r.b, h27);
    if (A.vmax2 && threadIdx.x == 0) atomicMax(A.vmax2, red);
}

template <int BC> __global__ __launch_bounds__(DEP_WG) void gkd_f32_kernel(GkdArgs A) { gkd_dense<BC>(A, blockIdx.x); }

// ---- sparse bricks: chunks along x
// Runs of consecutive non-empty bricks of one brick row (same y, z) whose counts are below
// GKD_DIRECT_MAX form chunks of at most GKD_CHUNK_B bricks (their particles are contiguous in
// the bucket order).  A chunk stages one phi window of
// (8 nbx + 3) x 11 x 11 nodes in LDS, so the phi lines its particles need are fetched once
// per chunk rather than once per particle stencil (the L1 gathers of the per-particle
// path are bound by the number of lines they touch).
static constexpr int GKD_CHUNK_B = 8;
// window rows a wave keeps in flight: with 4 waves x 32 >= (MAXB + 3)^2 rows the whole window
// is requested at once (a chunk is a chain of dependent latency phases, so each batch of
// rows costs a full HBM round trip: 4 batches of 8 rows took 0.70 ms, one batch 0.63 ms)
static constexpr int GKD_STAGE = 32;
static_assert((DEP_WG / 64) * GKD_STAGE >= (MAXB + 3) * (MAXB + 3), "one batch of window rows");

// Persistent over the chunk list that the scan of the bucket counts leaves (brick_starts_kernel);
// every workgroup leaves once the list is done.  Chunks are claimed one at a time (they hold 1 to
// GKD_CHUNK_B bricks), the following one while this one's particles are processed.  Chunks cut
// at fixed borders instead, a workgroup each, cost 0.74 ms against 0.62 at 512^3 (blobs): a
// fourth more of them.
// ONE: chunks of one brick each, and a workgroup for every brick (small lattices): nothing to
// claim, and a small window, whose 11-value rows would leave most of a wave idle (64^3 with 64
// particles per brick 15.7 -> 6.5 us; both forms in one kernel cost the wide one a tenth).
template <int BC, bool ONE>
__device__ __forceinline__ void gkd_chunk(const GkdArgs &A, const int4 *__restrict__ chunks, int *__restrict__ nchunk) {
    constexpr int WXM = (ONE ? 1 : GKD_CHUNK_B) * MAXB + 3, WYM = MAXB + 3;
    constexpr int NHM = ((ONE ? 1 : GKD_CHUNK_B) + 2) * 9;
    __shared__ float win[WXM * WYM * WYM];
    __shared__ int hist[NHM];
    __shared__ unsigned int red;
    __shared__ int claim;
    const int N = A.g.N, B = BC ? BC : A.g.B, NB = A.g.NB;
    const int total = nchunk[0];
    const float hn = 0.5f * (float)N;
    float vmax = 0.0f;
    if (threadIdx.x == 0) red = 0u;
    int ci = blockIdx.x;  // claims count from the grid's size
    while (ci < total) {
        const int4 ch = chunks[ci];
        const int b0 = ch.z, nbx = ch.w;
        const int bx0 = b0 % NB, by = (b0 / NB) % NB, bz = b0 / (NB * NB);
        const int ox = bx0 * B, oy = by * B, oz = bz * B;
        const int wx = nbx * B + 3, wy = B + 3, nh = (nbx + 2) * 9;
        for (int i = threadIdx.x; i < nh; i += DEP_WG) hist[i] = 0;
        // the chunk's first ITEM_P particles (all of them but where eight nearly dense bricks
        // meet) in flight while the window loads
        constexpr int CP = ITEM_P / DEP_WG;
        int pcell[CP];
        float pu[CP][3], pv[CP][3];
        auto fetch = [&](int q0) {
#pragma unroll
            for (int k = 0; k < CP; ++k) {
                const int q = q0 + threadIdx.x + k * DEP_WG;
                pcell[k] = 0;
                if (q < ch.y) {
                    pcell[k] = A.s.cell[q];
                    pu[k][0] = A.s.off[0][q]; pu[k][1] = A.s.off[1][q]; pu[k][2] = A.s.off[2][q];
                    pv[k][0] = A.s.vel[0][q]; pv[k][1] = A.s.vel[1][q]; pv[k][2] = A.s.vel[2][q];
                }
            }
        };
        fetch(ch.x);
        if constexpr (ONE) {
            // one brick: four rows (y, z) per wave
            constexpr int RB = DEP_WG / 16, ST = (WYM * WYM + RB - 1) / RB;
            const int x = threadIdx.x & 15, gx = wrapi(ox - 1 + min(x, wx - 1), N);
            float v[ST];
#pragma unroll
            for (int k = 0; k < ST; ++k) {
                const int row = (int)(threadIdx.x >> 4) + RB * k;
                v[k] = 0.0f;
                if (row < wy * wy)
                    v[k] = A.phi[site_index(N, A.h, gx, wrapi(oy - 1 + row % wy, N), wrapi(oz - 1 + row / wy, N))];
            }
#pragma unroll
            for (int k = 0; k < ST; ++k) {
                const int row = (int)(threadIdx.x >> 4) + RB * k;
                if (x < wx && row < wy * wy) win[x + wx * row] = v[k];
            }
        } else {
            // rows (y, z) of the window, one wave per row: the row's base index is wave-uniform,
            // a lane holds x = lane and x = lane + 64; every row's loads are issued before the
            // LDS stores (a load-store loop would wait out one HBM round trip per row)
            const int nrows = wy * wy;
            const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
            const int lane = threadIdx.x & 63;
            const int64_t G = (int64_t)N + 2 * A.h;
            const bool has0 = lane < wx, has1 = lane + 64 < wx;
            const int gx0 = wrapi(ox - 1 + lane, N) + A.h;
            const int gx1 = has1 ? wrapi(ox - 1 + 64 + lane, N) + A.h : 0;
            constexpr int NWV = DEP_WG / 64;
            for (int r0 = wave; r0 < nrows; r0 += NWV * GKD_STAGE) {
                float v0[GKD_STAGE], v1[GKD_STAGE];
#pragma unroll
                for (int k = 0; k < GKD_STAGE; ++k) {
                    const int row = r0 + NWV * k;
                    v0[k] = 0.0f;
                    v1[k] = 0.0f;
                    if (row < nrows) {
                        const int y = row % wy, z = row / wy;
                        const int64_t rb = G * ((int64_t)(wrapi(oy - 1 + y, N) + A.h) + G * (int64_t)(wrapi(oz - 1 + z, N) + A.h));
                        if (has0) v0[k] = A.phi[rb + gx0];
                        if (has1) v1[k] = A.phi[rb + gx1];
                    }
                }
#pragma unroll
                for (int k = 0; k < GKD_STAGE; ++k) {
                    const int row = r0 + NWV * k;
                    if (row < nrows) {
                        if (has0) win[lane + wx * row] = v0[k];
                        if (has1) win[lane + 64 + wx * row] = v1[k];
                    }
                }
            }
        }
        __syncthreads();
        if (!ONE && threadIdx.x == 0) claim = (int)gridDim.x + atomicAdd(&nchunk[1], 1);
        for (int q0 = ch.x; q0 < ch.y; q0 += ITEM_P) {
        if (q0 != ch.x) fetch(q0);
#pragma unroll
        for (int k = 0; k < CP; ++k) {
            const int p = q0 + threadIdx.x + k * DEP_WG;
            if (p >= ch.y) break;
            const int cell = pcell[k];
            float u[3] = {pu[k][0], pu[k][1], pu[k][2]}, vin[3] = {pv[k][0], pv[k][1], pv[k][2]};
            int cx, cy, cz;
            decode_cell(cell, A.g, cx, cy, cz);
            // window coordinates: cell c sits at c - o + 1
            const int lx = cx - ox + 1, ly = cy - oy + 1, lz = cz - oz + 1;
            const int xs[4] = {lx - 1, lx, lx + 1, lx + 2};
            const int ys[4] = {ly - 1, ly, ly + 1, ly + 2};
            const int zs[4] = {lz - 1, lz, lz + 1, lz + 2};
            float a[3];
            cic_force([&](int x, int y, int z) { return win[x + wx * (y + wy * z)]; }, xs, ys, zs, hn, u, a);
            const int newcell = kick_store(A, p, cx, cy, cz, u, vin, a, vmax);
            if (!A.drift) continue;
            // new bucket relative to the chunk: x in [-1, nbx], y and z in [-1, 1] (periodic)
            int nx, ny, nz;
            decode_cell(newcell, A.g, nx, ny, nz);
            nx /= B;
            ny /= B;
            nz /= B;
            int dx = nx - bx0, dy = ny - by, dz = nz - bz;
            dx += dx < 0 ? NB : 0;
            dy += dy < 0 ? NB : 0;
            dz += dz < 0 ? NB : 0;
            if (dx > nbx) dx -= NB;
            if (dy > 1) dy -= NB;
            if (dz > 1) dz -= NB;
            if (dx >= -1 && dy >= -1 && dz >= -1 && dy <= 1 && dz <= 1)
                atomicAdd(&hist[(dx + 1) + (nbx + 2) * ((dy + 1) + 3 * (dz + 1))], 1);
            else
                atomicAdd(&A.next_counts[nx + NB * (ny + NB * nz)], 1);
        }
        }
        __syncthreads();
        for (int i = threadIdx.x; i < nh; i += DEP_WG) {
            const int c = hist[i];
            if (c == 0) continue;
            const int ex = i % (nbx + 2) - 1, ey = (i / (nbx + 2)) % 3 - 1, ez = i / (3 * (nbx + 2)) - 1;
            const int bbx = (bx0 + ex + NB) % NB, bby = (by + ey + NB) % NB, bbz = (bz + ez + NB) % NB;
            atomicAdd(&A.next_counts[bbx + NB * (bby + NB * bbz)], c);
        }
        if constexpr (ONE) break;
        ci = claim;
        __syncthreads();
    }
    if (A.vmax2) {
        atomicMax(&red, __float_as_uint(vmax));
        __syncthreads();
        if (threadIdx.x == 0) atomicMax(A.vmax2, red);
    }
}

template <int BC>
__global__ __launch_bounds__(DEP_WG) void gkd_chunk_kernel(GkdArgs A, const int4 *__restrict__ chunks,
                                                           int *__restrict__ nchunk) {
    gkd_chunk<BC, false>(A, chunks, nchunk);
}

// small lattices: one launch, a workgroup per brick for the chunks, then those of the dense items
// (one launch of two costs 4.5 us of a step: 64^3 lattice, 32^3 particles, two steps 109 -> 100)
template <int BC>
__global__ __launch_bounds__(DEP_WG) void gkd_small_kernel(GkdArgs A, const int4 *__restrict__ chunks,
                                                           int *__restrict__ nchunk) {
    const int nbk = (int)A.g.nbk;
    if ((int)blockIdx.x < nbk) gkd_chunk<BC, true>(A, chunks, nchunk);
    else gkd_dense<BC>(A, (int)blockIdx.x - nbk);
}

// ---------------------------------------------------------------- F64
struct Dep64Args {
    Soa64 s;
    int64_t np;
    int N;
    double mass_nv;
    double *field;
    int h, tgt;
};

// NX, NY, NZ: nodes per axis (1 on a nearest-grid-point axis, whose weight is wx[0] = 1)
template <int NX = 2, int NY = 2, int NZ = 2>
__device__ __forceinline__ void add8_64(double *f, int C, int comp, int N, int h, int tgt, int cx, int cy, int cz,
                                        int lox, int loy, int loz, const double wx[2], const double wy[2],
                                        const double wz[2], double q) {
#pragma unroll
    for (int k = 0; k < NZ; ++k)
#pragma unroll
        for (int j = 0; j < NY; ++j)
#pragma unroll
            for (int i = 0; i < NX; ++i) {
                int x = cx + lox + i, y = cy + loy + j, z = cz + loz + k;
                if (tgt == LF2MI_DEP_PERIODIC) {
                    x = wrapi(x, N);
                    y = wrapi(y, N);
                    z = wrapi(z, N);
                }
                atomicAdd(&f[site_index(N, h, x, y, z) * C + comp], q * wx[i] * wy[j] * wz[k]);
            }
}

template <int KIND>
__global__ void deposit_f64_kernel(Dep64Args A) {
    constexpr int C = KindC<KIND>::C;
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= A.np) return;
    const int N = A.N;
    int c[3];
    double vw[3][2], lw[3][2];
    int llo[3];
    for (int d = 0; d < 3; ++d) {
        const double t = A.s.pos[d][p] * (double)N;
        c[d] = (int)floor(t) % N;
        const double u = t - floor(t);
        vw[d][0] = 1.0 - u;
        vw[d][1] = u;
        const double s = u - 0.5;
        if (s < 0) {
            llo[d] = -1;
            lw[d][0] = -s;
            lw[d][1] = 1.0 - lw[d][0];
        } else {
            llo[d] = 0;
            lw[d][1] = s;
            lw[d][0] = 1.0 - lw[d][1];
        }
    }
    const double m = A.s.mass ? A.s.mass[p] * A.mass_nv : A.mass_nv;
    if constexpr (KIND == 0) {
        add8_64(A.field, C, 0, N, A.h, A.tgt, c[0], c[1], c[2], 0, 0, 0, vw[0], vw[1], vw[2], m);
    } else {
        const double v[3] = {A.s.vel[0][p], A.s.vel[1][p], A.s.vel[2][p]};
        if constexpr (KIND == 1) {
            add8_64(A.field, C, 0, N, A.h, A.tgt, c[0], c[1], c[2], llo[0], 0, 0, lw[0], vw[1], vw[2], m * v[0]);
            add8_64(A.field, C, 1, N, A.h, A.tgt, c[0], c[1], c[2], 0, llo[1], 0, vw[0], lw[1], vw[2], m * v[1]);
            add8_64(A.field, C, 2, N, A.h, A.tgt, c[0], c[1], c[2], 0, 0, llo[2], vw[0], vw[1], lw[2], m * v[2]);
        } else if constexpr (KIND == 3) {
            const double one[2] = {1.0, 0.0};
            add8_64<1, 2, 2>(A.field, C, 0, N, A.h, A.tgt, c[0], c[1], c[2], 0, 0, 0, one, vw[1], vw[2], m * v[0]);
            add8_64<2, 1, 2>(A.field, C, 1, N, A.h, A.tgt, c[0], c[1], c[2], 0, 0, 0, vw[0], one, vw[2], m * v[1]);
            add8_64<2, 2, 1>(A.field, C, 2, N, A.h, A.tgt, c[0], c[1], c[2], 0, 0, 0, vw[0], vw[1], one, m * v[2]);
        } else if constexpr (KIND == 4) {
            const double one[2] = {1.0, 0.0};
            add8_64(A.field, C, 0, N, A.h, A.tgt, c[0], c[1], c[2], 0, 0, 0, vw[0], vw[1], vw[2], m * v[0] * v[0]);
            add8_64(A.field, C, 3, N, A.h, A.tgt, c[0], c[1], c[2], 0, 0, 0, vw[0], vw[1], vw[2], m * v[1] * v[1]);
            add8_64(A.field, C, 5, N, A.h, A.tgt, c[0], c[1], c[2], 0, 0, 0, vw[0], vw[1], vw[2], m * v[2] * v[2]);
            add8_64<1, 1, 2>(A.field, C, 1, N, A.h, A.tgt, c[0], c[1], c[2], 0, 0, 0, one, one, vw[2], m * v[0] * v[1]);
            add8_64<1, 2, 1>(A.field, C, 2, N, A.h, A.tgt, c[0], c[1], c[2], 0, 0, 0, one, vw[1], one, m * v[0] * v[2]);
            add8_64<2, 1, 1>(A.field, C, 4, N, A.h, A.tgt, c[0], c[1], c[2], 0, 0, 0, vw[0], one, one, m * v[1] * v[2]);
        } else {
            add8_64(A.field, C, 0, N, A.h, A.tgt, c[0], c[1], c[2], 0, 0, 0, vw[0], vw[1], vw[2], m * v[0] * v[0]);
            add8_64(A.field, C, 3, N, A.h, A.tgt, c[0], c[1], c[2], 0, 0, 0, vw[0], vw[1], vw[2], m * v[1] * v[1]);
            add8_64(A.field, C, 5, N, A.h, A.tgt, c[0], c[1], c[2], 0, 0, 0, vw[0], vw[1], vw[2], m * v[2] * v[2]);
            add8_64(A.field, C, 1, N, A.h, A.tgt, c[0], c[1], c[2], llo[0], llo[1], 0, lw[0], lw[1], vw[2], m * v[0] * v[1]);
            add8_64(A.field, C, 2, N, A.h, A.tgt, c[0], c[1], c[2], llo[0], 0, llo[2], lw[0], vw[1], lw[2], m * v[0] * v[2]);
            add8_64(A.field, C, 4, N, A.h, A.tgt, c[0], c[1], c[2], 0, llo[1], llo[2], vw[0], lw[1], lw[2], m * v[1] * v[2]);
        }
    }
}

// ---- brick windows
// One workgroup per group of consecutive particles of a brick: every particle's terms go into
// an LDS window of the brick's nodes, and the window's non-zero values then go to the field with
// one atomic each, consecutive lanes on consecutive addresses.  The window sums are FP64
// (W = double), or int64 of terms quantised one by one (W = unsigned long long, the fixed-point
// deposit).  No sort: a wave's particles rarely share a node, and nearly sorted ones would more
// often (LDS atomics of random cells 1500 G/s, of neighbouring ones 1290-1380).  FP32 container
// at 256^3, 512 particles per brick, microseconds, against sorting a brick's items by cell and
// summing runs in registers first: scalar 247 -> 218, vector 710 -> 460, VecVec 1572 -> 710,
// CIC-NGP 580 -> 384 and 1188 -> 675.  What bounds it: of VecVec's 945 us before the layout below
// the LDS atomics were 560 and the flush 59; of the FP64 container's 280 for a scalar the flush
// is half.  Without gain: int64 windows of scaled sums, whose LDS atomics are twice as fast but
// need a pass for the scale and conversions (equal to 25 % slower); nodes that only one window
// covers added to without atomics (280 -> 442, 945 -> 1066: loads at each workgroup's end).
// 512 threads for six components, whose window leaves room for three workgroups per CU.
template <int KIND> constexpr int bw_wg() { return KindC<KIND>::C == 6 ? 512 : 256; }
template <int KIND> constexpr int bw_edge() { return BRK + 1 - KindC<KIND>::LO; }
template <int KIND> constexpr int bw_size() {
    return bw_edge<KIND>() * bw_edge<KIND>() * bw_edge<KIND>() * KindC<KIND>::C;
}

// window values from a node to the next: components interleaved, or, of six, one after the other
// (interleaved their nodes lie 12 banks apart, and random nodes meet in a third of the banks:
// 1129 G atomics/s against 1505; 256^3 VecVec 945 -> 831 us; three interleaved components have no
// such conflict)
template <int KIND> constexpr int bw_stride() { return KindC<KIND>::C == 6 ? 1 : KindC<KIND>::C; }

template <typename T> struct BwParticle {
    int l[3];                // cell in the brick
    T vw[3][2], lw[3][2];    // vertex and link weights
    int llo[3];              // the first link node's offset (-1 or 0)
};
template <typename T> __device__ __forceinline__ void bw_weights(BwParticle<T> &P, int d, T u) {
    P.vw[d][0] = (T)1 - u;
    P.vw[d][1] = u;
    const T s = u - (T)0.5;
    if (s < 0) {
        P.llo[d] = -1;
        P.lw[d][0] = -s;
        P.lw[d][1] = (T)1 - P.lw[d][0];
    } else {
        P.llo[d] = 0;
        P.lw[d][1] = s;
        P.lw[d][0] = (T)1 - P.lw[d][1];
    }
}

// a term into the window: q w0 w1 w2, multiplied in the order of the per-particle path (FP64)
// or the weights first (FP32); fxs: the fixed point's scale
__device__ __forceinline__ void bw_term(double *p, double q, double w0, double w1, double w2, double) {
    lds_add(p, q * w0 * w1 * w2);
}
__device__ __forceinline__ void bw_term(double *p, float q, float w0, float w1, float w2, double) {
    lds_add(p, (double)(q * (w0 * w1 * w2)));
}
__device__ __forceinline__ void bw_term(unsigned long long *p, float q, float w0, float w1, float w2, double fxs) {
    atomicAdd(p, fx_term(q, w0 * w1 * w2, fxs));
}

template <int KIND, int COMP, typename W, typename T>
__device__ __forceinline__ void bw_add(W *__restrict__ win, const BwParticle<T> &P, T q, const double *fxs) {
    constexpr int M = Comp<KIND, COMP>::MASK, G = Comp<KIND, COMP>::NGP, E = bw_edge<KIND>();
    int b[3];
    T w[3][2];
    constexpr int n[3] = {(G & 1) ? 1 : 2, (G & 2) ? 1 : 2, (G & 4) ? 1 : 2};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const bool link = (M >> d) & 1, ngp = (G >> d) & 1;
        b[d] = P.l[d] - KindC<KIND>::LO + (link ? P.llo[d] : 0);
        w[d][0] = ngp ? (T)1 : (link ? P.lw[d][0] : P.vw[d][0]);
        w[d][1] = ngp ? (T)0 : (link ? P.lw[d][1] : P.vw[d][1]);
    }
    constexpr int SN = bw_stride<KIND>();
    W *o = win + SN * (b[0] + E * (b[1] + E * b[2])) + COMP * (SN == 1 ? E * E * E : 1);
#pragma unroll
    for (int k = 0; k < n[2]; ++k)
#pragma unroll
        for (int j = 0; j < n[1]; ++j)
#pragma unroll
            for (int i = 0; i < n[0]; ++i)
                bw_term(&o[SN * (i + E * (j + E * k))], q, w[0][i], w[1][j], w[2][k], fxs[COMP]);
}

// a particle's terms of every component
template <int KIND, typename W, typename T>
__device__ __forceinline__ void bw_particle(W *__restrict__ win, const BwParticle<T> &P, T m, const T (&v)[3],
                                            const double *fxs) {
    if constexpr (KIND == 0) {
        bw_add<KIND, 0>(win, P, m, fxs);
    } else if constexpr (KindC<KIND>::C == 3) {
        bw_add<KIND, 0>(win, P, m * v[0], fxs);
        bw_add<KIND, 1>(win, P, m * v[1], fxs);
        bw_add<KIND, 2>(win, P, m * v[2], fxs);
    } else {
        bw_add<KIND, 0>(win, P, m * v[0] * v[0], fxs);
        bw_add<KIND, 1>(win, P, m * v[0] * v[1], fxs);
        bw_add<KIND, 2>(win, P, m * v[0] * v[2], fxs);
        bw_add<KIND, 3>(win, P, m * v[1] * v[1], fxs);
        bw_add<KIND, 4>(win, P, m * v[1] * v[2], fxs);
        bw_add<KIND, 5>(win, P, m * v[2] * v[2], fxs);
    }
}

// the window's non-zero values into the field
template <int KIND, typename W, typename F>
__device__ __forceinline__ void bw_flush(const W *__restrict__ win, F *__restrict__ field, int N, int h, int tgt,
                                         int ox, int oy, int oz) {
    constexpr int C = KindC<KIND>::C, LO = KindC<KIND>::LO, E = bw_edge<KIND>();
    for (int i = threadIdx.x; i < bw_size<KIND>(); i += bw_wg<KIND>()) {
        const int c = i % C, n = i / C;
        const W v = bw_stride<KIND>() == 1 ? win[n + E * E * E * c] : win[i];
        if (v == W(0)) continue;
        int gx = ox + n % E + LO, gy = oy + (n / E) % E + LO, gz = oz + n / (E * E) + LO;
        if (tgt == LF2MI_DEP_PERIODIC) {
            gx = wrapi(gx, N);
            gy = wrapi(gy, N);
            gz = wrapi(gz, N);
        }
        atomicAdd(&field[site_index(N, h, gx, gy, gz) * C + c], (F)v);
    }
}

// below this many particles per brick the index, the windows' zeroing and their flush cost an
// FP64 container more than its particles' own atomics
static constexpr int64_t B64_OCC = 24;
// and below this many particles altogether the index's launches cost more than the atomics: two
// steps, by bricks and particle by particle, 20 000 particles on 32^3 129 and 105 us, on 40^3 126
// and 100; 40 000 on 32^3 139 / 144, on 64^3 127 / 122; 80 000 on 64^3 138 / 172, on 96^3 163 / 200
static constexpr int64_t B64_NP = 40000;
template <int KIND>
__global__ __launch_bounds__(bw_wg<KIND>()) void deposit_brick64_kernel(Dep64Args A, BrickIndex V, int merge) {
    constexpr int WG = bw_wg<KIND>();
    __shared__ double win[bw_size<KIND>()];
    BrickRange r;
    if (!brick_range(V, blockIdx.x, merge, r)) return;
    for (int i = threadIdx.x; i < bw_size<KIND>(); i += WG) win[i] = 0.0;
    __syncthreads();
    const int N = A.N;
    const double none[6] = {};
    for (int j = threadIdx.x; j < r.n; j += WG) {
        const int p = V.list[r.p0 + j];
        const int o[3] = {r.ox, r.oy, r.oz};
        BwParticle<double> P;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            // rounded like the per-particle path's: a product fused into the difference would
            // give other weights
            const double t = mul_rn(A.s.pos[d][p], (double)N);
            P.l[d] = (int)floor(t) % N - o[d];  // the cell as the index took it
            bw_weights(P, d, sub_rn(t, floor(t)));
        }
        const double m = A.s.mass ? A.s.mass[p] * A.mass_nv : A.mass_nv;
        double v[3] = {0.0, 0.0, 0.0};
        if constexpr (KIND > 0)
            for (int d = 0; d < 3; ++d) v[d] = A.s.vel[d][p];
        bw_particle<KIND>(win, P, m, v, none);
    }
    __syncthreads();
    bw_flush<KIND>(win, A.field, N, A.h, A.tgt, r.ox, r.oy, r.oz);
}

// The same windows for the FP32 container, whose buckets are its bricks (any edge up to 8):
// one workgroup per `merge` items of a brick, or a share of the groups of a work list
// (brick_starts_kernel), each in parts of `merge` items.  The terms' products are FP32.
template <int KIND, typename ACC>
__global__ __launch_bounds__(bw_wg<KIND>()) void deposit_brick32_kernel(DepArgs A, const int2 *__restrict__ groups,
                                                                        const int *__restrict__ ngroups,
                                                                        int merge) {
    constexpr int WG = bw_wg<KIND>(), GP = DEP_MERGE * ITEM_P;
    constexpr bool FX = sizeof(ACC) == 8;
    using W = std::conditional_t<FX, unsigned long long, double>;
    __shared__ W win[bw_size<KIND>()];
    const int N = A.g.N, NB = A.g.NB, B = A.g.B;
    auto group = [&](int b, int p0, int len) {
        const int p1 = min(A.start[b + 1], p0 + len);
        const int o[3] = {(b % NB) * B, ((b / NB) % NB) * B, (b / (NB * NB)) * B};
        for (int i = threadIdx.x; i < bw_size<KIND>(); i += WG) win[i] = W(0);
        __syncthreads();
        for (int p = p0 + (int)threadIdx.x; p < p1; p += WG) {
            // Every load before the first use of one: up to 9 % of all kinds but the native scalar, which
            // loses that where bricks are small (172^3, 22 particles each: 145 -> 152 us).  Loads a round
            // ahead gain nothing over it, and cost the kinds of few terms up to a fifth there.
            constexpr bool FIRST = KIND != 0 || FX;
            const int cell = A.s.cell[p];
            float u[3], v[3] = {0.f, 0.f, 0.f}, m = 0.f;
            if constexpr (FIRST) {
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    u[d] = A.s.off[d][p];
                    if constexpr (KIND > 0) v[d] = A.s.vel[d][p];
                }
                m = A.s.mass ? A.s.mass[p] * A.mass_nv : A.mass_nv;
            }
            int c[3];
            decode_cell(cell, A.g, c[0], c[1], c[2]);
            BwParticle<float> P;
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                P.l[d] = c[d] - o[d];
                bw_weights(P, d, FIRST ? u[d] : A.s.off[d][p]);
            }
            if constexpr (!FIRST) m = A.s.mass ? A.s.mass[p] * A.mass_nv : A.mass_nv;
            bw_particle<KIND>(win, P, m, v, A.fxs);
        }
        __syncthreads();
        if constexpr (FX) bw_flush<KIND>(win, A.fx, N, A.h, A.tgt, o[0], o[1], o[2]);
        else bw_flush<KIND>(win, A.field, N, A.h, A.tgt, o[0], o[1], o[2]);
    };
    if (groups) {
        // the groups' first parts, then their second ones, ...: a brick's last group need not fill
        // all of them, and the empty ones come last
        const int n = ngroups[0], total = n * (DEP_MERGE / merge);
        for (int gi = blockIdx.x; gi < total; gi += gridDim.x) {
            const int2 gr = groups[gi % n];
            const int p0 = A.start[gr.x] + gr.y * GP + gi / n * merge * ITEM_P;
            if (p0 >= A.start[gr.x + 1]) continue;
            group(gr.x, p0, merge * ITEM_P);
            __syncthreads();  // the window is reused
        }
        return;
    }
    const int it = blockIdx.x;
    if (it >= A.istart[A.g.nbk]) return;
    const int b = A.item_bucket[it], k = it - A.istart[b];
    if ((k & (merge - 1)) == 0) group(b, A.start[b] + k * ITEM_P, merge * ITEM_P);
}

struct Gkd64Args {
    Soa64 s;
    int64_t np;
    int N, h;
    const double *phi;
    double dt_kick, dt_drift;
    unsigned long long *vmax2;  // bits of max |v|^2 (non-negative double)
    int drift;                  // 0: a kick only, positions and cells stay
};

// kick with the gathered acceleration, drift and wrap (LATfield2_Particles.hpp:2028-2032)
__device__ __forceinline__ void kick_drift64(const Gkd64Args &A, int64_t p, const double xin[3], const double vin[3],
                                             const double a[3], double &v2) {
    const int N = A.N;
    int cn[3];
    v2 = 0.0;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        double v = vin[d];
        if (A.phi) {
            v = add_rn(v, mul_rn(A.dt_kick, a[d]));
            A.s.vel[d][p] = v;
        }
        v2 += v * v;
        if (!A.drift) continue;
        double x = add_rn(xin[d], mul_rn(A.dt_drift, v));
        if (x < 0.0) x = add_rn(x, 1.0);
        if (x >= 1.0) x = sub_rn(x, 1.0);
        // beyond the reference's range (|dt v| >= box) wrap fully so the cell stays valid
        if (x < 0.0 || x >= 1.0) x -= floor(x);
        A.s.pos[d][p] = x;
        cn[d] = (int)floor(x * (double)N) % N;
    }
    if (A.drift) A.s.cell[p] = cn[0] + N * (cn[1] + N * cn[2]);
}

// bits of |v|^2: as unsigned integers they are ordered like the values, a NaN above all of them, so
// that a maximum over them keeps a NaN (fmax drops it)
__device__ __forceinline__ unsigned long long v2_bits(double v2) { return (unsigned long long)__double_as_longlong(v2); }

// largest |v|^2 of the workgroup (its bits) into vmax2, one atomic (256 threads)
__device__ __forceinline__ void vmax64(const Gkd64Args &A, unsigned long long m) {
    __shared__ unsigned long long wm[4];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = max(m, __shfl_xor(m, o));
    if (lane_id() == 0) wm[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        m = max(max(wm[0], wm[1]), max(wm[2], wm[3]));
        // the value only grows, so one that is seen to be as large needs no atomic: tens of thousands of
        // them on one address were longer than the gather of a sparse lattice (1 M clustered particles on
        // 256^3: 458 us with the maximum, 185 without)
        if (m > __hip_atomic_load(A.vmax2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(A.vmax2, m);
    }
}

// one workgroup per group of items of a brick: the brick's window of phi, then its force
// nodes (the differences of gkd_f64_kernel, each formed once per node instead of once per
// particle and corner), both in LDS
static constexpr int G64_MERGE = 4;  // items per workgroup, at most
static constexpr int G64_PER = 2;  // particles per thread and round, their loads issued together
__global__ __launch_bounds__(256) void gkd_brick64_kernel(Gkd64Args A, BrickIndex V, int merge) {
    constexpr int PW = BRK + 3, FW = BRK + 1, RP = 256 * G64_PER;
    __shared__ double phw[PW * PW * PW];
    __shared__ double frc[3][FW * FW * FW];
    BrickRange r;
    if (!brick_range(V, blockIdx.x, merge, r)) return;
    const int N = A.N;
    int p[G64_PER];
    double x[G64_PER][3], vin[G64_PER][3];
    auto fetch = [&](int j0) {
#pragma unroll
        for (int k = 0; k < G64_PER; ++k) {
            const int j = j0 + (int)threadIdx.x + 256 * k;
            p[k] = j < r.n ? V.list[r.p0 + j] : -1;
        }
#pragma unroll
        for (int k = 0; k < G64_PER; ++k)
            if (p[k] >= 0) {
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    x[k][d] = A.s.pos[d][p[k]];
                    vin[k][d] = A.s.vel[d][p[k]];
                }
            }
    };
    // the first round's particles in flight while the window loads
    fetch(0);
    {
        constexpr int WK = (PW * PW * PW + 255) / 256;
        double w[WK];
#pragma unroll
        for (int k = 0; k < WK; ++k) {
            const int i = threadIdx.x + 256 * k;
            if (i < PW * PW * PW)
                w[k] = A.phi[site_index(N, A.h, wrapi(r.ox - 1 + i % PW, N), wrapi(r.oy - 1 + (i / PW) % PW, N),
                                        wrapi(r.oz - 1 + i / (PW * PW), N))];
        }
#pragma unroll
        for (int k = 0; k < WK; ++k) {
            const int i = threadIdx.x + 256 * k;
            if (i < PW * PW * PW) phw[i] = w[k];
        }
    }
    __syncthreads();
    const double hn = 0.5 * N;
    for (int i = threadIdx.x; i < FW * FW * FW; i += 256) {
        const int c = i % FW + 1 + PW * ((i / FW) % FW + 1 + PW * (i / (FW * FW) + 1));
        frc[0][i] = -(phw[c + 1] - phw[c - 1]) * hn;
        frc[1][i] = -(phw[c + PW] - phw[c - PW]) * hn;
        frc[2][i] = -(phw[c + PW * PW] - phw[c - PW * PW]) * hn;
    }
    __syncthreads();
    unsigned long long vmax = 0ull;
    for (int j0 = 0; j0 < r.n; j0 += RP) {
        if (j0 != 0) fetch(j0);
#pragma unroll
        for (int q = 0; q < G64_PER; ++q) {
            if (p[q] < 0) continue;
            int c[3];
            double u[3];
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                // the cell as the index took it (same expression on the same position)
                const double t = mul_rn(x[q][d], (double)N);
                c[d] = (int)floor(t) % N;
                u[d] = sub_rn(t, (double)(int)floor(t));
            }
            const double *f = &frc[0][c[0] - r.ox + FW * (c[1] - r.oy + FW * (c[2] - r.oz))];
            double a[3] = {0.0, 0.0, 0.0};
#pragma unroll
            for (int k = 0; k < 2; ++k)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int i = 0; i < 2; ++i) {
                        const double w = (i ? u[0] : 1.0 - u[0]) * (j ? u[1] : 1.0 - u[1]) * (k ? u[2] : 1.0 - u[2]);
                        const int n = i + FW * (j + FW * k);
                        a[0] += w * f[n];
                        a[1] += w * f[n + FW * FW * FW];
                        a[2] += w * f[n + 2 * FW * FW * FW];
                    }
            double v2;
            kick_drift64(A, p[q], x[q], vin[q], a, v2);
            vmax = max(vmax, v2_bits(v2));
        }
    }
    if (A.vmax2) vmax64(A, vmax);
}

// particle by particle, phi straight from HBM; also the drift without a potential
__global__ __launch_bounds__(256) void gkd_f64_kernel(Gkd64Args A) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool act = p < A.np;
    const int N = A.N;
    double v2 = 0.0;
    if (act) {
        double a[3] = {0.0, 0.0, 0.0}, x[3], vin[3];
        for (int d = 0; d < 3; ++d) {
            x[d] = A.s.pos[d][p];
            vin[d] = A.s.vel[d][p];
        }
        if (A.phi) {
            int c[3];
            double u[3];
            for (int d = 0; d < 3; ++d) {
                const double t = x[d] * (double)N;
                c[d] = (int)floor(t) % N;
                u[d] = t - (double)(int)floor(t);
            }
            const double hn = 0.5 * N;
            for (int k = 0; k < 2; ++k)
                for (int j = 0; j < 2; ++j)
                    for (int i = 0; i < 2; ++i) {
                        const double w = (i ? u[0] : 1.0 - u[0]) * (j ? u[1] : 1.0 - u[1]) * (k ? u[2] : 1.0 - u[2]);
                        const int nx = c[0] + i, ny = c[1] + j, nz = c[2] + k;
                        auto P = [&](int xx, int yy, int zz) {
                            return A.phi[site_index(N, A.h, wrapi(xx, N), wrapi(yy, N), wrapi(zz, N))];
                        };
                        a[0] += w * (-(P(nx + 1, ny, nz) - P(nx - 1, ny, nz)) * hn);
                        a[1] += w * (-(P(nx, ny + 1, nz) - P(nx, ny - 1, nz)) * hn);
                        a[2] += w * (-(P(nx, ny, nz + 1) - P(nx, ny, nz - 1)) * hn);
                    }
        }
        kick_drift64(A, p, x, vin, a, v2);
    }
    if (A.vmax2) vmax64(A, v2_bits(v2));
}

// ---------------------------------------------------------------- download / counts
__global__ void download_f32_kernel(int64_t np, Soa32 s, int N, double *__restrict__ pos, double *__restrict__ vel,
                                    double *__restrict__ mass, double mass_global) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= np) return;
    const int cell = s.cell[i];
    const int c[3] = {cell % N, (cell / N) % N, cell / (N * N)};
    for (int d = 0; d < 3; ++d) {
        if (pos) pos[3 * i + d] = add_rn((double)c[d], (double)s.off[d][i]) / (double)N;
        if (vel) vel[3 * i + d] = (double)s.vel[d][i];
    }
    if (mass) mass[i] = s.mass ? (double)s.mass[i] : mass_global;
}

__global__ void download_f64_kernel(int64_t np, Soa64 s, const int *__restrict__ slot, double *__restrict__ pos,
                                    double *__restrict__ vel) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= np) return;
    const int64_t j = slot ? slot[i] : i;
    for (int d = 0; d < 3; ++d) {
        if (pos) pos[3 * i + d] = s.pos[d][j];
        if (vel) vel[3 * i + d] = s.vel[d][j];
    }
}

// `words` values per particle into upload order
template <typename T>
__global__ void unsort_kernel(int64_t np, const T *__restrict__ src, int words, const int *__restrict__ slot,
                              T *__restrict__ dst) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= np) return;
    const int64_t j = slot[i];
    for (int w = 0; w < words; ++w) dst[i * words + w] = src[j * words + w];
}

// particles whose cell lies in the box [lo, hi) per axis, compacted through a cursor
struct BoxArgs {
    int lo[3], hi[3];
    int N;
    int64_t np, max_out;
    int *cursor;
    double *pos, *vel, *mass;
    double mass_global;
};
__global__ void download_box_f32_kernel(BoxArgs A, Soa32 s) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    bool in = false;
    int c[3] = {0, 0, 0};
    if (i < A.np) {
        const int cell = s.cell[i];
        if (cell >= 0) {
            c[0] = cell % A.N;
            c[1] = (cell / A.N) % A.N;
            c[2] = cell / (A.N * A.N);
            in = true;
            for (int d = 0; d < 3; ++d) in = in && c[d] >= A.lo[d] && c[d] < A.hi[d];
        }
    }
    const int j = agg_inc(A.cursor, 0, in);
    if (!in || j >= A.max_out) return;
    for (int d = 0; d < 3; ++d) {
        A.pos[3 * (int64_t)j + d] = add_rn((double)c[d], (double)s.off[d][i]) / (double)A.N;
        A.vel[3 * (int64_t)j + d] = (double)s.vel[d][i];
    }
    A.mass[j] = s.mass ? (double)s.mass[i] : A.mass_global;
}
__global__ void download_box_f64_kernel(BoxArgs A, Soa64 s) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    bool in = false;
    if (i < A.np) {
        const int cell = s.cell[i];
        const int c[3] = {cell % A.N, (cell / A.N) % A.N, cell / (A.N * A.N)};
        in = true;
        for (int d = 0; d < 3; ++d) in = in && c[d] >= A.lo[d] && c[d] < A.hi[d];
    }
    const int j = agg_inc(A.cursor, 0, in);
    if (!in || j >= A.max_out) return;
    for (int d = 0; d < 3; ++d) {
        A.pos[3 * (int64_t)j + d] = s.pos[d][i];
        A.vel[3 * (int64_t)j + d] = s.vel[d][i];
    }
    A.mass[j] = s.mass ? s.mass[i] : A.mass_global;
}

__global__ void cell_count_kernel(int64_t np, const int32_t *__restrict__ cell, int32_t *__restrict__ counts) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < np && cell[i] >= 0) atomicAdd(&counts[cell[i]], 1);
}

// keys of FP64 positions (AoS x,y,z) without a container; counts of the valid keys
__global__ void bin_keys_kernel(int64_t np, const double *__restrict__ pos, int N, int32_t *__restrict__ keys,
                                int32_t *__restrict__ counts) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= np) return;
    const double p[3] = {pos[3 * i], pos[3 * i + 1], pos[3 * i + 2]};
    int cell;
    float off[3];
    bin_one(p, N, cell, off);
    if (keys) keys[i] = cell;
    if (counts && cell >= 0) atomicAdd(&counts[cell], 1);
}

__global__ void fill_int_kernel(int *__restrict__ p, int64_t n, int v) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) p[i] = v;
}

// ---------------------------------------------------------------- particle statistics
// The output[] reductions of updateVel / moveParticles (particles/LATfield2_Particles.hpp:
// 788-807, 846-885) in FP64.  Each workgroup folds a grid-stride share of the particles and
// then its lanes by a fixed tree; one workgroup per quantity folds the workgroups' partials
// in the same way.  The summation order depends only on np, so results repeat exactly.
static constexpr int RED_Q = 8;        // quantities per call
static constexpr int RED_WG = 256;
static constexpr int RED_BLOCKS = 1024;
enum { RED_NONE = -1, RED_OP_SUM = 0, RED_OP_MIN = 1, RED_OP_MAX = 2 };

struct RedArgs {
    int64_t np;
    const float *vel32[3];
    const float *mass32;   // per-particle masses (F32 container) or null
    const double *vel64[3];
    const double *mass64;  // per-particle masses (F64 container) or null
    double mass;           // the global mass, when no per-particle one is used
    const int *slot;       // F64: place of each uploaded particle (null: upload order)
    int nq;
    int q[RED_Q];
    int op[RED_Q];
};

__device__ __forceinline__ double red_fold(int op, double a, double b) {
    return op == RED_OP_SUM ? a + b : (op == RED_OP_MIN ? fmin(a, b) : fmax(a, b));
}
__device__ __forceinline__ double red_identity(int op) {
    return op == RED_OP_SUM ? 0.0 : (op == RED_OP_MIN ? __builtin_inf() : -__builtin_inf());
}

template <bool F64>
__global__ __launch_bounds__(RED_WG) void parts_reduce_kernel(RedArgs A, double *__restrict__ partial) {
    double acc[RED_Q];
#pragma unroll
    for (int k = 0; k < RED_Q; ++k) acc[k] = red_identity(A.op[k]);
    const int64_t stride = (int64_t)gridDim.x * RED_WG;
    for (int64_t i = (int64_t)blockIdx.x * RED_WG + threadIdx.x; i < A.np; i += stride) {
        double v[3], m;
        if (F64) {
            const int64_t j = A.slot ? A.slot[i] : i;
            for (int d = 0; d < 3; ++d) v[d] = A.vel64[d][j];
            m = A.mass64 ? A.mass64[j] : A.mass;
        } else {
            for (int d = 0; d < 3; ++d) v[d] = (double)A.vel32[d][i];
            m = A.mass32 ? (double)A.mass32[i] : A.mass;
        }
        const double v2 = v[0] * v[0] + v[1] * v[1] + v[2] * v[2];
#pragma unroll
        for (int k = 0; k < RED_Q; ++k) {
            if (k >= A.nq || A.op[k] == RED_NONE) continue;
            double x;
            switch (A.q[k]) {
                case LF2MI_PQ_V2: x = v2; break;
                case LF2MI_PQ_MVX: x = m * v[0]; break;
                case LF2MI_PQ_MVY: x = m * v[1]; break;
                case LF2MI_PQ_MVZ: x = m * v[2]; break;
                case LF2MI_PQ_MASS: x = m; break;
                default: x = 0.5 * m * v2; break;
            }
            acc[k] = red_fold(A.op[k], acc[k], x);
        }
    }
    __shared__ double lds[RED_WG];
    for (int k = 0; k < A.nq; ++k) {
        lds[threadIdx.x] = acc[k];
        __syncthreads();
        for (int h = RED_WG / 2; h > 0; h >>= 1) {
            if ((int)threadIdx.x < h) lds[threadIdx.x] = red_fold(A.op[k], lds[threadIdx.x], lds[threadIdx.x + h]);
            __syncthreads();
        }
        if (threadIdx.x == 0) partial[(int64_t)blockIdx.x * RED_Q + k] = lds[0];
        __syncthreads();
    }
}

// out[k] = the reference's starting value folded with every workgroup's partial: one workgroup
// per quantity, each thread a fixed share of the partials, then a fixed tree (one thread
// folding 1024 partials one after the other took 211 us, a chain of dependent loads)
__global__ __launch_bounds__(RED_WG) void parts_reduce_final_kernel(RedArgs A, const double *__restrict__ partial,
                                                                    int nblocks, double *__restrict__ out) {
    const int k = blockIdx.x;
    const int op = A.op[k];
    if (op == RED_NONE) return;
    __shared__ double lds[RED_WG];
    double r = red_identity(op);
    for (int b = threadIdx.x; b < nblocks; b += RED_WG) r = red_fold(op, r, partial[(int64_t)b * RED_Q + k]);
    lds[threadIdx.x] = r;
    __syncthreads();
    for (int h = RED_WG / 2; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) lds[threadIdx.x] = red_fold(op, lds[threadIdx.x], lds[threadIdx.x + h]);
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const double init = op == RED_OP_SUM ? 0.0 : (op == RED_OP_MIN ? 9223372036854775807.0 : -9223372036854775807.0);
        out[k] = red_fold(op, init, lds[0]);
    }
}

}  // namespace lf2mi

// ---------------------------------------------------------------- container
struct lf2mi_parts_s {
    int N, dtype, flags, device;
    lf2mi::Geo g;
    int64_t cap, np;
    double mass_global;
    double total_mass;   // sum of masses (PM mean density with box volume 1)
    lf2mi::Soa32 b32[2];
    int cur;
    lf2mi::Soa64 b64;
    int *bstart, *bcount, *istart, *bsum, *item_bucket;  // bcount: zero between moves
    int *cursor;   // next place of each bucket during the scatter
    int2 *dgroups; // the dense bricks' groups (at most cap / group + bricks)
    int *ndgroup;  // their number
    int4 *chunks;  // the sparse gather's chunks (at most one per brick)
    int *nchunk;   // [number of chunks, claims (zero between moves)]
    lf2mi::BrickBuild bb;  // brick index of an F64 container
    int bricks;            // 1: there is one (b64_create)
    int *slot;             // F64: place of each uploaded particle
    int sorted;            // 1: the places are in brick order (else upload order, slot unused)
    void *tmp;             // F64: one 8-byte value per particle (reordering), with the index
    int moves;             // F64: drifts since the particles were last put into brick order
    int cap_moves;         // the same of the drifts recorded by the capture cap_id
    unsigned long long cap_id;
    int in_box;            // 1: every F64 position is in [0, 1) (a kick then leaves them alone)
    unsigned long long *fx;
    int64_t fx_n;
    int fx_used;  // fx is not cleared (new, or an error between a deposit and its taking)
    int fx_halo;  // -1, or the halo of a tiles deposit whose interior sums fx may still hold
    void *shell;          // shell and seam buffers of the tiles deposit kernel (grown on demand)
    int64_t shell_bytes;
    unsigned int *vmax_f32;
    unsigned long long *vmax_f64;
    double *red;   // statistics: RED_BLOCKS x RED_Q partials, then RED_Q results
    std::vector<void *> allocs;
    int64_t bytes;
    int plw;       // payload words (8 bytes) per particle, 0 without a payload
    int mass_src;  // deposits use: 0 the global mass, 1 the per-particle masses
    int64_t vec_off;  // vector deposits use: -1 the velocity, else the Real[3] at this payload offset
    int vec_real;     // that vector's Real type
    int64_t aos_vel;  // offset of vel in the uploaded structs (-1: none uploaded)
    void *vsrc;       // 3 planes of cap values (container precision) for the gathered vector
};

namespace lf2mi {

static int dalloc(lf2mi_parts_s *p, void **ptr, size_t bytes) {
    *ptr = nullptr;
    if (bytes == 0) return LF2MI_OK;
    hipError_t e = hipMalloc(ptr, bytes);
    if (e != hipSuccess) return hip_fail(e, "hipMalloc(particles)", __FILE__, __LINE__);
    p->allocs.push_back(*ptr);
    p->bytes += (int64_t)bytes;
    return LF2MI_OK;
}

static unsigned grid1(int64_t n, int t = 256) { return (unsigned)std::max<int64_t>(1, (n + t - 1) / t); }

static int fill_int(int *ptr, int64_t n, int v, hipStream_t st) {
    if (n <= 0) return LF2MI_OK;
    LF2MI_PROF("fill", st);
    fill_int_kernel<<<(unsigned)std::min<int64_t>(grid1(n), 65536), 256, 0, st>>>(ptr, n, v);
    LF2MI_LAUNCHED();
    return LF2MI_OK;
}

// bricks with fewer particles are deposited by deposit_tiles_kernel, the others by
// deposit_dense_kernel
static constexpr int DENSE_MIN = 1024;
// workgroups of the dense deposit kernel, each taking a static share of the work list (512^3
// blobs, about 13 K groups: 2048 / 4096 / 8192 / 16384 / 32768 workers 1.10 / 1.08 / 1.06 /
// 1.05 / 1.05 ms for the step's deposit)
static constexpr int DENSE_WORKERS = 16384;
// workgroups of the dense deposit's launch that add the tiles kernel's shells meanwhile
static constexpr int FOLD_BLOCKS = 1024;
// a dense brick's group holds 1024 particles or more: no more workgroups than that gives
static unsigned dense_workers(const lf2mi_parts_s *p) {
    return (unsigned)std::max<int64_t>(1, std::min<int64_t>(DENSE_WORKERS, p->np / DENSE_MIN));
}

static int64_t b64_bricks(int N) {
    const int64_t nb = (N + BRK - 1) / BRK;
    return nb * nb * nb;
}
// particles from which the F64 container's brick index is kept up
static int64_t b64_min(int N) { return std::max(B64_NP, B64_OCC * b64_bricks(N)); }
static bool b64_used(const lf2mi_parts_s *p) { return p->bricks && p->np >= b64_min(p->N); }

// The index of an F64 container that can hold enough particles for it: 20 bytes a particle beside
// the 52 of its state, which it can do without (it then works particle by particle), so only where
// the memory left over has room.  In one piece: nine allocations took 0.6 ms at 900 000 particles.
static void b64_create(lf2mi_parts_s *p) {
    const int N = p->N;
    const int64_t nbk = b64_bricks(N), cap = std::max<int64_t>(p->cap, 1);
    // the windows need distinct images of a brick's nodes, the scans at most 4096 blocks
    if (N < 16 || brick_blocks(nbk) > 4096 || p->cap < b64_min(N)) return;
    const int64_t items = brick_items(nbk, cap), blocks = brick_blocks(nbk);
    const int64_t ints = 2 * (nbk + 1) + nbk + 3 * blocks + items + 3 * cap;
    const size_t bytes = (size_t)cap * sizeof(double) + (size_t)ints * sizeof(int);
    if (bytes > spare_bytes()) return;
    void *mem = nullptr;
    if (hipMalloc(&mem, bytes) != hipSuccess) {
        (void)hipGetLastError();
        return;
    }
    p->allocs.push_back(mem);
    p->bytes += (int64_t)bytes;
    p->tmp = mem;
    int *q = (int *)((double *)mem + cap);
    auto take = [&q](int64_t n) {
        int *r = q;
        q += n;
        return r;
    };
    p->bb.start = take(nbk + 1);
    p->bb.istart = take(nbk + 1);
    p->bb.count = take(nbk);
    p->bb.bsum = take(3 * blocks);
    p->bb.item = take(items);
    p->bb.list = take(cap);
    p->bb.rank = take(cap);
    p->slot = take(cap);
    p->bricks = hipMemset(p->bb.count, 0, (size_t)nbk * sizeof(int)) == hipSuccess;
}
template <typename T> static int reorder_one(lf2mi_parts_s *p, T *a, int stride, hipStream_t st) {
    const unsigned g = grid1(p->np);
    reorder_gather_kernel<T><<<g, 256, 0, st>>>(p->np, a, stride, p->bb.list, (T *)p->tmp);
    LF2MI_LAUNCHED();
    reorder_store_kernel<T><<<g, 256, 0, st>>>(p->np, (const T *)p->tmp, a, stride);
    LF2MI_LAUNCHED();
    return LF2MI_OK;
}

// The index after a drift; every B64_REORDER drifts the particles are put into its order as
// well.  A particle that has left the brick whose place it lies in costs whole lines for
// single values: at 256^3 the gather slows from 0.45 to 0.9 ms over 400 steps without this;
// a reorder takes 0.9 ms.  A drift that is recorded runs with each replay and not now, so a
// capture counts its own drifts from 0: what a graph holds depends on the graph alone.
static constexpr int B64_REORDER = 32;
static int b64_moved(lf2mi_parts_s *p, bool captured, unsigned long long cap_id, hipStream_t st) {
    Soa64 &s = p->b64;
    if (int rc = brick_build(s.cell, p->np, p->N, p->bb, st)) return rc;
    if (captured && cap_id != p->cap_id) {
        p->cap_id = cap_id;
        p->cap_moves = 0;
    }
    int &moves = captured ? p->cap_moves : p->moves;
    if (++moves < B64_REORDER) return LF2MI_OK;
    moves = 0;
    int rc = reorder_one(p, s.cell, 1, st);
    for (int d = 0; d < 3 && !rc; ++d) {
        rc = reorder_one(p, s.pos[d], 1, st);
        if (!rc) rc = reorder_one(p, s.vel[d], 1, st);
    }
    if (!rc && s.mass) rc = reorder_one(p, s.mass, 1, st);
    if (!rc && s.id) rc = reorder_one(p, s.id, 1, st);
    for (int w = 0; w < p->plw && !rc; ++w) rc = reorder_one(p, s.pl + w, p->plw, st);
    if (rc) return rc;
    const unsigned g = grid1(p->np);
    reorder_inverse_kernel<<<g, 256, 0, st>>>(p->np, p->bb.list, p->bb.rank);
    LF2MI_LAUNCHED();
    reorder_slot_kernel<<<g, 256, 0, st>>>(p->np, p->bb.rank, p->slot, p->bb.list);
    LF2MI_LAUNCHED();
    return LF2MI_OK;
}

// new contents of the F64 container (p->np particles): staged arrays (`pos` and the rest,
// device) or, without `pos`, the synthetic particles of A; their brick order and index where
// the container keeps one
static int b64_fill(lf2mi_parts_s *p, const double *pos, const double *vel, const double *mass, const int64_t *id,
                    const unsigned long long *pl, const IcArgs &A, hipStream_t st) {
    const int N = p->N;
    const unsigned g = grid1(p->np);
    Order64 O{};
    p->sorted = b64_used(p);
    p->moves = 0;
    if (p->sorted) {
        const BrickIndex V = brick_view(p->bb, N);
        // the cells are kept in the list, which is written last
        if (pos) cells64_kernel<<<g, 256, 0, st>>>(p->np, pos, N, p->bb.list);
        else ic_stage64_kernel<<<g, 256, 0, st>>>(A, p->b64, N, p->bb.list);
        LF2MI_LAUNCHED();
        brick_count(p->np, p->bb.list, N, V.NB, V.lgN, p->bb, st);
        LF2MI_LAUNCHED();
        if (int rc = brick_scan(p->bb.scan(), V.nbk, st)) return rc;
        O.start = p->bb.start;
        O.rank = p->bb.rank;
        O.cell = p->bb.list;
        O.slot = p->slot;
        O.N = N;
        O.NB = V.NB;
        O.lgN = V.lgN;
    }
    if (pos) upload_f64_kernel<<<g, 256, 0, st>>>(p->np, pos, vel, mass, id, pl, p->plw, p->b64, N, O);
    else if (p->sorted) ic_place64_kernel<<<g, 256, 0, st>>>(p->np, p->b64, O);
    else ic_f64_kernel<<<g, 256, 0, st>>>(A, p->b64, N);
    LF2MI_LAUNCHED();
    if (p->sorted) {
        if (!pos) {
            ic_vel64_kernel<<<g, 256, 0, st>>>(A, p->b64, p->slot);
            LF2MI_LAUNCHED();
        }
        iota_kernel<<<g, 256, 0, st>>>(p->bb.list, p->np);
        LF2MI_LAUNCHED();
    }
    return LF2MI_OK;
}

// bricks per chunk of the sparse gather: one below 8192 bricks, where more would leave fewer than
// four chunks per CU or need the launch of their own (two steps, chunks of one and of four: 128^3
// uniform 210 against 232 us, clustered 289 / 313, 160^3 clustered 498 / 525, dense 276 / 277;
// of one and of eight: 192^3 uniform 421 / 399, 256^3 uniform 825 / 745)
static int chunk_width(const lf2mi_parts_s *p) { return p->g.nbk < 8192 ? 1 : GKD_CHUNK_B; }

// exclusive scans of bcount -> bstart and the cursors, items -> istart, and the dense bricks'
// groups; bcount comes out cleared
static int scan_buckets(lf2mi_parts_s *p, hipStream_t st) {
    const int64_t n = p->g.nbk;
    if (brick_blocks(n) > 4096) return fail(LF2MI_ERANGE, "too many buckets (%lld)", (long long)n);
    LF2MI_PROF("rebucket_scan", st);
    BrickScan S{};
    S.count = p->bcount;
    S.bsum = p->bsum;
    S.start = p->bstart;
    S.istart = p->istart;
    S.item = p->item_bucket;
    S.cursor = p->cursor;
    S.group = p->dgroups;
    S.ngroup = p->ndgroup;
    S.dense_min = DENSE_MIN;
    S.group_p = DEP_MERGE * ITEM_P;
    S.chunk = p->chunks;
    S.nchunk = p->nchunk;
    S.NB = p->g.NB;
    S.sparse_max = GKD_DIRECT_MAX;
    S.chunk_w = chunk_width(p);
    return brick_scan(S, (int)n, st);
}

static constexpr int64_t SCAT_FULL = 256 * 1024;  // four particles per thread fill 256 CUs

// counting sort of buffer `src` (counts already in bcount) into buffer 1 - src; drift: the
// particles move by dt on the way
static int sort_into_other(lf2mi_parts_s *p, int src, int64_t nsrc, bool drift, double dt, hipStream_t st) {
    if (int rc = scan_buckets(p, st)) return rc;
    LF2MI_PROF("rebucket_scatter", st);
    auto launch = [&](auto kernel, int per) {
        kernel<<<grid1(nsrc, 256 * per), 256, 0, st>>>(nsrc, p->b32[src], p->b32[1 - src], p->g, p->cursor, p->plw, dt);
    };
    // one particle per thread while four leave CUs without a block (32^3 particles: 10.1 -> 4.9 us)
    if (nsrc < SCAT_FULL) {
        if (drift) launch(scatter_kernel<true, 1>, 1);
        else launch(scatter_kernel<false, 1>, 1);
    } else {
        if (drift) launch(scatter_kernel<true, 4>, 4);
        else launch(scatter_kernel<false, 4>, 4);
    }
    LF2MI_LAUNCHED();
    p->cur = 1 - src;
    return LF2MI_OK;
}

static int read_total(lf2mi_parts_s *p, hipStream_t st, int64_t *out) {
    int tot = 0;
    LF2MI_HIP(hipMemcpyAsync(&tot, p->bstart + p->g.nbk, sizeof(int), hipMemcpyDeviceToHost, st));
    LF2MI_HIP(hipStreamSynchronize(st));
    *out = tot;
    return LF2MI_OK;
}

static int64_t item_grid(const lf2mi_parts_s *p) { return p->g.nbk + p->np / ITEM_P + 1; }

// the brick window deposit: every brick, or (groups) those of a work list of dense ones
template <int KIND, typename ACC>
static void launch_bricks(const lf2mi_parts_s *p, const DepArgs &A, unsigned grid, const int2 *groups, const int *ngroups,
                          hipStream_t st) {
    deposit_brick32_kernel<KIND, ACC><<<grid, bw_wg<KIND>(), 0, st>>>(A, groups, ngroups, merge_items(p->np, DEP_MERGE));
}

// the scalar deposit of a global mass into a periodic target with 8^3 bricks
static bool tiles_path(const lf2mi_parts_s *p, int kind, int target, bool pm) {
    return kind == LF2MI_PROJ_SCALAR && !pm && target == LF2MI_DEP_PERIODIC && p->g.B == 8 &&
           p->g.NB % TILE_B == 0 && p->N <= 1024;
}

// the shell and seam buffers of the tiles kernel (grown on demand): N^3 (9 + 8) / 64 values
// and 81 per tile
static int shell_buffers(lf2mi_parts_s *p, size_t esz, void **ysh, void **zsh, void **xsh) {
    const int64_t N = p->N, NB = p->g.NB;
    const int64_t ny = N * N * N / 64 * 9, nz = N * N * N / 64 * 8, nx = NB * NB * (NB / TILE_B) * 81;
    const int64_t bytes = (ny + nz + nx) * (int64_t)esz;
    if (p->shell_bytes < bytes) {
        if (p->shell) hipFree(p->shell);
        p->shell = nullptr;
        p->shell_bytes = 0;
        LF2MI_HIP(hipMalloc(&p->shell, (size_t)bytes));
        p->shell_bytes = bytes;
    }
    *ysh = p->shell;
    *zsh = (char *)p->shell + ny * (int64_t)esz;
    *xsh = (char *)p->shell + (ny + nz) * (int64_t)esz;
    return LF2MI_OK;
}

template <typename ACC>
static int launch_tiles_dense(lf2mi_parts_s *p, const DepArgs &A, bool overwrite, bool ghosts, hipStream_t st) {
    void *ysh = nullptr, *zsh = nullptr, *xsh = nullptr;
    if (int rc = shell_buffers(p, sizeof(ACC), &ysh, &zsh, &xsh)) return rc;
    const int64_t NB = p->g.NB, N = p->N;
    deposit_tiles_kernel<ACC><<<(unsigned)(NB * NB * (NB / TILE_B)), 64 * TILE_B, 0, st>>>(
        A, DENSE_MIN, overwrite ? 1 : 0, (ACC *)ysh, (ACC *)zsh, (ACC *)xsh);
    LF2MI_LAUNCHED();
    // without dense bricks every workgroup folds, so few particles do not make them few: added to a field,
    // 10 000 on 512^3, 325 us with 9 beside the fold's 1024, 268 with 1024, 249 with 7168
    const unsigned nodes = grid1(fold_nodes((unsigned)N, (unsigned)NB));
    const unsigned fold = std::min<unsigned>(FOLD_BLOCKS, nodes);
    const unsigned workers = std::max(dense_workers(p), std::min<unsigned>(7 * FOLD_BLOCKS, nodes - fold));
    deposit_dense_fold_kernel<ACC><<<fold + workers, DEP_WG, 0, st>>>(
        A, p->dgroups, p->ndgroup, (const ACC *)ysh, (const ACC *)zsh, (const ACC *)xsh, (int)fold, ghosts ? 1 : 0);
    LF2MI_LAUNCHED();
    return LF2MI_OK;
}

// The other kinds (and the scalar kind with per-particle masses) into a periodic target with 8^3
// bricks, four to a tile.  The tiles' cost is the field's, which they store once, the windows' the
// particles' and their bricks' flushes: tiles on large lattices with few particles per brick, all from
// 512^3; the CIC-NGP vector, with half the terms, up to more particles.  Evenly spread particles, microseconds, windows / tiles (the tiles' sums
// are also the same from run to run where no brick is dense):
//                               vector          VecVec           vector NGP     tensor NGP
//   128^3, 128 per brick          65 / 66         104 / 101        55 / 47        90 / 74
//   160^3, 128                    117 / 98        182 / 159        99 / 67        155 / 113
//   160^3, 512                    141 / 143       210 / 258        118 / 104      194 / 196
//   256^3, 256                    468 / 369       825 / 727        398 / 263      711 / 557
//   256^3, 512                    510 / 486       778 / 944        419 / 367      748 / 750
//   256^3, 1024                   607 / 880       1267 / 1746      435 / 680      862 / 1319
// Clustered ones take less by windows throughout (128^3, 128 per brick: vector 54 / 100, tensor NGP
// 68 / 121; 256^3, 256: vector 400 / 475, vector NGP 325 / 328), which the host cannot know.
static bool tiles_c_path(const lf2mi_parts_s *p, int kind, int target, bool pm) {
    if ((kind == LF2MI_PROJ_SCALAR && !pm) || target != LF2MI_DEP_PERIODIC || p->g.B != 8 || p->g.NB % TC_TB != 0 ||
        p->N > 1024)
        return false;
    return p->N >= 512 || (p->N >= 160 && p->np < (kind == LF2MI_PROJ_VECTOR_NGP ? 768 : 384) * p->g.nbk);
}

// the shell buffer of deposit_tiles_c_kernel (grown on demand), its layout, the fold and the
// window deposit of the dense bricks
template <int KIND>
static int launch_tiles_c(lf2mi_parts_s *p, DepArgs A, bool pm, bool overwrite, hipStream_t st) {
    constexpr int C = KindC<KIND>::C, TB = TC_TB;
    const int64_t N = p->N, NB = p->g.NB, ntile = NB / TB;
    TcArgs T{};
    TcFold F{};
    F.C = C;
    F.TX = 8 * TB;
    F.ntile = (int)ntile;
    bool ry[2] = {false, false}, rz[2] = {false, false}, rx[2] = {false, false};  // layers 0 / 7
    int64_t off = 0;
    for (int c = 0; c < C; ++c) {
        const int mask = TC_MASK[KIND][c], ngp = TC_NGP[KIND][c];
        T.shell_off[c] = F.shell_off[c] = off;
        F.rows[c] = tc_rows(mask, ngp);
        F.ns[c] = tc_nl(mask, 0) + tc_nh(ngp, 0);
        for (int d = 0; d < 3; ++d) {
            F.lo[c][d] = -tc_nl(mask, d);
            F.hi[c][d] = 7 + tc_nh(ngp, d);
            F.w[c][d] = tc_w(mask, ngp, d);
        }
        ry[0] |= tc_nh(ngp, 1) != 0;
        ry[1] |= tc_nl(mask, 1) != 0;
        rz[0] |= tc_nh(ngp, 2) != 0;
        rz[1] |= tc_nl(mask, 2) != 0;
        rx[0] |= tc_nh(ngp, 0) != 0;
        rx[1] |= tc_nl(mask, 0) != 0;
        off += NB * NB * F.rows[c] * N;
    }
    int64_t seams = 0;
    for (int c = 0; c < C; ++c) {
        T.seam_off[c] = F.seam_off[c] = off + seams;
        seams += NB * NB * ntile * tc_seam(TC_MASK[KIND][c], TC_NGP[KIND][c]);
    }
    auto layers = [](const bool (&r)[2], int last, int *s, int *cpl, int &ns) {
        ns = 0;
        int nc = 0;
        for (int l = 0; l <= 7; ++l) {
            const bool recv = (l == 0 && r[0]) || (l == 7 && r[1]);
            if (recv) s[ns++] = l == 7 ? last : 0;
            else if (cpl) cpl[nc++] = l;
        }
    };
    layers(ry, 7, F.sy, F.cy, F.ny);
    layers(rz, 7, F.sz, F.cz, F.nz);
    layers(rx, F.TX - 1, F.sx, nullptr, F.nx);
    const int64_t bytes = (off + seams) * (int64_t)sizeof(float);
    if (p->shell_bytes < bytes) {
        if (p->shell) hipFree(p->shell);
        p->shell = nullptr;
        p->shell_bytes = 0;
        LF2MI_HIP(hipMalloc(&p->shell, (size_t)bytes));
        p->shell_bytes = bytes;
    }
    float *shell = (float *)p->shell;
    const unsigned grid = (unsigned)(NB * NB * ntile);
    if (pm) deposit_tiles_c_kernel<KIND, true, TB><<<grid, 64 * TB, 0, st>>>(A, DENSE_MIN, overwrite ? 1 : 0, T, shell);
    else deposit_tiles_c_kernel<KIND, false, TB><<<grid, 64 * TB, 0, st>>>(A, DENSE_MIN, overwrite ? 1 : 0, T, shell);
    LF2MI_LAUNCHED();
    const int64_t rows = (int64_t)F.ny * NB * N + (int64_t)(8 - F.ny) * NB * F.nz * NB;
    if (rows > 0) {
        fold_rows_kernel<C><<<(unsigned)rows, 256, 0, st>>>(A.field, (int)N, A.h, (int)NB, F, shell);
        LF2MI_LAUNCHED();
    }
    const int64_t edges = (int64_t)F.nx * ntile * (8 - F.ny) * NB * (8 - F.nz) * NB;
    if (edges > 0) {
        fold_edges_kernel<C><<<grid1(edges), 256, 0, st>>>(A.field, (int)N, A.h, (int)NB, F, shell, edges);
        LF2MI_LAUNCHED();
    }
    launch_bricks<KIND, float>(p, A, dense_workers(p), p->dgroups, p->ndgroup, st);
    LF2MI_LAUNCHED();
    return LF2MI_OK;
}

static int ic_common(lf2mi_parts_s *p, IcArgs &A, hipStream_t st) {
    if (A.np > p->cap) return fail(LF2MI_ERANGE, "%lld particles exceed the capacity %lld", (long long)A.np, (long long)p->cap);
    if (p->dtype == LF2MI_F32) {
        if (int rc = fill_int(p->bcount, p->g.nbk, 0, st)) return rc;
        const int src = 1 - p->cur;
        ic_f32_kernel<<<grid1(A.np), 256, 0, st>>>(A, p->b32[src], p->g, p->bcount);
        LF2MI_LAUNCHED();
        if (p->plw && A.np > 0)
            LF2MI_HIP(hipMemsetAsync(p->b32[src].pl, 0, (size_t)A.np * p->plw * sizeof(unsigned long long), st));
        if (int rc = sort_into_other(p, src, A.np, false, 0.0, st)) return rc;
        if (int rc = read_total(p, st, &p->np)) return rc;
    } else {
        p->np = A.np;
        p->in_box = 1;
        if (A.np > 0)
            if (int rc = b64_fill(p, nullptr, nullptr, nullptr, nullptr, nullptr, A, st)) {
                p->np = 0;
                return rc;
            }
        if (p->plw && A.np > 0)
            LF2MI_HIP(hipMemsetAsync(p->b64.pl, 0, (size_t)A.np * p->plw * sizeof(unsigned long long), st));
        LF2MI_HIP(hipStreamSynchronize(st));
    }
    // synthetic particles: per-particle masses (when kept) are 1
    p->total_mass = (p->mass_src ? 1.0 : p->mass_global) * (double)p->np;
    return LF2MI_OK;
}

}  // namespace lf2mi

using namespace lf2mi;

namespace lf2mi {

// sum of the stored per-particle masses: per-workgroup partial sums (grid-stride, a tree in
// LDS), then mass_total_kernel adds the partials in order, so the total is the same from
// run to run
template <typename T>
__global__ __launch_bounds__(RED_WG) void mass_partial_kernel(int64_t np, const T *__restrict__ mass,
                                                              const int *__restrict__ slot,
                                                              double *__restrict__ partial) {
    __shared__ double lds[RED_WG];
    double m = 0.0;
    const int64_t stride = (int64_t)gridDim.x * RED_WG;
    for (int64_t i = (int64_t)blockIdx.x * RED_WG + threadIdx.x; i < np; i += stride)
        m += (double)mass[slot ? slot[i] : i];
    lds[threadIdx.x] = m;
    __syncthreads();
    for (int h = RED_WG / 2; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) lds[threadIdx.x] += lds[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = lds[0];
}
__global__ void mass_total_kernel(const double *__restrict__ partial, int nblocks, double *__restrict__ total) {
    double t = 0.0;
    for (int b = 0; b < nblocks; ++b) t += partial[b];
    *total = t;
}

// per-particle masses from the value of type S (double, or float) at byte `off` of each
// payload
template <typename T, typename S>
__global__ void payload_mass_kernel(int64_t np, const unsigned long long *__restrict__ pl, int plw, int64_t off,
                                    T *__restrict__ mass) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= np) return;
    const unsigned char *b = reinterpret_cast<const unsigned char *>(pl + i * plw);
    S v;
    memcpy(&v, b + off, sizeof(S));
    mass[i] = (T)v;
}

// the Real[3] at byte `off` of each payload into three planes of `cap` values
template <typename T, typename R>
__global__ void payload_vec_kernel(int64_t np, const unsigned long long *__restrict__ pl, int plw, int64_t off,
                                   T *__restrict__ out, int64_t cap) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= np) return;
    const unsigned char *b = reinterpret_cast<const unsigned char *>(pl + i * plw) + off;
    R v[3];
    memcpy(v, b, sizeof v);
    out[i] = (T)v[0];
    out[cap + i] = (T)v[1];
    out[2 * cap + i] = (T)v[2];
}

// point the deposit's velocity planes at the vector selected by lf2mi_parts_vector_from
// (gathered from the payload on this stream)
template <typename T>
static int vector_source(lf2mi_parts_s *p, const unsigned long long *pl, T *(&vel)[3], hipStream_t st) {
    if (p->vec_off < 0) return LF2MI_OK;
    const int64_t cap = std::max<int64_t>(p->cap, 1);
    if (!p->vsrc)
        if (int rc = dalloc(p, &p->vsrc, (size_t)cap * 3 * sizeof(T))) return rc;
    T *out = static_cast<T *>(p->vsrc);
    if (p->vec_real == LF2MI_F32)
        payload_vec_kernel<T, float><<<grid1(p->np), 256, 0, st>>>(p->np, pl, p->plw, p->vec_off, out, cap);
    else
        payload_vec_kernel<T, double><<<grid1(p->np), 256, 0, st>>>(p->np, pl, p->plw, p->vec_off, out, cap);
    LF2MI_LAUNCHED();
    for (int d = 0; d < 3; ++d) vel[d] = out + d * cap;
    return LF2MI_OK;
}

}  // namespace lf2mi

extern "C" {

int lf2mi_parts_create(int N, int64_t capacity, int dtype, int flags, lf2mi_parts *out) {
    if (!out) return fail(LF2MI_EINVAL, "lf2mi_parts_create: null output");
    *out = nullptr;
    if (N < 2 || N > 1290) return fail(LF2MI_ERANGE, "lattice size N=%d outside [2, 1290]", N);
    if (capacity < 0 || capacity > 2000000000LL) return fail(LF2MI_ERANGE, "capacity %lld outside [0, 2e9]", (long long)capacity);
    if (dtype != LF2MI_F32 && dtype != LF2MI_F64) return fail(LF2MI_EINVAL, "bad dtype %d", dtype);
    lf2mi_parts_s *p = new (std::nothrow) lf2mi_parts_s();
    if (!p) return fail(LF2MI_ENOMEM, "host allocation failed");
    p->N = N;
    p->dtype = dtype;
    p->flags = flags;
    hipGetDevice(&p->device);
    p->cap = capacity;
    p->np = 0;
    p->mass_global = 1.0;
    p->cur = 0;
    p->plw = 0;
    p->mass_src = (flags & LF2MI_PARTS_MASS) ? 1 : 0;
    p->vec_off = -1;
    p->vec_real = LF2MI_F32;
    p->aos_vel = -1;
    p->vsrc = nullptr;
    int B = 1;
    for (int b = MAXB; b >= 1; --b)
        if (N % b == 0) { B = b; break; }
    p->g.N = N;
    p->g.B = B;
    p->g.NB = N / B;
    p->g.nbk = (int64_t)p->g.NB * p->g.NB * p->g.NB;
    p->g.lgN = is_pow2(N) ? __builtin_ctz((unsigned)N) : -1;
    p->g.lgB = is_pow2(B) ? __builtin_ctz((unsigned)B) : -1;
    const size_t cap = (size_t)std::max<int64_t>(capacity, 1);
    int rc = LF2MI_OK;
    auto A = [&](void **ptr, size_t bytes) {
        if (!rc) rc = dalloc(p, ptr, bytes);
    };
    if (dtype == LF2MI_F32) {
        for (int k = 0; k < 2; ++k) {
            Soa32 &s = p->b32[k];
            A((void **)&s.cell, cap * sizeof(int32_t));
            for (int d = 0; d < 3; ++d) {
                A((void **)&s.off[d], cap * sizeof(float));
                A((void **)&s.vel[d], cap * sizeof(float));
            }
            s.mass = nullptr;
            s.id = nullptr;
            s.pl = nullptr;
            if (flags & LF2MI_PARTS_MASS) A((void **)&s.mass, cap * sizeof(float));
            if (flags & LF2MI_PARTS_ID) A((void **)&s.id, cap * sizeof(int64_t));
        }
        const size_t nb = (size_t)p->g.nbk + 1;
        A((void **)&p->bstart, nb * sizeof(int));
        A((void **)&p->istart, nb * sizeof(int));
        A((void **)&p->bcount, nb * sizeof(int));
        A((void **)&p->bsum, 3 * 4096 * sizeof(int));
        A((void **)&p->cursor, nb * sizeof(int));
        A((void **)&p->item_bucket, (size_t)(p->g.nbk + cap / ITEM_P + 1) * sizeof(int));
        A((void **)&p->vmax_f32, sizeof(unsigned int));
        A((void **)&p->dgroups, (size_t)(cap / (DEP_MERGE * ITEM_P) + p->g.nbk + 1) * sizeof(int2));
        A((void **)&p->ndgroup, sizeof(int));
        A((void **)&p->chunks, (size_t)p->g.nbk * sizeof(int4));
        A((void **)&p->nchunk, 2 * sizeof(int));
    } else {
        Soa64 &s = p->b64;
        A((void **)&s.cell, cap * sizeof(int32_t));
        for (int d = 0; d < 3; ++d) {
            A((void **)&s.pos[d], cap * sizeof(double));
            A((void **)&s.vel[d], cap * sizeof(double));
        }
        s.mass = nullptr;
        s.id = nullptr;
        s.pl = nullptr;
        if (flags & LF2MI_PARTS_MASS) A((void **)&s.mass, cap * sizeof(double));
        if (flags & LF2MI_PARTS_ID) A((void **)&s.id, cap * sizeof(int64_t));
        A((void **)&p->vmax_f64, sizeof(unsigned long long));
    }
    A((void **)&p->red, (size_t)(RED_BLOCKS + 1) * RED_Q * sizeof(double));
    if (rc) {
        for (void *q : p->allocs) hipFree(q);
        delete p;
        return rc;
    }
    if (dtype == LF2MI_F64) b64_create(p);
    if (dtype == LF2MI_F32) {
        hipMemset(p->bstart, 0, ((size_t)p->g.nbk + 1) * sizeof(int));
        hipMemset(p->istart, 0, ((size_t)p->g.nbk + 1) * sizeof(int));
        hipMemset(p->bcount, 0, ((size_t)p->g.nbk + 1) * sizeof(int));
        hipMemset(p->ndgroup, 0, sizeof(int));
        hipMemset(p->nchunk, 0, 2 * sizeof(int));
    }
    // the counters have to be clear before the first use, which may be on a stream that does not wait
    // for this one
    (void)hipStreamSynchronize(nullptr);
    *out = p;
    return LF2MI_OK;
}

int lf2mi_parts_destroy(lf2mi_parts p) {
    if (!p) return LF2MI_OK;
    for (void *q : p->allocs) hipFree(q);
    if (p->fx) hipFree(p->fx);
    if (p->shell) hipFree(p->shell);
    delete p;
    return LF2MI_OK;
}

int lf2mi_parts_set_mass(lf2mi_parts p, double m) {
    if (!p) return fail(LF2MI_EINVAL, "null container");
    if (p->total_mass != 0.0 && !(p->flags & LF2MI_PARTS_MASS)) p->total_mass = m * (double)p->np;
    p->mass_global = m;
    if (!(p->flags & LF2MI_PARTS_MASS)) p->total_mass = m * (double)p->np;
    return LF2MI_OK;
}

int lf2mi_parts_count(lf2mi_parts p, int64_t *np) {
    if (!p || !np) return fail(LF2MI_EINVAL, "null argument");
    *np = p->np;
    return LF2MI_OK;
}

int lf2mi_parts_bytes(lf2mi_parts p, int64_t *bytes) {
    if (!p || !bytes) return fail(LF2MI_EINVAL, "null argument");
    *bytes = p->bytes;
    return LF2MI_OK;
}

// the upload; pl (may be null) holds each input particle's payload (p->plw words, in input
// order), zeros when the container keeps payloads and none is given
static int upload_impl(lf2mi_parts p, int64_t np, const double *pos, const double *vel, const double *mass,
                       const int64_t *id, const unsigned char *pl, int64_t *kept, void *stream) {
    if (!p || np < 0 || (np > 0 && (!pos || !vel))) return fail(LF2MI_EINVAL, "lf2mi_parts_upload: bad argument");
    if (np > p->cap) return fail(LF2MI_ERANGE, "%lld particles exceed the capacity %lld", (long long)np, (long long)p->cap);
    if ((p->flags & LF2MI_PARTS_MASS) && np > 0 && !mass) return fail(LF2MI_EINVAL, "per-particle masses required");
    hipStream_t st = as_stream(stream);
    // drop what the reference's setCoord rejects (negative cell coordinates) on the host,
    // so the device arrays hold only valid particles
    std::vector<int64_t> keep;
    keep.reserve((size_t)np);
    int in_box = 1;
    for (int64_t i = 0; i < np; ++i) {
        bool ok = true;
        for (int d = 0; d < 3; ++d) {
            if ((int)floor(pos[3 * i + d] * (double)p->N) % p->N < 0) ok = false;
            if (!(pos[3 * i + d] >= 0.0 && pos[3 * i + d] < 1.0)) in_box = 0;
        }
        if (ok) keep.push_back(i);
    }
    const int64_t nk = (int64_t)keep.size();
    std::vector<double> hp((size_t)nk * 3), hv((size_t)nk * 3), hm(mass ? (size_t)nk : 0);
    std::vector<int64_t> hid((size_t)nk);
    double msum = 0.0;
    for (int64_t k = 0; k < nk; ++k) {
        const int64_t i = keep[(size_t)k];
        for (int d = 0; d < 3; ++d) {
            hp[3 * k + d] = pos[3 * i + d];
            hv[3 * k + d] = vel[3 * i + d];
        }
        if (mass) {
            hm[(size_t)k] = mass[i];
            msum += mass[i];
        }
        hid[(size_t)k] = id ? id[i] : i;
    }
    const size_t plb = (size_t)p->plw * sizeof(unsigned long long);
    std::vector<unsigned char> hpl(plb * (size_t)nk, 0);
    if (pl)
        for (int64_t k = 0; k < nk; ++k) memcpy(hpl.data() + plb * (size_t)k, pl + plb * (size_t)keep[(size_t)k], plb);
    double *dpos = nullptr, *dvel = nullptr, *dmass = nullptr;
    int64_t *did = nullptr;
    unsigned long long *dpl = nullptr;
    if (plb) LF2MI_HIP(hipMalloc((void **)&dpl, plb * (size_t)std::max<int64_t>(nk, 1)));
    const size_t n3 = (size_t)std::max<int64_t>(nk, 1) * 3;
    LF2MI_HIP(hipMalloc((void **)&dpos, n3 * sizeof(double)));
    LF2MI_HIP(hipMalloc((void **)&dvel, n3 * sizeof(double)));
    LF2MI_HIP(hipMalloc((void **)&did, (n3 / 3) * sizeof(int64_t)));
    if (mass) LF2MI_HIP(hipMalloc((void **)&dmass, (n3 / 3) * sizeof(double)));
    int rc = LF2MI_OK;
    hipError_t e = hipSuccess;
    if (nk > 0) {
        e = hipMemcpyAsync(dpos, hp.data(), nk * 3 * sizeof(double), hipMemcpyHostToDevice, st);
        if (e == hipSuccess) e = hipMemcpyAsync(dvel, hv.data(), nk * 3 * sizeof(double), hipMemcpyHostToDevice, st);
        if (e == hipSuccess) e = hipMemcpyAsync(did, hid.data(), nk * sizeof(int64_t), hipMemcpyHostToDevice, st);
        if (e == hipSuccess && mass) e = hipMemcpyAsync(dmass, hm.data(), nk * sizeof(double), hipMemcpyHostToDevice, st);
        if (e == hipSuccess && plb) e = hipMemcpyAsync(dpl, hpl.data(), plb * (size_t)nk, hipMemcpyHostToDevice, st);
    }
    if (e != hipSuccess) rc = hip_fail(e, "hipMemcpyAsync(upload)", __FILE__, __LINE__);
    if (!rc) {
        if (p->dtype == LF2MI_F32) {
            rc = fill_int(p->bcount, p->g.nbk, 0, st);
            const int src = 1 - p->cur;
            if (!rc && nk > 0) {
                bin_upload_kernel<<<grid1(nk), 256, 0, st>>>(nk, dpos, dvel, dmass, did, dpl, p->plw, p->b32[src], p->g,
                                                             p->bcount);
                if ((e = hipGetLastError()) != hipSuccess) rc = hip_fail(e, "bin_upload_kernel", __FILE__, __LINE__);
            }
            if (!rc) rc = sort_into_other(p, src, nk, false, 0.0, st);
            if (!rc) rc = read_total(p, st, &p->np);
        } else {
            p->np = nk;
            p->in_box = in_box;
            if (nk > 0) rc = b64_fill(p, dpos, dvel, dmass, did, dpl, IcArgs{}, st);
            if (rc) p->np = 0;
            if (!rc && (e = hipStreamSynchronize(st)) != hipSuccess) rc = hip_fail(e, "sync", __FILE__, __LINE__);
        }
    }
    hipStreamSynchronize(st);
    hipFree(dpos);
    hipFree(dvel);
    hipFree(did);
    if (dmass) hipFree(dmass);
    if (dpl) hipFree(dpl);
    if (rc) return rc;
    p->total_mass = mass && p->mass_src ? msum : p->mass_global * (double)p->np;
    if (kept) *kept = p->np;
    return LF2MI_OK;
}

int lf2mi_parts_upload(lf2mi_parts p, int64_t np, const double *pos, const double *vel, const double *mass,
                       const int64_t *id, int64_t *kept, void *stream) {
    return upload_impl(p, np, pos, vel, mass, id, nullptr, kept, stream);
}

int lf2mi_parts_download(lf2mi_parts p, double *pos, double *vel, double *mass, int64_t *id, int32_t *cell,
                         void *stream) {
    if (!p) return fail(LF2MI_EINVAL, "null container");
    hipStream_t st = as_stream(stream);
    const int64_t np = p->np;
    if (np == 0) return LF2MI_OK;
    double *dpos = nullptr, *dvel = nullptr, *dmass = nullptr;
    LF2MI_HIP(hipMalloc((void **)&dpos, np * 3 * sizeof(double)));
    LF2MI_HIP(hipMalloc((void **)&dvel, np * 3 * sizeof(double)));
    LF2MI_HIP(hipMalloc((void **)&dmass, np * sizeof(double)));
    int rc = LF2MI_OK;
    if (p->dtype == LF2MI_F32) {
        Soa32 s = p->b32[p->cur];
        if (!p->mass_src) s.mass = nullptr;  // the global mass is the one in use
        download_f32_kernel<<<grid1(np), 256, 0, st>>>(np, s, p->N, dpos, dvel, dmass, p->mass_global);
        hipError_t e = hipGetLastError();
        if (e == hipSuccess && pos) e = hipMemcpyAsync(pos, dpos, np * 3 * sizeof(double), hipMemcpyDeviceToHost, st);
        if (e == hipSuccess && vel) e = hipMemcpyAsync(vel, dvel, np * 3 * sizeof(double), hipMemcpyDeviceToHost, st);
        if (e == hipSuccess && mass) e = hipMemcpyAsync(mass, dmass, np * sizeof(double), hipMemcpyDeviceToHost, st);
        if (e == hipSuccess && id) {
            if (s.id) e = hipMemcpyAsync(id, s.id, np * sizeof(int64_t), hipMemcpyDeviceToHost, st);
            else rc = fail(LF2MI_EINVAL, "container keeps no IDs");
        }
        if (e == hipSuccess && cell) e = hipMemcpyAsync(cell, s.cell, np * sizeof(int32_t), hipMemcpyDeviceToHost, st);
        if (e != hipSuccess) rc = hip_fail(e, "download", __FILE__, __LINE__);
    } else {
        const Soa64 &s = p->b64;
        const int *slot = p->sorted ? p->slot : nullptr;
        download_f64_kernel<<<grid1(np), 256, 0, st>>>(np, s, slot, dpos, dvel);
        hipError_t e = hipGetLastError();
        if (e == hipSuccess && pos) e = hipMemcpyAsync(pos, dpos, np * 3 * sizeof(double), hipMemcpyDeviceToHost, st);
        if (e == hipSuccess && vel) e = hipMemcpyAsync(vel, dvel, np * 3 * sizeof(double), hipMemcpyDeviceToHost, st);
        // the other arrays go through dmass, which holds 8 bytes per particle, in upload order
        auto out = [&](auto *host, const auto *dev) {
            using T = std::remove_cv_t<std::remove_pointer_t<decltype(host)>>;
            static_assert(sizeof(T) <= sizeof(double), "staged in dmass");
            const T *from = dev;
            if (slot) {
                unsort_kernel<T><<<grid1(np), 256, 0, st>>>(np, dev, 1, slot, (T *)dmass);
                if ((e = hipGetLastError()) != hipSuccess) return;
                from = (const T *)dmass;
            }
            e = hipMemcpyAsync(host, from, np * sizeof(T), hipMemcpyDeviceToHost, st);
        };
        if (e == hipSuccess && mass) {
            if (s.mass && p->mass_src) out(mass, s.mass);
            else for (int64_t i = 0; i < np; ++i) mass[i] = p->mass_global;
        }
        if (e == hipSuccess && id) {
            if (s.id) out(id, s.id);
            else rc = fail(LF2MI_EINVAL, "container keeps no IDs");
        }
        if (e == hipSuccess && cell) out(cell, s.cell);
        if (e != hipSuccess) rc = hip_fail(e, "download", __FILE__, __LINE__);
    }
    hipStreamSynchronize(st);
    hipFree(dpos);
    hipFree(dvel);
    hipFree(dmass);
    return rc;
}

// ---------------------------------------------------------------- user structs
int lf2mi_parts_set_payload(lf2mi_parts p, int bytes) {
    if (!p) return fail(LF2MI_EINVAL, "null container");
    if (bytes < 0 || bytes > 4096 || bytes % 8) return fail(LF2MI_EINVAL, "payload of %d bytes: a multiple of 8 up to 4096", bytes);
    if (p->np > 0 || p->plw) return fail(LF2MI_EINVAL, "the payload is set once, before the first upload");
    if (bytes == 0) return LF2MI_OK;
    const size_t cap = (size_t)std::max<int64_t>(p->cap, 1);
    int rc = LF2MI_OK;
    if (p->dtype == LF2MI_F32) {
        for (int k = 0; k < 2 && !rc; ++k) {
            Soa32 &s = p->b32[k];
            rc = dalloc(p, (void **)&s.pl, cap * (size_t)bytes);
            if (!rc && !s.mass) rc = dalloc(p, (void **)&s.mass, cap * sizeof(float));
        }
    } else {
        rc = dalloc(p, (void **)&p->b64.pl, cap * (size_t)bytes);
        if (!rc && !p->b64.mass) rc = dalloc(p, (void **)&p->b64.mass, cap * sizeof(double));
    }
    if (rc) return rc;
    p->plw = bytes / 8;
    return LF2MI_OK;
}

static bool real_field_ok(int64_t off, int64_t size, int64_t stride) { return off < 0 || off + size <= stride; }

int lf2mi_parts_upload_aos(lf2mi_parts p, int64_t n, const void *base, int64_t stride, int real_dtype,
                           int64_t off_pos, int64_t off_vel, int64_t off_id, int64_t off_mass, int64_t *kept,
                           void *stream) {
    if (!p || n < 0 || (n > 0 && !base) || stride <= 0) return fail(LF2MI_EINVAL, "lf2mi_parts_upload_aos: bad argument");
    if (real_dtype != LF2MI_F32 && real_dtype != LF2MI_F64) return fail(LF2MI_EINVAL, "bad real dtype %d", real_dtype);
    const int64_t rs = real_dtype == LF2MI_F32 ? 4 : 8;
    if (off_pos < 0 || off_vel < 0 || !real_field_ok(off_pos, 3 * rs, stride) || !real_field_ok(off_vel, 3 * rs, stride) ||
        !real_field_ok(off_id, 8, stride) || !real_field_ok(off_mass, 8, stride))
        return fail(LF2MI_EINVAL, "field offsets outside the %lld-byte struct", (long long)stride);
    if (p->plw && stride != (int64_t)p->plw * 8)
        return fail(LF2MI_EINVAL, "struct of %lld bytes against a payload of %d", (long long)stride, p->plw * 8);
    if (off_mass >= 0 && !(p->dtype == LF2MI_F32 ? (void *)p->b32[0].mass : (void *)p->b64.mass))
        return fail(LF2MI_EINVAL, "per-particle masses need a container with masses or a payload");
    const unsigned char *b = static_cast<const unsigned char *>(base);
    std::vector<double> pos((size_t)n * 3), vel((size_t)n * 3), mass(off_mass >= 0 ? (size_t)n : 0);
    std::vector<int64_t> id(off_id >= 0 ? (size_t)n : 0);
    for (int64_t i = 0; i < n; ++i) {
        const unsigned char *q = b + i * stride;
        for (int d = 0; d < 3; ++d) {
            if (rs == 4) {
                float x, v;
                memcpy(&x, q + off_pos + 4 * d, 4);
                memcpy(&v, q + off_vel + 4 * d, 4);
                pos[3 * i + d] = x;
                vel[3 * i + d] = v;
            } else {
                memcpy(&pos[3 * i + d], q + off_pos + 8 * d, 8);
                memcpy(&vel[3 * i + d], q + off_vel + 8 * d, 8);
            }
        }
        if (off_id >= 0) memcpy(&id[(size_t)i], q + off_id, 8);
        if (off_mass >= 0) memcpy(&mass[(size_t)i], q + off_mass, 8);
    }
    if (p->plw) p->aos_vel = off_vel;
    // a container with per-particle masses whose structs carry none readable as a double (a
    // float member, gathered afterwards by lf2mi_parts_mass_from) starts at mass 0
    const bool zero_mass = off_mass < 0 && (p->flags & LF2MI_PARTS_MASS) && p->plw;
    if (zero_mass) mass.assign((size_t)n, 0.0);
    return upload_impl(p, n, pos.data(), vel.data(), (off_mass >= 0 || zero_mass) ? mass.data() : nullptr,
                       off_id >= 0 ? id.data() : nullptr, p->plw ? b : nullptr, kept, stream);
}

int lf2mi_parts_download_aos(lf2mi_parts p, void *base, int64_t n_room, int64_t stride, int real_dtype,
                             int64_t off_pos, int64_t off_vel, int64_t off_id, int64_t *n_out, void *stream) {
    if (!p || stride <= 0 || n_room < 0) return fail(LF2MI_EINVAL, "lf2mi_parts_download_aos: bad argument");
    if (real_dtype != LF2MI_F32 && real_dtype != LF2MI_F64) return fail(LF2MI_EINVAL, "bad real dtype %d", real_dtype);
    const int64_t rs = real_dtype == LF2MI_F32 ? 4 : 8;
    if (!real_field_ok(off_pos, 3 * rs, stride) || !real_field_ok(off_vel, 3 * rs, stride) || !real_field_ok(off_id, 8, stride))
        return fail(LF2MI_EINVAL, "field offsets outside the %lld-byte struct", (long long)stride);
    if (p->plw && stride != (int64_t)p->plw * 8)
        return fail(LF2MI_EINVAL, "struct of %lld bytes against a payload of %d", (long long)stride, p->plw * 8);
    const int64_t np = p->np;
    if (n_out) *n_out = np;
    if (np > n_room) return fail(LF2MI_ERANGE, "%lld particles exceed the room for %lld", (long long)np, (long long)n_room);
    if (np == 0) return LF2MI_OK;
    if (!base) return fail(LF2MI_EINVAL, "lf2mi_parts_download_aos: null buffer");
    hipStream_t st = as_stream(stream);
    std::vector<double> pos((size_t)np * 3), vel((size_t)np * 3);
    std::vector<int64_t> id(off_id >= 0 ? (size_t)np : 0);
    if (int rc = lf2mi_parts_download(p, pos.data(), vel.data(), nullptr, off_id >= 0 ? id.data() : nullptr, nullptr,
                                      stream))
        return rc;
    unsigned char *b = static_cast<unsigned char *>(base);
    if (p->plw) {
        const unsigned long long *pl = p->dtype == LF2MI_F32 ? p->b32[p->cur].pl : p->b64.pl;
        unsigned long long *tmp = nullptr;
        if (p->dtype == LF2MI_F64 && p->sorted) {
            LF2MI_HIP(hipMalloc((void **)&tmp, (size_t)np * p->plw * 8));
            unsort_kernel<unsigned long long><<<grid1(np), 256, 0, st>>>(np, pl, p->plw, p->slot, tmp);
            pl = tmp;
        }
        hipError_t e = hipGetLastError();
        if (e == hipSuccess) e = hipMemcpyAsync(b, pl, (size_t)np * p->plw * 8, hipMemcpyDeviceToHost, st);
        const hipError_t e2 = hipStreamSynchronize(st);
        if (tmp) hipFree(tmp);
        if (e != hipSuccess || e2 != hipSuccess) return hip_fail(e != hipSuccess ? e : e2, "payload", __FILE__, __LINE__);
    }
    for (int64_t i = 0; i < np; ++i) {
        unsigned char *q = b + i * stride;
        for (int d = 0; d < 3; ++d) {
            if (off_pos >= 0) {
                if (rs == 4) {
                    const float x = (float)pos[3 * i + d];
                    memcpy(q + off_pos + 4 * d, &x, 4);
                } else {
                    memcpy(q + off_pos + 8 * d, &pos[3 * i + d], 8);
                }
            }
            if (off_vel >= 0) {
                if (rs == 4) {
                    const float v = (float)vel[3 * i + d];
                    memcpy(q + off_vel + 4 * d, &v, 4);
                } else {
                    memcpy(q + off_vel + 8 * d, &vel[3 * i + d], 8);
                }
            }
        }
        if (off_id >= 0) memcpy(q + off_id, &id[(size_t)i], 8);
    }
    return LF2MI_OK;
}

int lf2mi_parts_mass_from(lf2mi_parts p, int where, int64_t offset, void *stream) {
    if (!p) return fail(LF2MI_EINVAL, "null container");
    if (where != LF2MI_MASS_INFO && where != LF2MI_MASS_PART && where != LF2MI_MASS_PART_F32)
        return fail(LF2MI_EINVAL, "bad mass source %d", where);
    if (where == LF2MI_MASS_INFO) {
        p->mass_src = 0;
        p->total_mass = p->mass_global * (double)p->np;
        return LF2MI_OK;
    }
    const bool has_mass = p->dtype == LF2MI_F32 ? p->b32[0].mass != nullptr : p->b64.mass != nullptr;
    if (!has_mass) return fail(LF2MI_EINVAL, "per-particle masses need a container with masses or a payload");
    const int64_t msize = where == LF2MI_MASS_PART_F32 ? 4 : 8;
    if (offset >= 0 && (!p->plw || offset + msize > (int64_t)p->plw * 8)) {
        return fail(LF2MI_EINVAL, "mass offset %lld outside the payload", (long long)offset);
    }
    hipStream_t st = as_stream(stream);
    double *res = p->red + (int64_t)RED_BLOCKS * RED_Q;  // the partials before it
    const int nb = (int)std::max<int64_t>(1, std::min<int64_t>(RED_BLOCKS, (p->np + RED_WG - 1) / RED_WG));
    if (offset >= 0 && p->np > 0) {
        const bool f4 = where == LF2MI_MASS_PART_F32;
        const unsigned g = grid1(p->np);
        if (p->dtype == LF2MI_F32) {
            Soa32 &s = p->b32[p->cur];
            if (f4) payload_mass_kernel<float, float><<<g, 256, 0, st>>>(p->np, s.pl, p->plw, offset, s.mass);
            else payload_mass_kernel<float, double><<<g, 256, 0, st>>>(p->np, s.pl, p->plw, offset, s.mass);
        } else {
            Soa64 &s = p->b64;
            if (f4) payload_mass_kernel<double, float><<<g, 256, 0, st>>>(p->np, s.pl, p->plw, offset, s.mass);
            else payload_mass_kernel<double, double><<<g, 256, 0, st>>>(p->np, s.pl, p->plw, offset, s.mass);
        }
        LF2MI_LAUNCHED();
    }
    if (p->dtype == LF2MI_F32) mass_partial_kernel<float><<<nb, RED_WG, 0, st>>>(p->np, p->b32[p->cur].mass, nullptr, p->red);
    else
        mass_partial_kernel<double><<<nb, RED_WG, 0, st>>>(p->np, p->b64.mass, p->sorted ? p->slot : nullptr, p->red);
    LF2MI_LAUNCHED();
    mass_total_kernel<<<1, 1, 0, st>>>(p->red, nb, res);
    LF2MI_LAUNCHED();
    double total = 0.0;
    LF2MI_HIP(hipMemcpyAsync(&total, res, sizeof(double), hipMemcpyDeviceToHost, st));
    LF2MI_HIP(hipStreamSynchronize(st));
    p->mass_src = 1;
    p->total_mass = total;
    return LF2MI_OK;
}

int lf2mi_parts_vector_from(lf2mi_parts p, int64_t offset, int real_dtype) {
    if (!p) return fail(LF2MI_EINVAL, "null container");
    // the payload's copy of vel is the uploaded one: the kicked velocity lives in the container
    if (offset < 0 || offset == p->aos_vel) {
        p->vec_off = -1;
        return LF2MI_OK;
    }
    if (real_dtype != LF2MI_F32 && real_dtype != LF2MI_F64) return fail(LF2MI_EINVAL, "bad real dtype %d", real_dtype);
    const int64_t rs = real_dtype == LF2MI_F32 ? 4 : 8;
    if (!p->plw || offset + 3 * rs > (int64_t)p->plw * 8)
        return fail(LF2MI_EINVAL, "vector offset %lld outside the payload", (long long)offset);
    p->vec_off = offset;
    p->vec_real = real_dtype;
    return LF2MI_OK;
}

int lf2mi_parts_download_box(lf2mi_parts p, const int *lo, const int *hi, int64_t max_out, double *pos, double *vel,
                             double *mass, int64_t *n_out, void *stream) {
    if (!p || !lo || !hi || !n_out || max_out < 0 || (max_out > 0 && (!pos || !vel || !mass)))
        return fail(LF2MI_EINVAL, "lf2mi_parts_download_box: bad argument");
    BoxArgs A{};
    for (int d = 0; d < 3; ++d) {
        if (lo[d] < 0 || hi[d] > p->N || lo[d] >= hi[d]) return fail(LF2MI_ERANGE, "box [%d, %d) outside [0, %d)", lo[d], hi[d], p->N);
        A.lo[d] = lo[d];
        A.hi[d] = hi[d];
    }
    *n_out = 0;
    if (p->np == 0) return LF2MI_OK;
    hipStream_t st = as_stream(stream);
    const int64_t m = std::max<int64_t>(max_out, 1);
    double *d_pos = nullptr, *d_vel = nullptr, *d_mass = nullptr;
    int *d_cur = nullptr;
    hipError_t e = hipMalloc((void **)&d_pos, m * 3 * sizeof(double));
    if (e == hipSuccess) e = hipMalloc((void **)&d_vel, m * 3 * sizeof(double));
    if (e == hipSuccess) e = hipMalloc((void **)&d_mass, m * sizeof(double));
    if (e == hipSuccess) e = hipMalloc((void **)&d_cur, sizeof(int));
    if (e == hipSuccess) e = hipMemsetAsync(d_cur, 0, sizeof(int), st);
    int cnt = 0;
    if (e == hipSuccess) {
        A.N = p->N;
        A.np = p->np;
        A.max_out = max_out;
        A.cursor = d_cur;
        A.pos = d_pos;
        A.vel = d_vel;
        A.mass = d_mass;
        A.mass_global = p->mass_global;
        Soa32 s32 = p->b32[p->cur];
        Soa64 s64 = p->b64;
        if (!p->mass_src) s32.mass = nullptr, s64.mass = nullptr;
        if (p->dtype == LF2MI_F32) download_box_f32_kernel<<<grid1(p->np), 256, 0, st>>>(A, s32);
        else download_box_f64_kernel<<<grid1(p->np), 256, 0, st>>>(A, s64);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpyAsync(&cnt, d_cur, sizeof(int), hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    const int64_t n = std::min<int64_t>(cnt, max_out);
    if (e == hipSuccess && n > 0) e = hipMemcpy(pos, d_pos, n * 3 * sizeof(double), hipMemcpyDeviceToHost);
    if (e == hipSuccess && n > 0) e = hipMemcpy(vel, d_vel, n * 3 * sizeof(double), hipMemcpyDeviceToHost);
    if (e == hipSuccess && n > 0) e = hipMemcpy(mass, d_mass, n * sizeof(double), hipMemcpyDeviceToHost);
    hipFree(d_pos);
    hipFree(d_vel);
    hipFree(d_mass);
    hipFree(d_cur);
    if (e != hipSuccess) return hip_fail(e, "lf2mi_parts_download_box", __FILE__, __LINE__);
    *n_out = cnt;
    if (cnt > max_out) return fail(LF2MI_ERANGE, "%d particles in the box exceed max_out %lld", cnt, (long long)max_out);
    return LF2MI_OK;
}

int lf2mi_bin_positions(const double *pos, int64_t np, int N, int32_t *keys, int32_t *counts, void *stream) {
    if (np < 0 || (np > 0 && !pos) || N < 1 || N > 1290) return fail(LF2MI_EINVAL, "lf2mi_bin_positions: bad argument");
    hipStream_t st = as_stream(stream);
    if (counts)
        if (int rc = fill_int(counts, (int64_t)N * N * N, 0, st)) return rc;
    if (np == 0 || (!keys && !counts)) return LF2MI_OK;
    LF2MI_PROF("bin_keys", st);
    bin_keys_kernel<<<grid1(np), 256, 0, st>>>(np, pos, N, keys, counts);
    LF2MI_LAUNCHED();
    return LF2MI_OK;
}

int lf2mi_parts_cell_counts(lf2mi_parts p, int32_t *counts, void *stream) {
    if (!p || !counts) return fail(LF2MI_EINVAL, "null argument");
    hipStream_t st = as_stream(stream);
    const int64_t nc = (int64_t)p->N * p->N * p->N;
    if (int rc = fill_int(counts, nc, 0, st)) return rc;
    const int32_t *cell = p->dtype == LF2MI_F32 ? p->b32[p->cur].cell : p->b64.cell;
    if (p->np > 0) {
        cell_count_kernel<<<grid1(p->np), 256, 0, st>>>(p->np, cell, counts);
        LF2MI_LAUNCHED();
    }
    return LF2MI_OK;
}

int lf2mi_parts_ic_lattice(lf2mi_parts p, int ng, double sigma_cells, double sigma_v, uint64_t seed, void *stream) {
    if (!p || ng < 1) return fail(LF2MI_EINVAL, "bad argument");
    IcArgs A{};
    A.kind = 0;
    A.np = (int64_t)ng * ng * ng;
    A.ng = ng;
    A.sigma_pos = sigma_cells / p->N;
    A.sigma_v = sigma_v;
    A.seed = seed;
    return ic_common(p, A, as_stream(stream));
}

int lf2mi_parts_ic_uniform(lf2mi_parts p, int64_t np, double sigma_v, uint64_t seed, void *stream) {
    if (!p || np < 0) return fail(LF2MI_EINVAL, "bad argument");
    IcArgs A{};
    A.kind = 1;
    A.np = np;
    A.sigma_v = sigma_v;
    A.seed = seed;
    return ic_common(p, A, as_stream(stream));
}

int lf2mi_parts_ic_blobs(lf2mi_parts p, int64_t np, int nblobs, double alpha, double sigma_cells, double frac_uniform,
                         double sigma_v, uint64_t seed, void *stream) {
    if (!p || np < 0 || nblobs < 1 || !(alpha > 0) || frac_uniform < 0 || frac_uniform > 1)
        return fail(LF2MI_EINVAL, "bad argument");
    const int64_t ncl = np - (int64_t)llround(frac_uniform * (double)np);
    // Pareto(alpha) occupancies w = u^(-1/alpha), counts by largest remainder
    std::vector<double> w((size_t)nblobs), cen((size_t)nblobs * 3);
    double ws = 0.0;
    for (int b = 0; b < nblobs; ++b) {
        double u = urand(seed ^ 0xB10Bull, (uint64_t)b, 0);
        if (u < 1e-300) u = 1e-300;
        w[(size_t)b] = pow(u, -1.0 / alpha);
        ws += w[(size_t)b];
        for (int d = 0; d < 3; ++d) cen[(size_t)b * 3 + d] = urand(seed ^ 0xCE47ull, (uint64_t)b, (uint32_t)d);
    }
    std::vector<int64_t> cnt((size_t)nblobs);
    std::vector<std::pair<double, int>> rem((size_t)nblobs);
    int64_t assigned = 0;
    for (int b = 0; b < nblobs; ++b) {
        const double exact = w[(size_t)b] / ws * (double)ncl;
        cnt[(size_t)b] = (int64_t)floor(exact);
        assigned += cnt[(size_t)b];
        rem[(size_t)b] = {exact - floor(exact), b};
    }
    std::sort(rem.begin(), rem.end(), [](const std::pair<double, int> &a, const std::pair<double, int> &b) {
        return a.first > b.first || (a.first == b.first && a.second < b.second);
    });
    for (int64_t k = 0; k < ncl - assigned; ++k) cnt[(size_t)rem[(size_t)(k % nblobs)].second]++;
    std::vector<int64_t> bst((size_t)nblobs + 1, 0);
    for (int b = 0; b < nblobs; ++b) bst[(size_t)b + 1] = bst[(size_t)b] + cnt[(size_t)b];
    hipStream_t st = as_stream(stream);
    double *dcen = nullptr;
    int64_t *dbst = nullptr;
    LF2MI_HIP(hipMalloc((void **)&dcen, cen.size() * sizeof(double)));
    LF2MI_HIP(hipMalloc((void **)&dbst, bst.size() * sizeof(int64_t)));
    LF2MI_HIP(hipMemcpy(dcen, cen.data(), cen.size() * sizeof(double), hipMemcpyHostToDevice));
    LF2MI_HIP(hipMemcpy(dbst, bst.data(), bst.size() * sizeof(int64_t), hipMemcpyHostToDevice));
    IcArgs A{};
    A.kind = 2;
    A.np = np;
    A.sigma_pos = sigma_cells / p->N;
    A.sigma_v = sigma_v;
    A.seed = seed;
    A.nblobs = nblobs;
    A.nclustered = ncl;
    A.centres = dcen;
    A.bstart = dbst;
    const int rc = ic_common(p, A, st);
    hipStreamSynchronize(st);
    hipFree(dcen);
    hipFree(dbst);
    return rc;
}

}  // extern "C"

// overwrite: the native scalar deposit on the tiles path stores every interior node instead of
// adding to it (the PM step's deposit into a field it would otherwise clear first)
static int deposit_impl(lf2mi_parts p, int kind, void *field, int halo, int target, int acc, bool overwrite,
                        void *stream) {
    if (!p || !field) return fail(LF2MI_EINVAL, "lf2mi_deposit: null argument");
    if (kind < LF2MI_PROJ_SCALAR || kind > LF2MI_PROJ_SYMTENSOR_NGP)
        return fail(LF2MI_EINVAL, "bad projection kind %d", kind);
    if (halo < 1) return fail(LF2MI_EINVAL, "the field has to have at least a halo of 1");
    if (target != LF2MI_DEP_UNFOLDED && target != LF2MI_DEP_PERIODIC) return fail(LF2MI_EINVAL, "bad target %d", target);
    if (acc != LF2MI_ACC_NATIVE && acc != LF2MI_ACC_FIXED64) return fail(LF2MI_EINVAL, "bad accumulation mode %d", acc);
    if (overwrite && target != LF2MI_DEP_PERIODIC) return fail(LF2MI_EINVAL, "an overwriting deposit is periodic");
    hipStream_t st = as_stream(stream);
    const int N = p->N;
    const double nv = (double)N * N * N;
    if (overwrite) {
        // the field's previous contents are replaced: the FP32 tiles kernels store every
        // interior node, so only the ghosts need clearing; the other paths but the fixed-point
        // one add into a cleared field
        static const int comps[5] = {1, 3, 6, 3, 6};
        const int C = comps[kind];
        const int64_t G = N + 2 * halo;
        const bool f32 = p->dtype == LF2MI_F32;
        const bool pmass = p->mass_src && (f32 ? p->b32[p->cur].mass != nullptr : p->b64.mass != nullptr);
        const bool stores = f32 && acc == LF2MI_ACC_NATIVE && p->np > 0 &&
                            (tiles_path(p, kind, target, pmass) || tiles_c_path(p, kind, target, pmass));
        if (stores) {
            // (the scalar tiles clear the ghosts in their second launch)
            if (!tiles_path(p, kind, target, pmass) || halo > TILE_GHOSTS)
                if (int rc = zero_ghosts(field, N, halo, C, p->dtype, st)) return rc;
        } else if (f32 && acc == LF2MI_ACC_FIXED64 && p->np > 0) {
            // the fixed-point sums are taken to every node
        } else {
            if (int rc = lf2mi_zero(field, G * G * G * C, p->dtype, stream)) return rc;
            overwrite = false;
        }
    }
    if (p->np == 0) return LF2MI_OK;
    if (p->dtype == LF2MI_F64) {
        if (acc != LF2MI_ACC_NATIVE) return fail(LF2MI_EUNSUPPORTED, "fixed-point deposit is an F32 option");
        Dep64Args A{};
        A.s = p->b64;
        A.np = p->np;
        A.N = N;
        A.mass_nv = p->mass_global * nv;
        A.field = (double *)field;
        A.h = halo;
        A.tgt = target;
        if (p->mass_src && p->b64.mass) A.mass_nv = nv;
        else A.s.mass = nullptr;
        if (kind != LF2MI_PROJ_SCALAR)
            if (int rc = vector_source(p, p->b64.pl, A.s.vel, st)) return rc;
        const unsigned g = grid1(p->np);
        static const char *const names64[5] = {"deposit_f64_scalar", "deposit_f64_vector", "deposit_f64_vecvec",
                                               "deposit_f64_vector_ngp", "deposit_f64_symtensor_ngp"};
        LF2MI_PROF(names64[kind], st);
        if (b64_used(p)) {
            const BrickIndex V = brick_view(p->bb, N);
            const unsigned gb = (unsigned)brick_items(V.nbk, p->np);
            const int mg = merge_items(p->np, DEP_MERGE);
            switch (kind) {
                case 0: deposit_brick64_kernel<0><<<gb, bw_wg<0>(), 0, st>>>(A, V, mg); break;
                case 1: deposit_brick64_kernel<1><<<gb, bw_wg<1>(), 0, st>>>(A, V, mg); break;
                case 2: deposit_brick64_kernel<2><<<gb, bw_wg<2>(), 0, st>>>(A, V, mg); break;
                case 3: deposit_brick64_kernel<3><<<gb, bw_wg<3>(), 0, st>>>(A, V, mg); break;
                default: deposit_brick64_kernel<4><<<gb, bw_wg<4>(), 0, st>>>(A, V, mg); break;
            }
            LF2MI_LAUNCHED();
            return LF2MI_OK;
        }
        switch (kind) {
            case 0: deposit_f64_kernel<0><<<g, 256, 0, st>>>(A); break;
            case 1: deposit_f64_kernel<1><<<g, 256, 0, st>>>(A); break;
            case 2: deposit_f64_kernel<2><<<g, 256, 0, st>>>(A); break;
            case 3: deposit_f64_kernel<3><<<g, 256, 0, st>>>(A); break;
            default: deposit_f64_kernel<4><<<g, 256, 0, st>>>(A); break;
        }
        LF2MI_LAUNCHED();
        return LF2MI_OK;
    }
    DepArgs A{};
    A.s = p->b32[p->cur];
    A.start = p->bstart;
    A.istart = p->istart;
    A.item_bucket = p->item_bucket;
    A.g = p->g;
    // per-particle masses only when chosen (lf2mi_parts_mass_from)
    const bool pm = p->mass_src && A.s.mass;
    if (!pm) A.s.mass = nullptr;
    A.mass_nv = (float)(pm ? nv : p->mass_global * nv);
    if (kind != LF2MI_PROJ_SCALAR)
        if (int rc = vector_source(p, A.s.pl, A.s.vel, st)) return rc;
    A.field = (float *)field;
    A.h = halo;
    A.tgt = target;
    const unsigned g = (unsigned)item_grid(p);
    if (acc == LF2MI_ACC_FIXED64) {
        static const int comps[5] = {1, 3, 6, 3, 6};
        const int C = comps[kind];
        const int64_t G = N + 2 * halo;
        const int64_t n = G * G * G * C;
        if (p->fx_n < n) {
            if (p->fx) hipFree(p->fx);
            p->fx = nullptr;
            p->fx_n = 0;
            LF2MI_HIP(hipMalloc((void **)&p->fx, n * sizeof(unsigned long long)));
            p->fx_n = n;
            p->fx_used = 1;
            p->fx_halo = -1;
        }
        // a deposit leaves the buffer cleared, or, by the tiles, with the interior that the next
        // such deposit stores again; a captured one, which runs later and perhaps after one that
        // failed, clears it first and leaves it cleared
        const bool tiles = tiles_path(p, kind, target, pm);
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
        LF2MI_HIP(hipStreamIsCapturing(st, &cap));
        const bool captured = cap != hipStreamCaptureStatusNone;
        if (p->fx_used || captured || (p->fx_halo >= 0 && !(tiles && p->fx_halo == halo))) {
            fill_u64_kernel<<<(unsigned)std::min<int64_t>(grid1(p->fx_n), 65536), 256, 0, st>>>(p->fx, p->fx_n);
            LF2MI_LAUNCHED();
        }
        A.fx = p->fx;
        FxScales S{};
        if (kind == LF2MI_PROJ_SCALAR && !pm) {
            // one global mass: dimensionless weights in 2^-32 units
            const double mref = A.mass_nv;
            A.fxs[0] = 4294967296.0 / mref;
            S.inv[0] = mref / 4294967296.0;
        } else {
            // per component a power-of-two scale 2^(62 - e) with np max|q| max|v_a| max|v_b| < 2^e
            // (the scalar kind with per-particle masses: np max|q| < 2^e): no node (nor any
            // partial sum) can leave the int64 range, the quantum is 2^-62 of that bound, and
            // the integer sums do not depend on the order of the particles
            unsigned int *dmax = nullptr, hmax[4] = {0u, 0u, 0u, 0u};
            LF2MI_HIP(hipMallocAsync((void **)&dmax, 4 * sizeof(unsigned int), st));
            fill_int_kernel<<<1, 64, 0, st>>>(reinterpret_cast<int *>(dmax), 4, 0);
            dep_max_kernel<<<(unsigned)std::min<int64_t>(grid1(p->np), DMAX_BLOCKS), 256, 0, st>>>(p->np, A.s, A.mass_nv,
                                                                                          dmax);
            hipError_t e = hipGetLastError();
            if (e == hipSuccess) e = hipMemcpyAsync(hmax, dmax, sizeof hmax, hipMemcpyDeviceToHost, st);
            if (e == hipSuccess) e = hipStreamSynchronize(st);
            hipFreeAsync(dmax, st);
            if (e != hipSuccess) return hip_fail(e, "fixed-point bound", __FILE__, __LINE__);
            float mx[4];
            memcpy(mx, hmax, sizeof mx);
            static const int va[5][6] = {{-1}, {0, 1, 2}, {0, 0, 0, 1, 1, 2}, {0, 1, 2}, {0, 0, 0, 1, 1, 2}};
            static const int vb[5][6] = {{-1}, {-1, -1, -1}, {0, 1, 2, 1, 2, 2}, {-1, -1, -1}, {0, 1, 2, 1, 2, 2}};
            for (int c = 0; c < C; ++c) {
                double bound = (double)p->np * (double)mx[0];
                if (va[kind][c] >= 0) bound *= (double)mx[1 + va[kind][c]];
                if (vb[kind][c] >= 0) bound *= (double)mx[1 + vb[kind][c]];
                double sc = 1.0;
                if (bound > 0.0 && bound < 1e300) {
                    int ex;
                    frexp(bound, &ex);
                    sc = ldexp(1.0, 62 - ex);
                }
                A.fxs[c] = sc;
                S.inv[c] = 1.0 / sc;
            }
        }
        if (!captured) p->fx_used = 1;
        {
            static const char *const namesfx[5] = {"deposit_f32_fixed64", "deposit_f32_vector_fixed64",
                                                   "deposit_f32_vecvec_fixed64", "deposit_f32_vector_ngp_fixed64",
                                                   "deposit_f32_symtensor_ngp_fixed64"};
            LF2MI_PROF(namesfx[kind], st);
            if (tiles) {
                // the sums of the interior are stored
                if (int rc = launch_tiles_dense<unsigned long long>(p, A, true, false, st)) return rc;
            } else {
                switch (kind) {
                    case 0: launch_bricks<0, unsigned long long>(p, A, g, nullptr, nullptr, st); break;
                    case 1: launch_bricks<1, unsigned long long>(p, A, g, nullptr, nullptr, st); break;
                    case 2: launch_bricks<2, unsigned long long>(p, A, g, nullptr, nullptr, st); break;
                    case 3: launch_bricks<3, unsigned long long>(p, A, g, nullptr, nullptr, st); break;
                    default: launch_bricks<4, unsigned long long>(p, A, g, nullptr, nullptr, st); break;
                }
            }
            LF2MI_LAUNCHED();
        }
        {
            LF2MI_PROF("fixed_to_field", st);
            const unsigned gf = (unsigned)std::min<int64_t>(grid1(n, 256 * FX_PER), 65536);
            float *f = (float *)field;
            const int clear = captured || !tiles;
            if (C == 1 && overwrite) fixed_to_field_kernel<true><<<gf, 256, 0, st>>>(p->fx, f, n, clear, S.inv[0]);
            else if (C == 1) fixed_to_field_kernel<false><<<gf, 256, 0, st>>>(p->fx, f, n, clear, S.inv[0]);
            else if (overwrite) fixed_to_field_c_kernel<true><<<gf, 256, 0, st>>>(p->fx, f, n, C, clear, S);
            else fixed_to_field_c_kernel<false><<<gf, 256, 0, st>>>(p->fx, f, n, C, clear, S);
            LF2MI_LAUNCHED();
            if (!captured) {
                p->fx_used = 0;
                p->fx_halo = tiles ? halo : -1;
            }
        }
        return LF2MI_OK;
    }
    static const char *const names32[5] = {"deposit_f32_scalar", "deposit_f32_vector", "deposit_f32_vecvec",
                                           "deposit_f32_vector_ngp", "deposit_f32_symtensor_ngp"};
    LF2MI_PROF(names32[kind], st);
    if (tiles_path(p, kind, target, pm)) return launch_tiles_dense<float>(p, A, overwrite, overwrite && halo <= TILE_GHOSTS, st);
    if (tiles_c_path(p, kind, target, pm)) {
        switch (kind) {
            case 0: return launch_tiles_c<0>(p, A, pm, overwrite, st);
            case 1: return launch_tiles_c<1>(p, A, pm, overwrite, st);
            case 2: return launch_tiles_c<2>(p, A, pm, overwrite, st);
            case 3: return launch_tiles_c<3>(p, A, pm, overwrite, st);
            default: return launch_tiles_c<4>(p, A, pm, overwrite, st);
        }
    }
    switch (kind) {
        case 0: launch_bricks<0, float>(p, A, g, nullptr, nullptr, st); break;
        case 1: launch_bricks<1, float>(p, A, g, nullptr, nullptr, st); break;
        case 2: launch_bricks<2, float>(p, A, g, nullptr, nullptr, st); break;
        case 3: launch_bricks<3, float>(p, A, g, nullptr, nullptr, st); break;
        default: launch_bricks<4, float>(p, A, g, nullptr, nullptr, st); break;
    }
    LF2MI_LAUNCHED();
    return LF2MI_OK;
}

extern "C" {

int lf2mi_deposit(lf2mi_parts p, int kind, void *field, int halo, int target, int acc, void *stream) {
    if (target == LF2MI_DEP_PERIODIC_SET)
        return deposit_impl(p, kind, field, halo, LF2MI_DEP_PERIODIC, acc, true, stream);
    return deposit_impl(p, kind, field, halo, target, acc, false, stream);
}

int lf2mi_gather_kick_drift(lf2mi_parts p, const void *phi, int halo, double dt_kick, double dt_drift, double *vmax2,
                            void *stream) {
    if (!p || halo < 0) return fail(LF2MI_EINVAL, "lf2mi_gather_kick_drift: bad argument");
    if (!phi && dt_kick != 0.0) return fail(LF2MI_EINVAL, "lf2mi_gather_kick_drift: a kick needs the potential field");
    hipStream_t st = as_stream(stream);
    if (p->np == 0) {
        if (vmax2) *vmax2 = 0.0;
        return LF2MI_OK;
    }
    if (p->dtype == LF2MI_F64) {
        Gkd64Args A{};
        A.s = p->b64;
        A.np = p->np;
        A.N = p->N;
        A.h = halo;
        A.phi = (const double *)phi;
        A.dt_kick = dt_kick;
        A.dt_drift = dt_drift;
        A.vmax2 = vmax2 ? p->vmax_f64 : nullptr;
        // a kick alone leaves positions and cells as they are (in_box: none is due a wrap)
        A.drift = dt_drift != 0.0 || !p->in_box;
        const bool bricks = b64_used(p);
        const BrickIndex V = brick_view(p->bb, p->N);
        if (vmax2) LF2MI_HIP(hipMemsetAsync(p->vmax_f64, 0, sizeof(unsigned long long), st));
        {
            LF2MI_PROF("gkd_f64", st);
            if (bricks && phi) gkd_brick64_kernel<<<(unsigned)brick_items(V.nbk, p->np), 256, 0, st>>>(A, V, merge_items(p->np, G64_MERGE));
            else gkd_f64_kernel<<<grid1(p->np), 256, 0, st>>>(A);
            LF2MI_LAUNCHED();
        }
        if (A.drift) {
            unsigned long long cap_id;
            const bool captured = capturing(st, &cap_id);
            if (!captured) p->in_box = 1;  // a recorded drift has moved nothing yet
            if (bricks) {
                LF2MI_PROF("brick_index", st);
                if (int rc = b64_moved(p, captured, cap_id, st)) return rc;
            }
        }
        if (vmax2) {
            unsigned long long bits = 0;
            LF2MI_HIP(hipMemcpyAsync(&bits, p->vmax_f64, sizeof(bits), hipMemcpyDeviceToHost, st));
            LF2MI_HIP(hipStreamSynchronize(st));
            double v;
            memcpy(&v, &bits, sizeof(v));
            *vmax2 = v;
        }
        return LF2MI_OK;
    }
    GkdArgs A{};
    A.s = p->b32[p->cur];
    A.start = p->bstart;
    A.istart = p->istart;
    A.item_bucket = p->item_bucket;
    A.g = p->g;
    A.phi = (const float *)phi;
    A.h = halo;
    A.dt_kick = (float)dt_kick;
    A.dt_drift = dt_drift;
    A.next_counts = p->bcount;
    A.vmax2 = vmax2 ? p->vmax_f32 : nullptr;
    A.chunked = phi != nullptr;
    A.drift = dt_drift != 0.0;
    if (vmax2) LF2MI_HIP(hipMemsetAsync(p->vmax_f32, 0, sizeof(unsigned int), st));
    const bool b8 = p->g.B == 8;
    const unsigned items = (unsigned)item_grid(p);
    if (A.chunked && chunk_width(p) == 1) {
        LF2MI_PROF("gkd_f32", st);
        const unsigned grid = (unsigned)p->g.nbk + items;
        if (b8) gkd_small_kernel<8><<<grid, DEP_WG, 0, st>>>(A, p->chunks, p->nchunk);
        else gkd_small_kernel<0><<<grid, DEP_WG, 0, st>>>(A, p->chunks, p->nchunk);
        LF2MI_LAUNCHED();
    } else {
        {
            LF2MI_PROF("gkd_f32", st);
            if (b8) gkd_f32_kernel<8><<<items, DEP_WG, 0, st>>>(A);
            else gkd_f32_kernel<0><<<items, DEP_WG, 0, st>>>(A);
            LF2MI_LAUNCHED();
        }
        if (A.chunked) {
            // persistent: a few workgroups per CU walk the chunk list
            LF2MI_PROF("gkd_f32_chunks", st);
            const unsigned grid = (unsigned)std::min<int64_t>(p->g.nbk, 2048);
            if (b8) gkd_chunk_kernel<8><<<grid, DEP_WG, 0, st>>>(A, p->chunks, p->nchunk);
            else gkd_chunk_kernel<0><<<grid, DEP_WG, 0, st>>>(A, p->chunks, p->nchunk);
            LF2MI_LAUNCHED();
        }
    }
    // (the scan clears the claims)
    if (A.drift) {
        if (int rc = sort_into_other(p, p->cur, p->np, true, dt_drift, st)) return rc;
    } else if (A.chunked) {
        if (int rc = fill_int(p->nchunk + 1, 1, 0, st)) return rc;
    }
    if (vmax2) {
        unsigned int bits = 0;
        LF2MI_HIP(hipMemcpyAsync(&bits, p->vmax_f32, sizeof(bits), hipMemcpyDeviceToHost, st));
        LF2MI_HIP(hipStreamSynchronize(st));
        float v;
        memcpy(&v, &bits, sizeof(v));
        *vmax2 = v;
    }
    return LF2MI_OK;
}

int lf2mi_parts_reduce(lf2mi_parts p, int n, const int *quantity, const int *reduce_type, double *out, void *stream) {
    if (!p || n < 0 || n > RED_Q || (n > 0 && (!quantity || !reduce_type || !out)))
        return fail(LF2MI_EINVAL, "lf2mi_parts_reduce: bad argument (at most %d quantities)", RED_Q);
    if (n == 0) return LF2MI_OK;
    RedArgs A{};
    A.np = p->np;
    A.nq = n;
    for (int k = 0; k < RED_Q; ++k) {
        A.q[k] = 0;
        A.op[k] = RED_NONE;
    }
    for (int k = 0; k < n; ++k) {
        if (quantity[k] < LF2MI_PQ_V2 || quantity[k] > LF2MI_PQ_EKIN)
            return fail(LF2MI_EINVAL, "lf2mi_parts_reduce: unknown quantity %d", quantity[k]);
        const int rt = reduce_type[k];
        A.q[k] = quantity[k];
        A.op[k] = (rt & (LF2MI_RED_SUM | LF2MI_RED_SUM_LOCAL))   ? RED_OP_SUM
                  : (rt & (LF2MI_RED_MIN | LF2MI_RED_MIN_LOCAL)) ? RED_OP_MIN
                  : (rt & (LF2MI_RED_MAX | LF2MI_RED_MAX_LOCAL)) ? RED_OP_MAX
                                                                 : RED_NONE;
    }
    A.mass = p->mass_global;
    hipStream_t st = as_stream(stream);
    const int nb = (int)std::max<int64_t>(1, std::min<int64_t>(RED_BLOCKS, (p->np + RED_WG - 1) / RED_WG));
    double *res = p->red + (int64_t)RED_BLOCKS * RED_Q;
    LF2MI_PROF("parts_reduce", st);
    if (p->dtype == LF2MI_F32) {
        const Soa32 &s = p->b32[p->cur];
        for (int d = 0; d < 3; ++d) A.vel32[d] = s.vel[d];
        A.mass32 = p->mass_src ? s.mass : nullptr;
        parts_reduce_kernel<false><<<nb, RED_WG, 0, st>>>(A, p->red);
    } else {
        for (int d = 0; d < 3; ++d) A.vel64[d] = p->b64.vel[d];
        A.mass64 = p->mass_src ? p->b64.mass : nullptr;
        A.slot = p->sorted ? p->slot : nullptr;
        parts_reduce_kernel<true><<<nb, RED_WG, 0, st>>>(A, p->red);
    }
    LF2MI_LAUNCHED();
    parts_reduce_final_kernel<<<n, RED_WG, 0, st>>>(A, p->red, nb, res);
    LF2MI_LAUNCHED();
    double host[RED_Q];
    LF2MI_HIP(hipMemcpyAsync(host, res, sizeof(double) * n, hipMemcpyDeviceToHost, st));
    LF2MI_HIP(hipStreamSynchronize(st));
    for (int k = 0; k < n; ++k)
        if (A.op[k] != RED_NONE) out[k] = host[k];
    return LF2MI_OK;
}

int lf2mi_pm_step(lf2mi_parts p, lf2mi_fft_plan plan, void *rho, void *phi, int halo, double dt_kick, double dt_drift,
                  int acc, void *stream) {
    if (!p || !plan || !rho || !phi) return fail(LF2MI_EINVAL, "lf2mi_pm_step: null argument");
    const int N = p->N;
    // rho replaced by the deposit (the FP32 tiles kernels store its interior)
    if (int rc = deposit_impl(p, LF2MI_PROJ_SCALAR, rho, halo, LF2MI_DEP_PERIODIC, acc, true, stream)) return rc;
    // box volume 1: the mean density is the total mass
    const double scale = 1.0 / ((double)N * N * N);
    if (int rc = lf2mi_poisson_solve(plan, rho, phi, p->total_mass, scale, stream)) return rc;
    return lf2mi_gather_kick_drift(p, phi, halo, dt_kick, dt_drift, nullptr, stream);
}

}  // extern "C"
