// Differentiable PM on one gfx950 device: nsteps of a kick-drift leapfrog of the PM
// step, with hand-written adjoint kernels.  No counterpart in the reference; it
// differentiates the reference's forward pieces:
//   deposit  rho = sum_p q W(X - X_p), q = m N^3   (scalarProjectionCIC_project,
//            particles/projections.hpp:76-300, periodic)
//   Poisson  phi = G rho, G = -K^-2, zero mode 0   (examples/poissonSolver.cpp:99-111)
//   force    F_d = -D_d phi, D_d the central difference (N/2)(f(n+e_d) - f(n-e_d))
//   gather   a_p = sum_corners W F(corner)          (updateVel, Particles.hpp:825-828)
//   leapfrog v += dt a(x);  x += dt v, wrapped into the box (moveParticles)
//   loss     L = sum_cells (rho(x_final) - target)^2
// Adjoint (x in box units, X = x N in cell units; lambda_x = dL/dx, lambda_v = dL/dv):
//   final state          lambda_x = q N grad_X interp(2 (rho - target))(X_p)
//   per step, backwards  lambda_v += dt lambda_x;  mu = dt lambda_v
//                        lambda_x += N sum_d mu_d grad_X interp(F_d)(X_p)   (gather weights)
//                        F-bar_d = sum_p mu_{p,d} W(X - X_p)  (the gather's transpose is a deposit)
//                        phi-bar = sum_d D_d F-bar_d          (D_d is antisymmetric)
//                        rho-bar = G phi-bar                  (G is symmetric: the same FFT solve)
//                        lambda_x += q N grad_X interp(rho-bar)(X_p)   (deposit weights)
// A particle keeps its place in all states, so gradients stay attached to it; a brick index
// (bricks.hpp) of every state lets the deposits and gathers work brick by brick.  The starting
// state of every step is checkpointed in HBM, and so are its potential and its index (4 bytes
// beside a particle's 28 or 52) where the memory left over has room for them (spare_bytes); else
// these are computed again on the way back.  Positions are kept as (cell, offset in cell units)
// and re-anchored in FP64 after each drift, as in the PM step.  T = float or double selects the
// precision of the whole path (fields, FFTs, offsets, velocities, adjoints).
#include <algorithm>
#include <cmath>
#include <new>

#include "bricks.hpp"
#include "common.hpp"

namespace lf2mi {

namespace {

template <typename T> struct DpState {
    int N;
    int64_t np;
    int32_t *cell;
    T *off[3];
    T *vel[3];
};

constexpr int DP_WG = 256;

inline unsigned dp_grid(int64_t n) { return (unsigned)std::max<int64_t>(1, std::min<int64_t>((n + DP_WG - 1) / DP_WG, 1 << 16)); }

__device__ __forceinline__ int wrapn(int v, int N) { return v < 0 ? v + N : (v >= N ? v - N : v); }

__device__ __forceinline__ void decode(int cell, int N, int c[3]) {
    c[0] = cell % N;
    c[1] = (cell / N) % N;
    c[2] = cell / (N * N);
}

__device__ __forceinline__ double add_nc(double a, double b) {
#pragma clang fp contract(off)
    return a + b;
}
__device__ __forceinline__ double mul_nc(double a, double b) {
#pragma clang fp contract(off)
    return a * b;
}

template <typename T> __device__ __forceinline__ T below_one();
template <> __device__ __forceinline__ float below_one<float>() { return 0x1.fffffep-1f; }
template <> __device__ __forceinline__ double below_one<double>() { return 0x1.fffffffffffffp-1; }

// X (cell units, FP64) -> (cell, offset) with periodic wrap
template <typename T> __device__ __forceinline__ void anchor(double X, int N, int &c, T &o) {
    if (X < 0.0 || X >= (double)N) X -= (double)N * floor(X / (double)N);
    const double fl = floor(X);
    c = (int)fl;
    if (c >= N) c = N - 1;
    if (c < 0) c = 0;
    o = (T)(X - fl);
    if (!(o < (T)1)) o = below_one<T>();
}

template <typename T> __device__ __forceinline__ T wsel(int i, T u) { return i ? u : (T)1 - u; }

// clears up to two fields on the side of a launch that covers the chip: beside a small mesh the
// launches count (32^3: about 3 us each), beside a large one the clears hide behind the
// particles' latency
template <typename T> struct DpClear {
    T *a, *b;  // may be null
    int64_t n;
};
template <typename T> __device__ __forceinline__ void dp_clear(const DpClear<T> &c) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < c.n; i += stride) {
        if (c.a) c.a[i] = (T)0;
        if (c.b) c.b[i] = (T)0;
    }
}

// The states hold the particles in the brick order of the initial positions (slot[i]: the place
// of the caller's particle i): the particles move a few cells over a run, so the brick lists of
// every state read memory nearly in order, whatever order the caller's arrays have (128^3 FP32
// lattice, 10 steps: adjoint 86 -> 68 us a launch, density 41 -> 33; 64^3 in random order: the
// whole evaluation 7.0 -> 1.6 ms against particles in the caller's order with global atomics).
// Here: the initial cells and the particles' places in their bricks.
template <typename T, typename I>
__global__ __launch_bounds__(DP_WG) void dp_cells_kernel(int64_t np, const I *__restrict__ pos, int N, int NB,
                                                         int *__restrict__ count, int *__restrict__ rank, DpClear<T> clear,
                                                         double *__restrict__ loss) {
    const int64_t p = (int64_t)blockIdx.x * DP_WG + threadIdx.x;
    const bool in = p < np;
    int c[3] = {0, 0, 0};
    if (in)
        for (int d = 0; d < 3; ++d) {
            T o;
            anchor<T>(mul_nc((double)pos[3 * p + d], (double)N), N, c[d], o);
        }
    const int r = brick_rank(count, brick_of(c[0], c[1], c[2], NB), in);
    if (in) rank[p] = r;
    if (p == 0) *loss = 0.0;
    dp_clear(clear);
}

template <typename T, typename I>
__global__ void dp_init_kernel(DpState<T> s, const I *__restrict__ pos, const I *__restrict__ vel, int NB,
                               const int *__restrict__ start, const int *__restrict__ rank, int *__restrict__ slot,
                               int *__restrict__ list) {
    for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < s.np; p += (int64_t)gridDim.x * blockDim.x) {
        int c[3];
        T o[3];
        for (int d = 0; d < 3; ++d) anchor<T>(mul_nc((double)pos[3 * p + d], (double)s.N), s.N, c[d], o[d]);
        const int j = start[brick_of(c[0], c[1], c[2], NB)] + rank[p];
        slot[p] = j;
        list[j] = j;
        for (int d = 0; d < 3; ++d) {
            s.off[d][j] = o[d];
            s.vel[d][j] = vel ? (T)vel[3 * p + d] : (T)0;
        }
        s.cell[j] = c[0] + s.N * (c[1] + s.N * c[2]);
    }
}

template <typename T, typename I>
__global__ void dp_state_out_kernel(DpState<T> s, const int *__restrict__ slot, I *__restrict__ pos, I *__restrict__ vel) {
    for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < s.np; p += (int64_t)gridDim.x * blockDim.x) {
        const int64_t j = slot[p];
        int c[3];
        decode(s.cell[j], s.N, c);
        for (int d = 0; d < 3; ++d) {
            if (pos) pos[3 * p + d] = (I)(add_nc((double)c[d], (double)s.off[d][j]) / (double)s.N);
            if (vel) vel[3 * p + d] = (I)s.vel[d][j];
        }
    }
}

// ---- brick windows (bricks.hpp): one workgroup per group of items of a brick
static constexpr int DP_MERGE = 4;
static constexpr int DP_FW = BRK + 1, DP_F3 = DP_FW * DP_FW * DP_FW;  // nodes [o, o + 8]
static constexpr int DP_PW = BRK + 3, DP_P3 = DP_PW * DP_PW * DP_PW;  // nodes [o - 1, o + 9]

// density: the brick's terms q w summed in an FP64 window, its nodes added to rho (128^3 FP32
// particles in lattice order: 33 us; 390 us with 8 global atomics per particle)
template <typename T>
__global__ __launch_bounds__(DP_WG) void dp_density_kernel(DpState<T> s, BrickIndex V, T *__restrict__ rho, T q) {
    __shared__ double win[DP_F3];
    BrickRange r;
    if (!brick_range(V, blockIdx.x, DP_MERGE, r)) return;
    const int N = s.N;
    for (int i = threadIdx.x; i < DP_F3; i += DP_WG) win[i] = 0.0;
    __syncthreads();
    for (int j = threadIdx.x; j < r.n; j += DP_WG) {
        const int p = V.list[r.p0 + j];
        int c[3];
        brick_decode(s.cell[p], N, V.lgN, c[0], c[1], c[2]);
        const T u[3] = {s.off[0][p], s.off[1][p], s.off[2][p]};
        double *o = win + (c[0] - r.ox + DP_FW * (c[1] - r.oy + DP_FW * (c[2] - r.oz)));
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int j2 = 0; j2 < 2; ++j2)
#pragma unroll
                for (int i = 0; i < 2; ++i)
                    lds_add(&o[i + DP_FW * (j2 + DP_FW * k)], (double)(q * (wsel(i, u[0]) * wsel(j2, u[1]) * wsel(k, u[2]))));
    }
    __syncthreads();
    for (int i = threadIdx.x; i < DP_F3; i += DP_WG) {
        const double w = win[i];
        if (w == 0.0) continue;
        const int x = r.ox + i % DP_FW, y = r.oy + (i / DP_FW) % DP_FW, z = r.oz + i / (DP_FW * DP_FW);
        atomicAdd(&rho[site_index(N, 1, wrapn(x, N), wrapn(y, N), wrapn(z, N))], (T)w);
    }
}

// the brick's window of phi into LDS (every load issued before the stores), then the force
// F = -D phi on its nodes; barriers inside
template <typename T>
__device__ __forceinline__ void brick_forces(const T *__restrict__ phi, int N, const BrickRange &r, T *__restrict__ phw,
                                             T (*__restrict__ frc)[DP_F3]) {
    constexpr int WK = (DP_P3 + DP_WG - 1) / DP_WG;
    T w[WK];
#pragma unroll
    for (int k = 0; k < WK; ++k) {
        const int i = threadIdx.x + DP_WG * k;
        if (i < DP_P3)
            w[k] = phi[site_index(N, 1, wrapn(r.ox - 1 + i % DP_PW, N), wrapn(r.oy - 1 + (i / DP_PW) % DP_PW, N),
                                  wrapn(r.oz - 1 + i / (DP_PW * DP_PW), N))];
    }
#pragma unroll
    for (int k = 0; k < WK; ++k) {
        const int i = threadIdx.x + DP_WG * k;
        if (i < DP_P3) phw[i] = w[k];
    }
    __syncthreads();
    const T hn = (T)0.5 * (T)N;
    for (int i = threadIdx.x; i < DP_F3; i += DP_WG) {
        const int c = i % DP_FW + 1 + DP_PW * ((i / DP_FW) % DP_FW + 1 + DP_PW * (i / (DP_FW * DP_FW) + 1));
        frc[0][i] = -(phw[c + 1] - phw[c - 1]) * hn;
        frc[1][i] = -(phw[c + DP_PW] - phw[c - DP_PW]) * hn;
        frc[2][i] = -(phw[c + DP_PW * DP_PW] - phw[c - DP_PW * DP_PW]) * hn;
    }
    __syncthreads();
}

// v += dt a(X); X += dt N v; re-anchor: state s -> state t (the particles keep their numbers)
template <typename T>
__global__ __launch_bounds__(DP_WG) void dp_step_kernel(DpState<T> s, DpState<T> t, BrickIndex V,
                                                        const T *__restrict__ phi, T dt, DpClear<T> clear) {
    __shared__ T phw[DP_P3];
    __shared__ T frc[3][DP_F3];
    dp_clear(clear);
    BrickRange r;
    if (!brick_range(V, blockIdx.x, DP_MERGE, r)) return;
    const int N = s.N;
    brick_forces(phi, N, r, phw, frc);
    for (int j = threadIdx.x; j < r.n; j += DP_WG) {
        const int p = V.list[r.p0 + j];
        int c[3];
        brick_decode(s.cell[p], N, V.lgN, c[0], c[1], c[2]);
        const T u[3] = {s.off[0][p], s.off[1][p], s.off[2][p]};
        const T vin[3] = {s.vel[0][p], s.vel[1][p], s.vel[2][p]};
        const int o = c[0] - r.ox + DP_FW * (c[1] - r.oy + DP_FW * (c[2] - r.oz));
        T a[3] = {(T)0, (T)0, (T)0};
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int j2 = 0; j2 < 2; ++j2)
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const T w = wsel(i, u[0]) * wsel(j2, u[1]) * wsel(k, u[2]);
#pragma unroll
                    for (int d = 0; d < 3; ++d) a[d] += w * frc[d][o + i + DP_FW * (j2 + DP_FW * k)];
                }
        int cn[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const T v = vin[d] + dt * a[d];
            t.vel[d][p] = v;
            const double X = add_nc(add_nc((double)c[d], (double)u[d]), mul_nc(mul_nc((double)dt, (double)v), (double)N));
            T on;
            anchor<T>(X, N, cn[d], on);
            t.off[d][p] = on;
        }
        t.cell[p] = cn[0] + N * (cn[1] + N * cn[2]);
    }
}

// resid = 2 (rho - target) on the interior; loss += sum (rho - target)^2 in FP64;
// rho_out (x fastest, may be null) receives the interior of rho
template <typename T, typename I>
__global__ void dp_resid_kernel(const T *__restrict__ rho, const I *__restrict__ target, T *__restrict__ resid,
                                I *__restrict__ rho_out, int N, double *__restrict__ loss) {
    __shared__ double red[DP_WG];
    const int64_t n = (int64_t)N * N * N;
    double acc = 0.0;
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (int64_t)gridDim.x * blockDim.x) {
        const int x = (int)(t % N), y = (int)((t / N) % N), z = (int)(t / ((int64_t)N * N));
        const int64_t i = site_index(N, 1, x, y, z);
        const T r = rho[i] - (target ? (T)target[t] : (T)0);
        resid[i] = (T)2 * r;
        if (rho_out) rho_out[t] = (I)rho[i];
        acc += (double)r * (double)r;
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int o = DP_WG / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) atomicAdd(loss, red[0]);
}

// gradient (per cell unit) of the CIC interpolant of g at (c, u)
template <typename T>
__device__ __forceinline__ void interp_grad(const T *__restrict__ g, int N, const int c[3], const T u[3], T gr[3]) {
    gr[0] = gr[1] = gr[2] = (T)0;
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const T v = g[site_index(N, 1, wrapn(c[0] + i, N), wrapn(c[1] + j, N), wrapn(c[2] + k, N))];
                const T wx = wsel(i, u[0]), wy = wsel(j, u[1]), wz = wsel(k, u[2]);
                gr[0] += (i ? v : -v) * wy * wz;
                gr[1] += wx * (j ? v : -v) * wz;
                gr[2] += wx * wy * (k ? v : -v);
            }
}

// lambda_x (AoS, np*3) = (init ? 0 : lambda_x) + qN grad_X interp(g); init: lambda_v = 0 too
template <typename T>
__global__ void dp_pos_grad_kernel(DpState<T> s, const T *__restrict__ g, T qN, T *__restrict__ lx, T *__restrict__ lv,
                                   int init, DpClear<T> clear) {
    for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < s.np; p += (int64_t)gridDim.x * blockDim.x) {
        int c[3];
        decode(s.cell[p], s.N, c);
        const T u[3] = {s.off[0][p], s.off[1][p], s.off[2][p]};
        T gr[3];
        interp_grad(g, s.N, c, u, gr);
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            lx[3 * p + d] = (init ? (T)0 : lx[3 * p + d]) + qN * gr[d];
            if (init) lv[3 * p + d] = (T)0;
        }
    }
    dp_clear(clear);
}

// One backward step's particle part, and phi-bar = sum_d D_d F-bar_d with
// F-bar_d = sum_p mu_d W: F-bar is summed per brick in three FP64 LDS windows and its
// differences are formed there, so that a brick adds one value to each node of its
// [o - 1, o + 9] window of phi-bar instead of 24 terms per particle to a three-component
// field (128^3 FP32 particles: 68 us; 1960 us with global atomics, and a pass over the field for
// the differences).
template <typename T>
__global__ __launch_bounds__(DP_WG) void dp_adj_kernel(DpState<T> s, BrickIndex V, const T *__restrict__ phi, T dt,
                                                       T *__restrict__ lx, T *__restrict__ lv, T *__restrict__ phib) {
    __shared__ T frc[3][DP_F3];
    __shared__ double fb[3][DP_F3];  // the window of phi before
    static_assert(sizeof(double) * 3 * DP_F3 >= sizeof(T) * DP_P3, "the window of phi fits");
    BrickRange r;
    if (!brick_range(V, blockIdx.x, DP_MERGE, r)) return;
    const int N = s.N;
    brick_forces(phi, N, r, reinterpret_cast<T *>(&fb[0][0]), frc);
    for (int i = threadIdx.x; i < 3 * DP_F3; i += DP_WG) (&fb[0][0])[i] = 0.0;
    __syncthreads();
    for (int j = threadIdx.x; j < r.n; j += DP_WG) {
        const int p = V.list[r.p0 + j];
        int c[3];
        brick_decode(s.cell[p], N, V.lgN, c[0], c[1], c[2]);
        const T u[3] = {s.off[0][p], s.off[1][p], s.off[2][p]};
        T mu[3], l[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            l[d] = lx[3 * (int64_t)p + d];
            const T v = lv[3 * (int64_t)p + d] + dt * l[d];
            lv[3 * (int64_t)p + d] = v;
            mu[d] = dt * v;
        }
        const int o = c[0] - r.ox + DP_FW * (c[1] - r.oy + DP_FW * (c[2] - r.oz));
        T add[3] = {(T)0, (T)0, (T)0};
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int j2 = 0; j2 < 2; ++j2)
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const int n = o + i + DP_FW * (j2 + DP_FW * k);
                    const T wx = wsel(i, u[0]), wy = wsel(j2, u[1]), wz = wsel(k, u[2]);
                    const T mf = mu[0] * frc[0][n] + mu[1] * frc[1][n] + mu[2] * frc[2][n];
                    add[0] += (i ? mf : -mf) * wy * wz;
                    add[1] += wx * (j2 ? mf : -mf) * wz;
                    add[2] += wx * wy * (k ? mf : -mf);
                    const T w = wx * wy * wz;
#pragma unroll
                    for (int d = 0; d < 3; ++d) lds_add(&fb[d][n], (double)(mu[d] * w));
                }
#pragma unroll
        for (int d = 0; d < 3; ++d) lx[3 * (int64_t)p + d] = l[d] + (T)N * add[d];
    }
    __syncthreads();
    const double hn = 0.5 * (double)N;
    for (int i = threadIdx.x; i < DP_P3; i += DP_WG) {
        const int x = i % DP_PW - 1, y = (i / DP_PW) % DP_PW - 1, z = i / (DP_PW * DP_PW) - 1;
        auto F = [&](int d, int xx, int yy, int zz) {
            const bool in = xx >= 0 && xx < DP_FW && yy >= 0 && yy < DP_FW && zz >= 0 && zz < DP_FW;
            return in ? fb[d][xx + DP_FW * (yy + DP_FW * zz)] : 0.0;
        };
        const double w = (F(0, x + 1, y, z) - F(0, x - 1, y, z)) + (F(1, x, y + 1, z) - F(1, x, y - 1, z)) +
                         (F(2, x, y, z + 1) - F(2, x, y, z - 1));
        if (w == 0.0) continue;
        atomicAdd(&phib[site_index(N, 1, wrapn(r.ox + x, N), wrapn(r.oy + y, N), wrapn(r.oz + z, N))], (T)(w * hn));
    }
}

// the adjoints in the caller's order (gv may be null)
template <typename T, typename I>
__global__ void dp_grad_out_kernel(int64_t np, const int *__restrict__ slot, const T *__restrict__ lx,
                                   const T *__restrict__ lv, I *__restrict__ gp, I *__restrict__ gv) {
    for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < np; p += (int64_t)gridDim.x * blockDim.x) {
        const int64_t j = slot[p];
        for (int d = 0; d < 3; ++d) {
            gp[3 * p + d] = (I)lx[3 * j + d];
            if (gv) gv[3 * p + d] = (I)lv[3 * j + d];
        }
    }
}

}  // namespace
}  // namespace lf2mi

struct lf2mi_diffpm_s {
    int N, nsteps, dtype, io_dtype;
    int64_t np, G3;
    double mass, dt;
    lf2mi_fft_plan plan;
    size_t tsize;   // sizeof(T)
    void *ck_mem;   // nsteps + 1 particle states (cell, off[3], vel[3])
    void *rho, *phi, *resid, *phib, *rhob;  // (N+2)^3 fields of T
    void *index_mem;  // the first state's brick index, scratch of the builds, slots
    size_t index_bytes;
    lf2mi::BrickBuild bricks;  // index of the first state
    int64_t index_ints;        // size of one index
    // kept for the way back where there is room, else null: the potentials of the steps after the
    // first, then an index for each state after the first.  Without it the states share the first
    // index and one potential, and both are made again on the way back.
    char *phi_kept;
    int *index_more;
    size_t kept_bytes;
    int *slot;        // place of the caller's particles in the states
    void *lx, *lv;  // adjoints, np*3 of T
    double *loss_dev;
    bool forward_done;
};

namespace lf2mi {
namespace {

size_t dp_state_bytes(int64_t np, size_t tsize) { return (((size_t)np * 4 + 255) & ~(size_t)255) + (size_t)np * 6 * tsize; }

template <typename T> DpState<T> dp_view(const lf2mi_diffpm_s *m, int k) {
    char *base = (char *)m->ck_mem + dp_state_bytes(m->np, sizeof(T)) * (size_t)k;
    DpState<T> s;
    s.N = m->N;
    s.np = m->np;
    s.cell = (int32_t *)base;
    T *f = (T *)(base + (((size_t)m->np * 4 + 255) & ~(size_t)255));
    for (int d = 0; d < 3; ++d) s.off[d] = f + d * m->np;
    for (int d = 0; d < 3; ++d) s.vel[d] = f + (3 + d) * m->np;
    return s;
}

int dp_malloc(void **p, size_t bytes) {
    *p = nullptr;
    hipError_t e = hipMalloc(p, bytes);
    if (e != hipSuccess) {
        *p = nullptr;
        return hip_fail(e, "hipMalloc(diffpm)", __FILE__, __LINE__);
    }
    return LF2MI_OK;
}

// the arrays of state k's brick index
BrickBuild dp_index(const lf2mi_diffpm_s *m, int k) {
    BrickBuild B = m->bricks;
    if (k > 0 && m->index_more) {
        int *q = m->index_more + (int64_t)(k - 1) * m->index_ints;
        const int *q0 = m->bricks.start;  // the first index is in one piece, in the same order
        B.start = q;
        B.istart = q + (m->bricks.istart - q0);
        B.item = q + (m->bricks.item - q0);
        B.list = q + (m->bricks.list - q0);
    }
    return B;
}

// the potential of step k
template <typename T> T *dp_phi(const lf2mi_diffpm_s *m, int k) {
    return k > 0 && m->phi_kept ? (T *)m->phi_kept + (size_t)(k - 1) * m->G3 : (T *)m->phi;
}

unsigned dp_bricks_grid(const lf2mi_diffpm_s *m) {
    const int64_t nb = (m->N + BRK - 1) / BRK;
    return (unsigned)brick_items(nb * nb * nb, m->np);
}

// a thread per particle, and enough to clear fields beside few particles
unsigned dp_clear_grid(const lf2mi_diffpm_s *m) {
    return std::max(blocks_for(m->np, DP_WG), std::min(blocks_for(m->G3, DP_WG), 2048u));
}

// density of state k, whose brick index is at hand, in m->rho (cleared before)
template <typename T> int dp_density(lf2mi_diffpm_s *m, int k, hipStream_t st) {
    const double n3 = (double)m->N * m->N * m->N;
    dp_density_kernel<T><<<dp_bricks_grid(m), DP_WG, 0, st>>>(dp_view<T>(m, k), brick_view(dp_index(m, k), m->N),
                                                              (T *)m->rho, (T)(m->mass * n3));
    LF2MI_LAUNCHED();
    return LF2MI_OK;
}

// density and potential of state k
template <typename T> int dp_potential(lf2mi_diffpm_s *m, int k, hipStream_t st) {
    if (int rc = dp_density<T>(m, k, st)) return rc;
    const double n3 = (double)m->N * m->N * m->N;
    return lf2mi_poisson_solve(m->plan, m->rho, dp_phi<T>(m, k), m->mass * (double)m->np, 1.0 / n3, st);
}

template <typename T, typename I>
int dp_forward(lf2mi_diffpm_s *m, const I *pos0, const I *vel0, const I *target, I *rho_out, double *loss, hipStream_t st) {
    const int N = m->N, NB = (N + BRK - 1) / BRK;
    const DpClear<T> clear_rho{(T *)m->rho, nullptr, m->G3};
    dp_cells_kernel<T, I><<<dp_clear_grid(m), DP_WG, 0, st>>>(m->np, pos0, N, NB, m->bricks.count, m->bricks.rank,
                                                              clear_rho, m->loss_dev);
    LF2MI_LAUNCHED();
    if (int rc = brick_scan(m->bricks.scan(), NB * NB * NB, st)) return rc;
    dp_init_kernel<T, I><<<dp_grid(m->np), DP_WG, 0, st>>>(dp_view<T>(m, 0), pos0, vel0, NB, m->bricks.start,
                                                           m->bricks.rank, m->slot, m->bricks.list);
    LF2MI_LAUNCHED();
    for (int s = 0; s < m->nsteps; ++s) {
        const DpState<T> xs = dp_view<T>(m, s), xn = dp_view<T>(m, s + 1);
        if (int rc = dp_potential<T>(m, s, st)) return rc;
        dp_step_kernel<T><<<dp_bricks_grid(m), DP_WG, 0, st>>>(xs, xn, brick_view(dp_index(m, s), N),
                                                               dp_phi<T>(m, s), (T)m->dt, clear_rho);
        LF2MI_LAUNCHED();
        if (int rc = brick_build(xn.cell, m->np, N, dp_index(m, s + 1), st)) return rc;
    }
    if (int rc = dp_density<T>(m, m->nsteps, st)) return rc;
    const double n3 = (double)N * N * N;
    dp_resid_kernel<T, I><<<std::min<unsigned>(dp_grid((int64_t)n3), 1024), DP_WG, 0, st>>>(
        (const T *)m->rho, target, (T *)m->resid, rho_out, N, m->loss_dev);
    LF2MI_LAUNCHED();
    if (loss) {
        LF2MI_HIP(hipMemcpyAsync(loss, m->loss_dev, sizeof(double), hipMemcpyDeviceToHost, st));
        LF2MI_HIP(hipStreamSynchronize(st));
    }
    return LF2MI_OK;
}

template <typename T, typename I> int dp_backward(lf2mi_diffpm_s *m, I *grad_pos, I *grad_vel, hipStream_t st) {
    const double n3 = (double)m->N * m->N * m->N;
    const T qN = (T)(m->mass * n3 * m->N);
    T *lx = (T *)m->lx, *lv = (T *)m->lv;
    const DpClear<T> clear{m->phi_kept ? nullptr : (T *)m->rho, (T *)m->phib, m->G3};
    dp_pos_grad_kernel<T><<<dp_clear_grid(m), DP_WG, 0, st>>>(dp_view<T>(m, m->nsteps), (const T *)m->resid, qN, lx, lv, 1,
                                                            clear);
    LF2MI_LAUNCHED();
    for (int s = m->nsteps - 1; s >= 0; --s) {
        const DpState<T> xs = dp_view<T>(m, s);
        if (!m->phi_kept) {  // nor its index
            if (int rc = brick_build(xs.cell, m->np, m->N, m->bricks, st)) return rc;
            if (int rc = dp_potential<T>(m, s, st)) return rc;
        }
        dp_adj_kernel<T><<<dp_bricks_grid(m), DP_WG, 0, st>>>(xs, brick_view(dp_index(m, s), m->N), dp_phi<T>(m, s),
                                                              (T)m->dt, lx, lv, (T *)m->phib);
        LF2MI_LAUNCHED();
        if (int rc = lf2mi_poisson_solve(m->plan, m->phib, m->rhob, 0.0, 1.0 / n3, st)) return rc;
        dp_pos_grad_kernel<T><<<dp_clear_grid(m), DP_WG, 0, st>>>(xs, (const T *)m->rhob, qN, lx, lv, 0, clear);
        LF2MI_LAUNCHED();
    }
    dp_grad_out_kernel<T, I><<<dp_grid(m->np), DP_WG, 0, st>>>(m->np, m->slot, lx, lv, grad_pos, grad_vel);
    LF2MI_LAUNCHED();
    return LF2MI_OK;
}

template <typename T, typename I> int dp_state(lf2mi_diffpm_s *m, int step, I *pos, I *vel, hipStream_t st) {
    dp_state_out_kernel<T, I><<<dp_grid(m->np), DP_WG, 0, st>>>(dp_view<T>(m, step), m->slot, pos, vel);
    LF2MI_LAUNCHED();
    return LF2MI_OK;
}

}  // namespace
}  // namespace lf2mi

using namespace lf2mi;

extern "C" {

int lf2mi_diffpm_bytes(lf2mi_diffpm m, int64_t *bytes) {
    if (!m || !bytes) return fail(LF2MI_EINVAL, "lf2mi_diffpm_bytes: null argument");
    int64_t fft = 0;
    if (int rc = lf2mi_fft_plan_bytes(m->plan, &fft)) return rc;
    *bytes = (int64_t)(dp_state_bytes(m->np, m->tsize) * (size_t)(m->nsteps + 1) + 5 * (size_t)m->G3 * m->tsize + m->index_bytes +
                       m->kept_bytes + 6 * (size_t)m->np * m->tsize + sizeof(double)) + fft;
    return LF2MI_OK;
}

int lf2mi_diffpm_create(int N, int64_t np, int nsteps, double mass, double dt, int dtype, lf2mi_diffpm *out) {
    return lf2mi_diffpm_create_keep(N, np, nsteps, mass, dt, dtype, -1, out);
}

int lf2mi_diffpm_create_keep(int N, int64_t np, int nsteps, double mass, double dt, int dtype, int64_t keep_bytes,
                             lf2mi_diffpm *out) {
    if (!out) return fail(LF2MI_EINVAL, "lf2mi_diffpm_create: null output");
    *out = nullptr;
    if (N < 8 || !is_pow2(N) || np < 1 || np > INT32_MAX || nsteps < 0 || !(mass > 0) || !std::isfinite(dt))
        return fail(LF2MI_EINVAL, "lf2mi_diffpm_create: bad argument (N=%d np=%lld nsteps=%d)", N, (long long)np, nsteps);
    if (dtype != LF2MI_F32 && dtype != LF2MI_F64) return fail(LF2MI_EINVAL, "lf2mi_diffpm_create: dtype must be F32 or F64");
    lf2mi_diffpm_s *m = new (std::nothrow) lf2mi_diffpm_s();
    if (!m) return fail(LF2MI_ENOMEM, "host allocation failed");
    m->N = N;
    m->np = np;
    m->nsteps = nsteps;
    m->mass = mass;
    m->dt = dt;
    m->dtype = dtype;
    m->tsize = dtype == LF2MI_F32 ? 4 : 8;
    m->G3 = (int64_t)(N + 2) * (N + 2) * (N + 2);
    const size_t fb = (size_t)m->G3 * m->tsize;
    int rc = lf2mi_fft_plan_create(N, 1, 1, 0, dtype, &m->plan);
    if (!rc) rc = dp_malloc(&m->ck_mem, dp_state_bytes(np, m->tsize) * (size_t)(nsteps + 1));
    if (!rc) rc = dp_malloc(&m->rho, fb);
    if (!rc) rc = dp_malloc(&m->phi, fb);
    if (!rc) rc = dp_malloc(&m->resid, fb);
    const int64_t nb = (N + BRK - 1) / BRK, nbk = nb * nb * nb, items = brick_items(nbk, np);
    // an index: starts, item starts, items, list; once: counts, block totals, ranks, slots
    m->index_ints = 2 * (nbk + 1) + items + np;
    m->index_bytes = sizeof(int) * (size_t)(m->index_ints + nbk + 3 * brick_blocks(nbk) + 2 * np);
    if (!rc) rc = dp_malloc(&m->index_mem, m->index_bytes);
    if (!rc) {
        int *q = (int *)m->index_mem;
        auto take = [&q](int64_t n) {
            int *r = q;
            q += n;
            return r;
        };
        m->bricks.start = take(nbk + 1);
        m->bricks.istart = take(nbk + 1);
        m->bricks.item = take(items);
        m->bricks.list = take(np);
        m->bricks.count = take(nbk);
        m->bricks.bsum = take(3 * brick_blocks(nbk));
        m->bricks.rank = take(np);
        m->slot = take(np);
        hipError_t e = hipMemset(m->bricks.count, 0, sizeof(int) * (size_t)nbk);
        if (e != hipSuccess) rc = hip_fail(e, "hipMemset(diffpm)", __FILE__, __LINE__);
    }
    if (!rc) rc = dp_malloc(&m->phib, fb);
    if (!rc) rc = dp_malloc(&m->rhob, fb);
    if (!rc) rc = dp_malloc(&m->lx, (size_t)np * 3 * m->tsize);
    if (!rc) rc = dp_malloc(&m->lv, (size_t)np * 3 * m->tsize);
    if (!rc) rc = dp_malloc((void **)&m->loss_dev, sizeof(double));
    if (!rc) {
        // the ghosts of these fields are never written by the kernels here; keep them defined
        for (void *p : {m->rho, m->phi, m->resid, m->phib, m->rhob}) {
            hipError_t e = hipMemset(p, 0, fb);
            if (e != hipSuccess) {
                rc = hip_fail(e, "hipMemset(diffpm)", __FILE__, __LINE__);
                break;
            }
        }
    }
    if (!rc && nsteps > 0) {
        // last, so that nothing the model needs can fail for it
        const size_t phis = fb * (size_t)(nsteps - 1);
        const size_t kept = phis + sizeof(int) * (size_t)m->index_ints * (size_t)nsteps;
        void *p = nullptr;
        if (kept <= (keep_bytes < 0 ? spare_bytes() : (size_t)keep_bytes)) {
            if (hipMalloc(&p, kept) == hipSuccess) {
                m->phi_kept = (char *)p;
                m->index_more = (int *)((char *)p + phis);
                m->kept_bytes = kept;
            } else {
                (void)hipGetLastError();
            }
        }
    }
    if (rc) {
        lf2mi_diffpm_destroy(m);
        return rc;
    }
    // the counters have to be clear before the first use, which may be on a stream that does not wait
    // for this one
    (void)hipStreamSynchronize(nullptr);
    *out = m;
    return LF2MI_OK;
}

int lf2mi_diffpm_destroy(lf2mi_diffpm m) {
    if (!m) return LF2MI_OK;
    if (m->plan) lf2mi_fft_plan_destroy(m->plan);
    for (void *p : {m->ck_mem, m->index_mem, (void *)m->phi_kept, m->rho, m->phi, m->resid, m->phib, m->rhob, m->lx, m->lv, (void *)m->loss_dev})
        if (p) (void)hipFree(p);
    delete m;
    return LF2MI_OK;
}

int lf2mi_diffpm_forward(lf2mi_diffpm m, const void *pos0, const void *vel0, const void *target, int io_dtype,
                         void *rho_out, double *loss, void *stream) {
    if (!m || !pos0) return fail(LF2MI_EINVAL, "lf2mi_diffpm_forward: null argument");
    if (io_dtype != LF2MI_F32 && io_dtype != LF2MI_F64) return fail(LF2MI_EINVAL, "lf2mi_diffpm_forward: io dtype must be F32 or F64");
    hipStream_t st = as_stream(stream);
    LF2MI_PROF("diffpm_forward", st);
    m->forward_done = false;
    int rc;
    if (m->dtype == LF2MI_F32) {
        if (io_dtype == LF2MI_F32)
            rc = dp_forward<float, float>(m, (const float *)pos0, (const float *)vel0, (const float *)target, (float *)rho_out, loss, st);
        else
            rc = dp_forward<float, double>(m, (const double *)pos0, (const double *)vel0, (const double *)target, (double *)rho_out, loss, st);
    } else {
        if (io_dtype == LF2MI_F32)
            rc = dp_forward<double, float>(m, (const float *)pos0, (const float *)vel0, (const float *)target, (float *)rho_out, loss, st);
        else
            rc = dp_forward<double, double>(m, (const double *)pos0, (const double *)vel0, (const double *)target, (double *)rho_out, loss, st);
    }
    if (rc) return rc;
    m->io_dtype = io_dtype;
    m->forward_done = true;
    return LF2MI_OK;
}

int lf2mi_diffpm_backward(lf2mi_diffpm m, void *grad_pos, void *grad_vel, void *stream) {
    if (!m || !grad_pos) return fail(LF2MI_EINVAL, "lf2mi_diffpm_backward: null argument");
    if (!m->forward_done) return fail(LF2MI_EINVAL, "lf2mi_diffpm_backward: no forward pass to differentiate");
    hipStream_t st = as_stream(stream);
    LF2MI_PROF("diffpm_backward", st);
    if (m->dtype == LF2MI_F32)
        return m->io_dtype == LF2MI_F32 ? dp_backward<float, float>(m, (float *)grad_pos, (float *)grad_vel, st)
                                        : dp_backward<float, double>(m, (double *)grad_pos, (double *)grad_vel, st);
    return m->io_dtype == LF2MI_F32 ? dp_backward<double, float>(m, (float *)grad_pos, (float *)grad_vel, st)
                                    : dp_backward<double, double>(m, (double *)grad_pos, (double *)grad_vel, st);
}

int lf2mi_diffpm_state(lf2mi_diffpm m, int step, void *pos, void *vel, int io_dtype, void *stream) {
    if (!m || (!pos && !vel)) return fail(LF2MI_EINVAL, "lf2mi_diffpm_state: null argument");
    if (!m->forward_done) return fail(LF2MI_EINVAL, "lf2mi_diffpm_state: no forward pass");
    if (step < 0 || step > m->nsteps) return fail(LF2MI_ERANGE, "lf2mi_diffpm_state: step %d outside [0, %d]", step, m->nsteps);
    if (io_dtype != LF2MI_F32 && io_dtype != LF2MI_F64) return fail(LF2MI_EINVAL, "lf2mi_diffpm_state: io dtype must be F32 or F64");
    hipStream_t st = as_stream(stream);
    if (m->dtype == LF2MI_F32)
        return io_dtype == LF2MI_F32 ? dp_state<float, float>(m, step, (float *)pos, (float *)vel, st)
                                     : dp_state<float, double>(m, step, (double *)pos, (double *)vel, st);
    return io_dtype == LF2MI_F32 ? dp_state<double, float>(m, step, (float *)pos, (float *)vel, st)
                                 : dp_state<double, double>(m, step, (double *)pos, (double *)vel, st);
}

}  // extern "C"
