// Dimensionally split sweep kernels, generic over the physics P.
//
// Data layout: structure-of-arrays primitive planes in HBM, plane f of cell
// (i, j) at in[f * plane + i * nx + j], x (j) contiguous.  No ghost cells are
// stored: the transmissive/periodic ghosts of the reference's
// insertBoundaryCells[2D] (Solvers/solvers.cpp:7-143) are produced by index
// mapping at load time (ghost_index).
//
// X sweep: one thread per cell along a row, tiles of BS cells overlapping by the
// stencil halo; neighbour states and face fluxes are exchanged through LDS so
// that each face flux is computed once (the reference computes it once per
// adjacent cell, secondordersolver.cpp:90-93; both evaluations are identical).
// Y sweep: one thread per column, sliding down H rows with the stencil window in
// registers -- every load is a coalesced row segment, no LDS and no barriers.
// The last sweep of a step can fold the next step's CFL wave-speed maximum into
// its stores (fuse_max).
#pragma once

#include "vg_device.h"
#include "vg_scheme.h"

namespace vg {

template <class P>
struct SweepArgs {
    const double *in;
    double *out;
    long long plane;
    int ny, nx;
    int bc, limiter;
    double dx, bias;
    double dt_scale;   // 0.5 for the half-step X sweeps of the 2D split, else 1
    int dim;           // 1 or 2: selects the wave-speed formula of the fused max
    int fuse_max;
    typename P::Params m;
    Clock *clk;
    unsigned long long *partials;   // one wave-speed key per block when fuse_max
    int fixed_params = 0;           // keep m as given (a per-sweep call): no per-step parameters from the clock
};

// Per-step scalars, computed identically in every thread.
struct StepScalars {
    double half_c, lf_c, ri_c, up_c;
    __device__ __forceinline__ explicit StepScalars(double ts, double dx)
    {
        half_c = 0.5 * (ts / dx);  // computeEvolutionVector (solvers.cpp:601-609)
        lf_c = dx / ts;            // computeLaxFriedrichsFlux (firstordersolver.cpp:83)
        ri_c = ts / dx;            // computeRichtmyerFlux (:169), computeFORCEUpdate (:431)
        up_c = ts / dx;
    }
};

template <int NF>
__device__ __forceinline__ void load_prim(const double *__restrict__ in, long long plane, long long idx, double (&w)[NF])
{
#pragma unroll
    for (int f = 0; f < NF; f++) w[f] = in[f * plane + idx];
}

template <int NF>
__device__ __forceinline__ void store_prim(double *__restrict__ out, long long plane, long long idx, const double (&w)[NF])
{
#pragma unroll
    for (int f = 0; f < NF; f++) out[f * plane + idx] = w[f];
}

// Block-level maximum of the wave-speed keys, written to this block's slot of
// the partials array (no atomics: every block owns one slot, and the 1-block
// clock kernel reduces the slots, so the result does not depend on ordering).
template <int BS>
__device__ __forceinline__ void block_max_to(unsigned long long *partials, unsigned long long key)
{
    __shared__ unsigned long long s_w[BS / kWave];
    key = wave_max_u64(key);
    if ((threadIdx.x & (kWave - 1)) == 0) s_w[threadIdx.x / kWave] = key;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long mx = 0;
#pragma unroll
        for (int k = 0; k < BS / kWave; k++) mx = (s_w[k] > mx) ? s_w[k] : mx;
        partials[(long long)blockIdx.y * gridDim.x + blockIdx.x] = mx;
    }
}

// One tile of a sweep along DIR: the block's threads are BS / LW positions along
// the line by LW lines, thread tid holding position tid / LW of line tid % LW, so
// its neighbours along the line are tid - LW and tid + LW (x tiles: LW = 1).
// Thread tid holds the primitive state w of its cell, whose position in the grid
// is the tile's first output - G + tid / LW (boundary-mapped by the caller);
// positions G .. BS / LW - G - 1 with `write` set compute and store the updated
// cell at out[f * plane + out_idx].  Returns the wave-speed key of the stored cell
// when want_key (else 0).  Ends with a barrier, so the LDS arrays can be reused by
// the next tile.  s_a and s_e hold NF and 2 NF fields per thread; COMPACT (SLIC): NF
// and NF, the left evolved states taking s_a's place once the cells' vectors have been
// read, at two more barriers for a third less LDS.
template <class P, int DIR, int ORDER, int MODE, int BS, int LW, bool BRANCHES, bool COMPACT>
__device__ __forceinline__ unsigned long long line_tile(const typename P::Params &m, const StepScalars &sc, double bias,
                                                        int limiter, const double (&w)[P::NF], bool write,
                                                        double *__restrict__ out, long long plane, long long out_idx,
                                                        int dim, bool want_key, double *s_a, double *s_e)
{
    constexpr int NF = P::NF;
    constexpr int G = (ORDER == 2) ? 2 : 1;
    constexpr int NP = BS / LW;
    constexpr bool kCompact = COMPACT && ORDER == 2;
    using S = Scheme<P, DIR, MODE, BRANCHES>;
    const int tid = threadIdx.x, pos = tid / LW;
    double U[NF], Fp[NF];
    if (ORDER == 2) {
        S::cons(m, w, U);
#pragma unroll
        for (int f = 0; f < NF; f++) s_a[f * BS + tid] = U[f];
        __syncthreads();
        ConsFlux<NF> left, right;
        if (pos >= 1 && pos <= NP - 2) {
            double UL[NF], UR[NF];
#pragma unroll
            for (int f = 0; f < NF; f++) {
                UL[f] = s_a[f * BS + tid - LW];
                UR[f] = s_a[f * BS + tid + LW];
            }
            S::evolve(m, UL, U, UR, bias, limiter, sc.half_c, left, right);
        }
        double *s_u = kCompact ? s_a : s_e, *s_f = kCompact ? s_e : s_e + NF * BS;
        if (kCompact) __syncthreads();   // every neighbour's vector has been read
        if (pos >= 1 && pos <= NP - 2) {
#pragma unroll
            for (int f = 0; f < NF; f++) {
                s_u[f * BS + tid] = left.U[f];
                s_f[f * BS + tid] = left.F[f];
            }
        }
        __syncthreads();
        if (pos >= 1 && pos <= NP - 3) {
            ConsFlux<NF> nb;
#pragma unroll
            for (int f = 0; f < NF; f++) {
                nb.U[f] = s_u[f * BS + tid + LW];
                nb.F[f] = s_f[f * BS + tid + LW];
            }
            S::force_face(m, right, nb, sc.lf_c, sc.ri_c, Fp);   // face pos + 1/2
        }
        if (kCompact) __syncthreads();   // every left state has been read
        if (pos >= 1 && pos <= NP - 3) {
#pragma unroll
            for (int f = 0; f < NF; f++) s_a[f * BS + tid] = Fp[f];
        }
        __syncthreads();
    } else {
        ConsFlux<NF> cf;
        S::cons_flux_of_prim(m, w, cf);
#pragma unroll
        for (int f = 0; f < NF; f++) {
            U[f] = cf.U[f];
            s_e[f * BS + tid] = cf.U[f];
            s_e[(NF + f) * BS + tid] = cf.F[f];
        }
        __syncthreads();
        if (pos <= NP - 2) {
            ConsFlux<NF> nb;
#pragma unroll
            for (int f = 0; f < NF; f++) {
                nb.U[f] = s_e[f * BS + tid + LW];
                nb.F[f] = s_e[(NF + f) * BS + tid + LW];
            }
            S::force_face(m, cf, nb, sc.lf_c, sc.ri_c, Fp);
#pragma unroll
            for (int f = 0; f < NF; f++) s_a[f * BS + tid] = Fp[f];
        }
        __syncthreads();
    }
    unsigned long long key = 0;
    if (pos >= G && pos < NP - G && write) {
        double Fm[NF], wn[NF];
#pragma unroll
        for (int f = 0; f < NF; f++) Fm[f] = s_a[f * BS + tid - LW];
        S::update(m, U, Fm, Fp, sc.up_c, wn);
        store_state<P>(out, plane, out_idx, wn);
        if (want_key) key = max_key(P::wave_speed(m, wn, dim));
    }
    __syncthreads();
    return key;
}

// Start of a step: finish the previous one (t += dt; it += 1 as in
// secondordersolver.cpp:307-308), evaluate the loop condition, then
// dt = CFL * (dx / S), x0.2 for the first six steps, clipped to the final time
// (Solvers/solvers.cpp:392, 437-452).  mx: the wave-speed key of the grid.
// Returns whether a step starts; the clock must not be done.
__device__ __forceinline__ bool clock_advance(Clock &c, unsigned long long mx)
{
    c.smax = mx;
    if (c.pending) {
        c.t += c.dt;
        c.it += 1;
        c.pending = 0;
    }
    if (!(c.t < c.t_final) || (c.max_steps > 0 && c.it >= c.max_steps)) {
        c.done = 1;
        return false;
    }
    double S = __longlong_as_double((long long)mx);
    if (c.corner > S) S = c.corner;
    double dt = c.cfl * (c.dx / S);
    if (c.it <= 5) dt *= 0.2;
    if ((c.t + dt) > c.t_final) dt = c.t_final - c.t;
    if (!(dt > 0.0) || !(c.t + dt > c.t)) {
        // The reference would repeat this step forever (t never reaches t_final);
        // stop and report instead.
        c.done = 1;
        c.stalled = 1;
        return false;
    }
    c.dt = dt;
    c.S = S;
    if (c.steps_this_run == 0 || dt < c.dt_min) c.dt_min = dt;
    if (c.steps_this_run == 0 || dt > c.dt_max) c.dt_max = dt;
    c.steps_this_run += 1;
    c.pending = 1;
    return true;
}

// Whether the small tiles take the compact layout: where the block is one wave its
// barriers cost nothing, and tiles of nine and more fields are bound by the waves
// their LDS lets in (MHD y tiles 55 KB: two blocks of four waves a CU; 37 KB: four).
template <class P, int ORDER, int BS>
constexpr bool kCompactTile = ORDER == 2 && (P::NF >= 9 || BS == kWave);

// Whether walked sweeps take the limiter by branches (Scheme).
template <class P>
constexpr bool kWalkBranches = P::NF <= 9;

// The rows of one x-sweep block, under time step dt and maximum wave speed S.
template <class P, int ORDER, int MODE, int BS, int RX>
__device__ __forceinline__ void sweep_x_rows(const SweepArgs<P> &a, double dt, double S)
{
    constexpr int NF = P::NF;
    constexpr int G = (ORDER == 2) ? 2 : 1;
    constexpr int OUT = BS - 2 * G;
    constexpr bool WALK = RX > 1, BRANCHES = WALK && kWalkBranches<P>;
    constexpr bool COMPACT = !WALK && kCompactTile<P, ORDER, BS>;
    __shared__ double s_a[NF * BS];       // cell conserved vectors, later face fluxes
    // left evolved state (SLIC) / cell state (FORCE): U and F, or F only
    __shared__ double s_e[(COMPACT ? 1 : 2) * NF * BS];

    const double ts = dt * a.dt_scale;
    const StepScalars sc(ts, a.dx);
    typename P::Params m = a.m;
    if (ORDER == 2 && !a.fixed_params) P::begin_step(m, S);   // first-order solvers never set c_h

    const int tid = threadIdx.x;
    const int j = blockIdx.x * OUT - G + tid;
    const int nx = a.nx;
    const int jj = (j >= -G && j < nx + G) ? ghost_index(j, nx, a.bc) : (j < 0 ? 0 : nx - 1);
    const int i_begin = blockIdx.y * RX;
    unsigned long long key = 0;
    auto tile = [&](int i, const double(&w)[NF]) {
        const unsigned long long k2 = line_tile<P, 0, ORDER, MODE, BS, 1, BRANCHES, COMPACT>(
            m, sc, a.bias, a.limiter, w, j < nx, a.out, a.plane, (long long)i * nx + j, a.dim, a.fuse_max != 0, s_a, s_e);
        key = (k2 > key) ? k2 : key;
    };
    double wnext[NF];
    load_state<P>(a.in, a.plane, (long long)i_begin * nx + jj, wnext);
    if constexpr (RX == 1) {
        tile(i_begin, wnext);
    } else {
        // Each block walks RX rows; the next row's cells are loaded while the
        // current row is computed.
        const int i_end = (i_begin + RX < a.ny) ? i_begin + RX : a.ny;
        for (int i = i_begin; i < i_end; i++) {
            double w[NF];
#pragma unroll
            for (int f = 0; f < NF; f++) w[f] = wnext[f];
            if (i + 1 < i_end) load_state<P>(a.in, a.plane, (long long)(i + 1) * nx + jj, wnext);
            tile(i, w);
        }
    }
    if (a.fuse_max) block_max_to<BS>(a.partials, key);
}

template <class P, int ORDER, int MODE, int BS, int RX>
__global__ __launch_bounds__(BS) void sweep_x_kernel(SweepArgs<P> a)
{
    if (a.clk->done) return;
    sweep_x_rows<P, ORDER, MODE, BS, RX>(a, a.clk->dt, a.clk->S);
}

// The first x sweep of a step together with the start of the step: every block
// reduces the wave-speed keys of the last step and advances its own copy of the
// clock, the first block writes the advanced clock and the dt log.  The advanced
// clock is another slot than the one read (and the keys this sweep may write other
// slots than those it reads), since blocks still to start read the old ones.
// Bound by latency: of a 3.1 us clock_begin_kernel launch on a 200 x 200 grid 1.5
// us remain here.  Every block reads every key, so it is for few keys only
// (kBeginSlots).
constexpr int kBeginSlots = 1024;

struct StepBegin {
    const Clock *from;
    Clock *to;
    const unsigned long long *keys;
    int n_keys;
    double *dt_log;
    int dt_cap;
};

template <class P, int ORDER, int MODE>
__global__ __launch_bounds__(kWave) void sweep_x_begin_kernel(SweepArgs<P> a, StepBegin b)
{
    Clock c = *b.from;
    const bool first = blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0;
    bool run = false;
    if (!c.done) {
        unsigned long long key = 0;
#pragma unroll 8
        for (int k = threadIdx.x; k < b.n_keys; k += kWave) {
            const unsigned long long v = b.keys[k];
            key = (v > key) ? v : key;
        }
        run = clock_advance(c, wave_max_u64(key));
        if (run && first && b.dt_log && c.steps_this_run <= b.dt_cap) b.dt_log[c.steps_this_run - 1] = c.dt;
    }
    if (first) *b.to = c;
    if (run) sweep_x_rows<P, ORDER, MODE, kWave, 1>(a, c.dt, c.S);
}

// The y sweep in LDS tiles of LW columns by BS / LW rows, one cell per thread: the
// whole sweep of a cell is one pass of the stencil instead of the walk below, at
// the cost of the tile's halo rows (2 G of BS / LW) being computed twice.
template <class P, int ORDER, int MODE, int BS, int LW>
__device__ __forceinline__ void sweep_y_tile(const SweepArgs<P> &a)
{
    constexpr int NF = P::NF;
    constexpr int G = (ORDER == 2) ? 2 : 1;
    constexpr int NP = BS / LW, OUT = NP - 2 * G;
    __shared__ double s_a[NF * BS];
    constexpr bool COMPACT = kCompactTile<P, ORDER, BS>;
    __shared__ double s_e[(COMPACT ? 1 : 2) * NF * BS];

    if (a.clk->done) return;
    const double ts = a.clk->dt * a.dt_scale;
    const StepScalars sc(ts, a.dx);
    typename P::Params m = a.m;
    if (ORDER == 2 && !a.fixed_params) P::begin_step(m, a.clk->S);   // first-order solvers never set c_h

    const int tid = threadIdx.x;
    const int ny = a.ny, nx = a.nx;
    const int i = blockIdx.y * OUT - G + tid / LW, j = blockIdx.x * LW + tid % LW;
    const int ii = (i >= -G && i < ny + G) ? ghost_index(i, ny, a.bc) : (i < 0 ? 0 : ny - 1);
    const int jj = (j < nx) ? j : nx - 1;
    double w[NF];
    load_state<P>(a.in, a.plane, (long long)ii * nx + jj, w);
    // The y sweep never ends a step, so it writes no CFL partials.
    line_tile<P, 1, ORDER, MODE, BS, LW, false, COMPACT>(m, sc, a.bias, a.limiter, w, i < ny && j < nx, a.out, a.plane,
                                         (long long)i * nx + j, a.dim, false, s_a, s_e);
}

template <class P, int ORDER, int MODE, int BS, int LW>
__global__ __launch_bounds__(BS) void sweep_y_tile_kernel(SweepArgs<P> a)
{
    sweep_y_tile<P, ORDER, MODE, BS, LW>(a);
}

// The tile sweeps of two grids of one shape in one launch (the launch's third
// dimension picks the grid): on small grids one grid's tiles leave the device half
// empty.
template <class P>
struct SweepPair {
    SweepArgs<P> a, b;
};

template <class P, int ORDER, int MODE>
__global__ __launch_bounds__(kWave) void sweep_x_pair_kernel(SweepPair<P> p)
{
    const SweepArgs<P> a = blockIdx.z ? p.b : p.a;
    if (a.clk->done) return;
    sweep_x_rows<P, ORDER, MODE, kWave, 1>(a, a.clk->dt, a.clk->S);
}

template <class P, int ORDER, int MODE, int BS, int LW>
__global__ __launch_bounds__(BS) void sweep_y_tile_pair_kernel(SweepPair<P> p)
{
    const SweepArgs<P> a = blockIdx.z ? p.b : p.a;
    sweep_y_tile<P, ORDER, MODE, BS, LW>(a);
}

// A thread per column walks H rows with the stencil window in registers.  The y
// sweep never ends a step, so it writes no CFL partials.
template <class P, int ORDER, int MODE, int BS, int H>
__global__ __launch_bounds__(BS) void sweep_y_kernel(SweepArgs<P> a)
{
    constexpr int NF = P::NF;
    using S = Scheme<P, 1, MODE, kWalkBranches<P>>;

    if (a.clk->done) return;
    const double ts = a.clk->dt * a.dt_scale;
    const StepScalars sc(ts, a.dx);
    typename P::Params m = a.m;
    if (ORDER == 2 && !a.fixed_params) P::begin_step(m, a.clk->S);   // first-order solvers never set c_h

    const int j = blockIdx.x * BS + threadIdx.x;
    const int ny = a.ny, nx = a.nx;
    const int i0 = blockIdx.y * H;
    const int i1 = (i0 + H < ny) ? i0 + H : ny;
    if (j >= nx) return;
    auto row_of = [&](int r) -> long long { return (long long)ghost_index(r, ny, a.bc) * nx + j; };
    if (ORDER == 2) {
        double A[NF], B[NF], C[NF], w[NF];
        load_state<P>(a.in, a.plane, row_of(i0 - 2), w);
        S::cons(m, w, A);
        load_state<P>(a.in, a.plane, row_of(i0 - 1), w);
        S::cons(m, w, B);
        load_state<P>(a.in, a.plane, row_of(i0), w);   // row e + 1 of the first iteration
        ConsFlux<NF> er_prev;
        double Fprev[NF];
        for (int e = i0 - 1; e <= i1; e++) {
            S::cons(m, w, C);
            if (e + 2 <= i1 + 1) load_state<P>(a.in, a.plane, row_of(e + 2), w);   // prefetch
            ConsFlux<NF> L, R;
            S::evolve(m, A, B, C, a.bias, a.limiter, sc.half_c, L, R);
            double Fnew[NF];
            if (e >= i0) S::force_face(m, er_prev, L, sc.lf_c, sc.ri_c, Fnew);   // face e - 1/2
            if (e >= i0 + 1) {
                double wn[NF];
                S::update(m, A, Fprev, Fnew, sc.up_c, wn);                       // row e - 1
                store_state<P>(a.out, a.plane, (long long)(e - 1) * nx + j, wn);
            }
#pragma unroll
            for (int f = 0; f < NF; f++) {
                Fprev[f] = Fnew[f];
                er_prev.U[f] = R.U[f];
                er_prev.F[f] = R.F[f];
                A[f] = B[f];
                B[f] = C[f];
            }
        }
    } else {
        double w[NF];
        ConsFlux<NF> prev;
        double Fprev[NF];
        load_state<P>(a.in, a.plane, row_of(i0 - 1), w);
        S::cons_flux_of_prim(m, w, prev);
        for (int e = i0; e <= i1; e++) {
            ConsFlux<NF> cur;
            load_state<P>(a.in, a.plane, row_of(e), w);
            S::cons_flux_of_prim(m, w, cur);
            double Fnew[NF];
            S::force_face(m, prev, cur, sc.lf_c, sc.ri_c, Fnew);                 // face e - 1/2
            if (e >= i0 + 1) {
                double wn[NF];
                S::update(m, prev.U, Fprev, Fnew, sc.up_c, wn);                  // row e - 1
                store_state<P>(a.out, a.plane, (long long)(e - 1) * nx + j, wn);
            }
#pragma unroll
            for (int f = 0; f < NF; f++) {
                Fprev[f] = Fnew[f];
                prev.U[f] = cur.U[f];
                prev.F[f] = cur.F[f];
            }
        }
    }
}

// Wave-speed maximum of a whole grid (the first step, or after the caller
// changed the state).
template <class P>
__global__ __launch_bounds__(256) void wave_max_kernel(const double *__restrict__ in, long long plane, long long cells,
                                                       int dim, typename P::Params m, unsigned long long *partials)
{
    constexpr int NF = P::NF;
    unsigned long long key = 0;
    for (long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x; c < cells; c += (long long)gridDim.x * blockDim.x) {
        double w[NF];
        load_prim<NF>(in, plane, c, w);
        const unsigned long long k2 = max_key(P::wave_speed(m, w, dim));
        key = (k2 > key) ? k2 : key;
    }
    block_max_to<256>(partials, key);
}

// The same of two grids, the second's keys after the first's.
template <class P>
__global__ __launch_bounds__(256) void wave_max_pair_kernel(const double *__restrict__ in_a, const double *__restrict__ in_b,
                                                            long long plane, long long cells, int dim,
                                                            typename P::Params ma, typename P::Params mb,
                                                            unsigned long long *partials)
{
    constexpr int NF = P::NF;
    const double *in = blockIdx.y ? in_b : in_a;
    const typename P::Params m = blockIdx.y ? mb : ma;
    unsigned long long key = 0;
    for (long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x; c < cells; c += (long long)gridDim.x * blockDim.x) {
        double w[NF];
        load_prim<NF>(in, plane, c, w);
        const unsigned long long k2 = max_key(P::wave_speed(m, w, dim));
        key = (k2 > key) ? k2 : key;
    }
    block_max_to<256>(partials, key);
}

// Reduces n partial keys with one block of kReduceThreads threads; returns the
// maximum in thread 0.
constexpr int kReduceThreads = 1024;

__device__ __forceinline__ unsigned long long reduce_partials(const unsigned long long *partials, int n)
{
    __shared__ unsigned long long s_r[kReduceThreads / kWave];
    unsigned long long key = 0;
    // eight loads in flight: the small tiles of a 1531 x 1000 grid leave 26,027 slots
    int k = threadIdx.x;
    for (; k + 7 * kReduceThreads < n; k += 8 * kReduceThreads) {
        unsigned long long v[8];
#pragma unroll
        for (int q = 0; q < 8; q++) v[q] = partials[k + q * kReduceThreads];
#pragma unroll
        for (int q = 0; q < 8; q++) key = (v[q] > key) ? v[q] : key;
    }
    for (; k < n; k += kReduceThreads) key = (partials[k] > key) ? partials[k] : key;
    key = wave_max_u64(key);
    if ((threadIdx.x & (kWave - 1)) == 0) s_r[threadIdx.x / kWave] = key;
    __syncthreads();
    unsigned long long mx = 0;
    if (threadIdx.x == 0) {
        for (int k = 0; k < kReduceThreads / kWave; k++) mx = (s_r[k] > mx) ? s_r[k] : mx;
    }
    return mx;
}

static __global__ __launch_bounds__(kReduceThreads) void reduce_max_kernel(const unsigned long long *partials, int n, Clock *clk)
{
    const unsigned long long mx = reduce_partials(partials, n);
    if (threadIdx.x == 0) clk->smax = mx;
}

// Default-state wave speed (2D transmissive corner ghosts) into clk->corner.
template <class P>
__global__ void corner_speed_kernel(typename P::Params m, int dim, Clock *clk)
{
    double w[P::NF];
    P::default_state(w);
    clk->corner = P::wave_speed(m, w, dim);
}

static __global__ __launch_bounds__(kReduceThreads) void clock_begin_kernel(Clock *c, const unsigned long long *partials,
                                                                    int n_partials, double *dt_log, int dt_cap)
{
    if (c->done) return;   // uniform: nothing pending once done
    const unsigned long long mx = reduce_partials(partials, n_partials);
    if (threadIdx.x != 0) return;
    Clock h = *c;
    if (clock_advance(h, mx) && dt_log && h.steps_this_run <= dt_cap) dt_log[h.steps_this_run - 1] = h.dt;
    *c = h;
}

// End of a run: finishes its last step.  With `keys`, the run's last wave-speed keys, n of
// them, stand in the second set and move to the first, where the next run looks for them.
static __global__ void clock_finish_kernel(Clock *c, unsigned long long *keys = nullptr, long long slots = 0, int n = 0)
{
    if (keys)
        for (int k = threadIdx.x; k < n; k += blockDim.x) keys[k] = keys[slots + k];
    if (threadIdx.x == 0 && c->pending) {
        c->t += c->dt;
        c->it += 1;
        c->pending = 0;
    }
}

// Array-of-structures (the reference's layout) <-> structure-of-arrays planes.
template <int NF>
__global__ __launch_bounds__(256) void aos_to_soa_kernel(const double *__restrict__ aos, double *__restrict__ soa,
                                                         long long plane, long long cells)
{
    for (long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x; c < cells; c += (long long)gridDim.x * blockDim.x) {
#pragma unroll
        for (int f = 0; f < NF; f++) soa[f * plane + c] = aos[c * NF + f];
    }
}

template <int NF>
__global__ __launch_bounds__(256) void soa_to_aos_kernel(const double *__restrict__ soa, double *__restrict__ aos,
                                                         long long plane, long long cells)
{
    for (long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x; c < cells; c += (long long)gridDim.x * blockDim.x) {
#pragma unroll
        for (int f = 0; f < NF; f++) aos[c * NF + f] = soa[f * plane + c];
    }
}

// Counts cells whose state is not finite or not admissible for the physics
// (P::admissible: e.g. a real sound speed), and records the smallest such flat index.
template <class P>
__global__ __launch_bounds__(256) void nonfinite_kernel(const double *__restrict__ soa, long long plane, long long cells,
                                                        typename P::Params m, unsigned long long *count,
                                                        unsigned long long *first)
{
    constexpr int NF = P::NF;
    for (long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x; c < cells; c += (long long)gridDim.x * blockDim.x) {
        double w[NF];
        bool bad = false;
#pragma unroll
        for (int f = 0; f < NF; f++) {
            w[f] = (f < StoredFields<P>::n) ? soa[f * plane + c] : 0.0;
            bad = bad || !isfinite(w[f]);
        }
        bad = bad || !P::admissible(m, w);
        if (bad) {
            atomicAdd(count, 1ull);
            atomicMin(first, (unsigned long long)c);
        }
    }
}

}  // namespace vg
