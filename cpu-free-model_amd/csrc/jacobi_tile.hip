// Register-tile Jacobi sweeps: several sweeps between two device-wide
// barriers, with the field's tile held in the registers of one workgroup.
//
// A workgroup loads a tile (its own rows and columns plus `depth` more on every
// side that has a neighbour), advances all of it by `depth` sweeps without
// leaving the registers, and stores the points it owns; the outermost ring goes
// stale by one row/column per sweep, so exactly the owned points are
// right after the last one.  Every value comes from the single-sweep expression,
// so the results are the single-sweep kernels' bits.
//
// The streaming kernels (jacobi.hip) need a field long enough to stream: a
// 1024^2 field gives them 64 wavefronts, each walking 70 rows one after the
// other.  Here the whole chip works on such a field at once, and a sweep costs
// one workgroup barrier, not a device-wide one.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "jacobi_dev.hpp"
#include "jacobi_host.hpp"

namespace cfm {

namespace {

// N consecutive elements at any element-aligned address.
template <typename T, int N>
struct VecAt {
    typedef T type __attribute__((ext_vector_type(N), aligned(sizeof(T))));
};

// A lane's N elements at row[x .. x+N), and one of them.  THROUGH: past the L2 (scope bit sc1), for
// grid_barrier_through; offsets are 32-bit, so jacobi_tile_configure declines rows of 2 GiB and more.
template <bool THROUGH, typename T, int N>
__device__ __forceinline__ typename VecAt<T, N>::type load_at(const T *row, int x) {
    typedef typename VecAt<T, N>::type V;
    if constexpr (THROUGH) {
        static_assert(sizeof(T) * N == 16, "one 16-byte vector");
        const auto rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)row, (short)0, 0x7fffffff, 0x00020000);
        return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b128(rsrc, x * (int)sizeof(T), 0, kSc1));
    } else {
        return *reinterpret_cast<const V *>(row + x);
    }
}
template <bool THROUGH, typename T>
__device__ __forceinline__ T load_one(const T *p) {
    if constexpr (THROUGH)
        return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else
        return *p;
}
template <bool THROUGH, typename T, int N, typename V>
__device__ __forceinline__ void store_at(T *row, int x, V v) {
    if constexpr (THROUGH) {
        typedef unsigned int U4 __attribute__((ext_vector_type(4)));
        const auto rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)row, (short)0, 0x7fffffff, 0x00020000);
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(U4, v), rsrc, x * (int)sizeof(T), 0, kSc1);
    } else {
        *reinterpret_cast<V *>(row + x) = v;
    }
}
template <bool THROUGH, typename T>
__device__ __forceinline__ void store_one(T *p, T v) {
    if constexpr (THROUGH)
        __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else
        *p = v;
}

// ------------------------------------------------------------------ 2D ----
// WAVES wavefronts, one above the other; each spans the tile's C columns (VX
// per lane) and holds R rows.  The rows just outside a wavefront's own come
// from its neighbours through LDS (two buffers: one workgroup barrier per
// sweep); they are published before, and needed only after, the R - 2 inner
// rows, which hide the barrier.  x-neighbours are DPP shifts.
template <typename T, int VX, int R, int WAVES>
struct Tile2D {
    static constexpr int C = 64 * VX;
    static constexpr int H = R * WAVES;
    typedef T Edge[2][WAVES][2][C];

    T a[R][VX];
    int wave, lane;
    bool xin[VX];            // column is updated (not a face, not outside)
    bool xown[VX];           // column is this tile's
    int row_lo, row_hi;      // rows r in [row_lo, row_hi) are updated
    int own_lo, own_hi;      // rows r in [own_lo, own_hi) are this tile's

    // No branches: a row that is not updated (a face, outside the field) is computed and dropped,
    // which keeps the rows in one straight line (with a branch per row the 16-row shapes spill).
    template <bool MASK, bool NORM>
    __device__ __forceinline__ void update(int r, T (&c)[VX], const T (&S)[VX], const T (&N)[VX], double &acc) {
        const T quarter = T(0.25);
        const T west = lane_up1z(c[VX - 1]);
        const T east = lane_dn1z(c[0]);
        const bool live = r >= row_lo && r < row_hi;  // uniform over the wavefront
        const bool count = NORM && r >= own_lo && r < own_hi;
        T out[VX];
#pragma unroll
        for (int k = 0; k < VX; ++k) {
            const T E = k < VX - 1 ? c[k + 1] : east;
            const T W = k > 0 ? c[k - 1] : west;
            const T v = quarter * (E + W + N[k] + S[k]);
            out[k] = !MASK || (xin[k] && live) ? v : c[k];
            if (NORM) {
                const double d = (double)v - (double)c[k];
                acc = (count && xown[k] && xin[k]) ? acc + d * d : acc;
            }
        }
#pragma unroll
        for (int k = 0; k < VX; ++k) {
            c[k] = out[k];
            // pins the row here: left free, the compiler starts rows early and ends them late, and
            // the tall shapes run out of registers
            asm volatile("" : "+v"(c[k]));
        }
    }

    // one sweep of the tile; e: this sweep's LDS buffer
    template <bool MASK, bool NORM>
    __device__ __forceinline__ void sweep(T (&e)[WAVES][2][C], double &acc) {
        typedef typename VecAt<T, VX>::type V;
        if (MASK || NORM)  // (opaque: hoisted out of the sweep loop, the row tests would hold two scalar registers a row)
            asm volatile("" : "+s"(row_lo), "+s"(row_hi), "+s"(own_lo), "+s"(own_hi));
        V lo, hi;
#pragma unroll
        for (int k = 0; k < VX; ++k) {
            lo[k] = a[0][k];
            hi[k] = a[R - 1][k];
        }
        *reinterpret_cast<V *>(&e[wave][0][lane * VX]) = lo;
        *reinterpret_cast<V *>(&e[wave][1][lane * VX]) = hi;
        T second[VX], prev[VX];
#pragma unroll
        for (int k = 0; k < VX; ++k) prev[k] = a[0][k];
#pragma unroll
        for (int r = 1; r < R - 1; ++r) {
            T old[VX];
#pragma unroll
            for (int k = 0; k < VX; ++k) old[k] = a[r][k];
            update<MASK, NORM>(r, a[r], prev, a[r + 1], acc);
#pragma unroll
            for (int k = 0; k < VX; ++k) {
                if (r == 1) second[k] = old[k];
                prev[k] = old[k];
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();
        // the tile's own outer rows have no neighbour: any value does, they are stale already
        const V up = *reinterpret_cast<const V *>(&e[wave > 0 ? wave - 1 : 0][1][lane * VX]);
        const V dn = *reinterpret_cast<const V *>(&e[wave < WAVES - 1 ? wave + 1 : wave][0][lane * VX]);
        T u[VX], d[VX];
#pragma unroll
        for (int k = 0; k < VX; ++k) {
            u[k] = up[k];
            d[k] = dn[k];
        }
        update<MASK, NORM>(0, a[0], u, second, acc);
        update<MASK, NORM>(R - 1, a[R - 1], prev, d, acc);
    }
};

// Row that a wrapped row index stands for: the interior rows 1..ny-2 repeat.
__device__ __forceinline__ int wrap_row(int y, int ny) {
    const int p = ny - 2;
    int m = (y - 1) % p;
    if (m < 0) m += p;
    return 1 + m;
}

// Where a tile lies, the same for the whole workgroup.
struct Place2D {
    int x0, xo, xo_end;  // first column; owned columns [xo, xo_end)
    int y0, yo, yo_end;  // first row; owned rows [yo, yo_end), interior rows only
    bool wrap;           // rows repeat beyond the interior
};

// One tile, one pass.  EDGE = false: the tile touches no face and none of the pass's sweeps wants
// its update norm, so nothing is tested per row or column.
template <bool EDGE, bool THROUGH, typename T, int VX, int R, int WAVES>
__device__ __forceinline__ void pass_tile2d(const JacobiArgs &A, const Place2D &P, const T *__restrict__ src,
                                            T *__restrict__ dst, int steps, int it, bool first,
                                            typename Tile2D<T, VX, R, WAVES>::Edge &edge, double *lds) {
    typedef typename VecAt<T, VX>::type V;
    const int nx = A.nx, ny = A.ny;
    Tile2D<T, VX, R, WAVES> t;
    t.lane = threadIdx.x & 63;
    t.wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int x = P.x0 + t.lane * VX;  // first column of this lane
    const int y = P.y0 + t.wave * R;   // first row of this wavefront
    t.own_lo = P.yo - y;
    t.own_hi = P.yo_end - y;
    if constexpr (EDGE) {
#pragma unroll
        for (int e = 0; e < VX; ++e) {
            t.xin[e] = x + e >= 1 && x + e <= nx - 2;
            t.xown[e] = x + e >= P.xo && x + e < P.xo_end;
        }
        t.row_lo = P.wrap ? 0 : 1 - y;
        t.row_hi = P.wrap ? R : ny - 1 - y;
    }
    // load the tile; what lies outside the field is never updated and never read by a point that is
    int row = P.wrap ? wrap_row(y, ny) : y;
    if (!EDGE && row + R <= ny - 1) {  // (wrapped rows may cross the seam)
        const T *p = src + (size_t)row * nx + P.x0;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const V v = load_at<THROUGH, T, VX>(p + (size_t)r * nx, t.lane * VX);
#pragma unroll
            for (int e = 0; e < VX; ++e) t.a[r][e] = v[e];
        }
    } else {
        const bool lane_in = !EDGE || (x >= 0 && x + VX <= nx);
#pragma unroll
        for (int r = 0; r < R; ++r) {
#pragma unroll
            for (int e = 0; e < VX; ++e) t.a[r][e] = T(0);
            if (!EDGE || (row >= 0 && row < ny)) {  // uniform
                const T *p = src + (size_t)row * nx;
                if (lane_in) {
                    const V v = load_at<THROUGH, T, VX>(p, x);
#pragma unroll
                    for (int e = 0; e < VX; ++e) t.a[r][e] = v[e];
                } else {
#pragma unroll
                    for (int e = 0; e < VX; ++e)
                        if (x + e >= 0 && x + e < nx) t.a[r][e] = load_one<THROUGH>(p + x + e);
                }
            }
            ++row;
            if (P.wrap && row == ny - 1) row = 1;
        }
    }
    // wait for the loads here: left to the first use, they are waited for again before every store
    // below (a pass could have no sweeps, for all the compiler knows), and so is each store before it
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    double acc = 0.0;
    if constexpr (!EDGE) {
        for (int s = 0; s < steps; ++s) t.template sweep<false, false>(edge[s & 1], acc);
    } else {
        int to_norm = A.norm_every > 0 ? (A.norm_every - it % A.norm_every) % A.norm_every : steps;
        for (int s = 0; s < steps;) {
            const int stop = min(steps, to_norm);
            for (; s < stop; ++s) t.template sweep<true, false>(edge[s & 1], acc);
            if (s < steps) {  // uniform over the grid: this sweep's update norm is wanted
                acc = 0.0;
                t.template sweep<true, true>(edge[s & 1], acc);
                const double sum = block_sum_waves<WAVES>(acc, lds);
                double *slot = A.norm_part + (size_t)((it + s) / A.norm_every) * gridDim.x + blockIdx.x;
                if (threadIdx.x == 0) *slot = first ? sum : *slot + sum;
                ++s;
                to_norm += A.norm_every;
            }
        }
    }
    // store the owned points; the halo rows of a wrapped field are copies of whole rows
    const bool periodic = A.bc == CFM_BC_PERIODIC;
    const bool whole = x >= P.xo && x + VX <= P.xo_end && x >= 1 && x + VX <= nx - 1;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        if (r >= t.own_lo && r < t.own_hi) {  // uniform
            V v;
#pragma unroll
            for (int e = 0; e < VX; ++e) v[e] = t.a[r][e];
            T *p = dst + (size_t)(y + r) * nx;
            if (whole) {
                store_at<THROUGH, T, VX>(p, x, v);
            } else {
#pragma unroll
                for (int e = 0; e < VX; ++e)
                    if (x + e >= P.xo && x + e < P.xo_end && x + e >= 1 && x + e <= nx - 2)
                        store_one<THROUGH, T>(p + x + e, v[e]);
            }
            if (periodic && (y + r == 1 || y + r == ny - 2)) {
#pragma unroll
                for (int e = 0; e < VX; ++e)
                    if (x + e >= P.xo && x + e < P.xo_end) {
                        if (y + r == ny - 2) store_one<THROUGH, T>(dst + x + e, v[e]);
                        if (y + r == 1) store_one<THROUGH, T>(dst + (size_t)(ny - 1) * nx + x + e, v[e]);
                    }
            }
        }
    }
}

// (128 registers a lane at most: two 8-wavefront workgroups, or one of 16, per CU)
// Shapes for fields of few tiles go past the L2 (a tile is read once a pass, and each pass's
// lines are another workgroup's by the next): the light barrier is worth more than the L2's hits
// on the halos.  The shape for fields of many tiles keeps the L2.
template <typename T, int VX, int R, int WAVES, bool TIMED>
__global__ void __launch_bounds__(64 * WAVES, 4) jacobi2d_tile_kernel(JacobiArgs A) {
    constexpr int C = 64 * VX;
    constexpr bool THROUGH = WAVES > 8;
    __shared__ typename Tile2D<T, VX, R, WAVES>::Edge edge;
    __shared__ double lds[WAVES];
    __shared__ unsigned long long clk_lds[kClockWords];
    PhaseClock<TIMED> clk{clk_lds};
    clk.start();
    const int nx = A.nx, ny = A.ny;
    const bool periodic = A.bc == CFM_BC_PERIODIC;
    const int ntiles = A.ntx * A.nty;
    const int first = xcd_block_id();
    unsigned int epoch = 0;
    int pass = 0;
    for (int k = 0; k < A.niter; ++pass) {
        // Periodic rows: the first sweep reads the caller's halo rows, which need not be copies
        // of the opposite ends yet; from the second on the rows simply repeat.
        Place2D P;
        P.wrap = periodic && k > 0;
        const int steps = (periodic && k == 0) ? 1 : min(A.depth, A.niter - k);
        const int it = A.it0 + k;
        const bool norm = A.norm_every > 0 && (it + A.norm_every - 1) / A.norm_every * A.norm_every < it + steps;
        const T *src = static_cast<const T *>((pass & 1) ? A.buf1 : A.buf0);
        T *dst = static_cast<T *>((pass & 1) ? A.buf0 : A.buf1);
        for (int u = first; u < ntiles; u += gridDim.x) {
            const int ty = u / A.ntx, tx = u - ty * A.ntx;
            P.xo = tx * A.tile_sx;
            P.xo_end = min(P.xo + A.tile_sx, nx);
            P.x0 = P.xo - A.tile_hx;
            P.yo = 1 + ty * A.tile_sy;
            P.yo_end = min(P.yo + A.tile_sy, ny - 1);
            P.y0 = P.yo - A.tile_hy;
            const bool face = P.x0 < 1 || P.x0 + C > nx - 1 || (!P.wrap && (P.y0 < 1 || P.y0 + R * WAVES > ny - 1));
            if (face || norm)  // uniform over the workgroup
                pass_tile2d<true, THROUGH, T, VX, R, WAVES>(A, P, src, dst, steps, it, u == first, edge, lds);
            else
                pass_tile2d<false, THROUGH, T, VX, R, WAVES>(A, P, src, dst, steps, it, u == first, edge, lds);
            // the next tile's first publication must not overtake this one's last reads
            __syncthreads();
        }
        k += steps;
        if (k < A.niter) {
            if (!pass_barrier<THROUGH>(A, epoch, clk)) return;
        }
    }
    clk.mark(CFM_PHASE_SPMV);
    clk.flush(A.timers);
}

struct Shape2D {
    int vx, r, waves;
    KernelFn fn[2];  // [timed]
};

template <typename T, int VX, int R, int WAVES>
Shape2D shape2d() {
    return {VX, R, WAVES, {(KernelFn)jacobi2d_tile_kernel<T, VX, R, WAVES, false>,
                           (KernelFn)jacobi2d_tile_kernel<T, VX, R, WAVES, true>}};
}

struct Split2D {
    int hx, hy, ntx, nty, sx, sy;
};

// Tiles of one shape at one depth.  A field that one tile spans needs no halo on that axis.
Split2D split2d(const cfm_jacobi_params &p, const Shape2D &s, int depth) {
    const int C = 64 * s.vx, H = s.r * s.waves, interior = p.ny - 2;
    const bool one_x = p.nx <= C, one_y = p.bc == CFM_BC_DIRICHLET && p.ny <= H;
    Split2D o;
    o.hx = one_x ? 0 : (depth + s.vx - 1) / s.vx * s.vx;
    o.hy = one_y ? 1 : depth;
    const int ox = one_x ? C : C - 2 * o.hx, oy = one_y ? H : H - 2 * o.hy;
    if (ox < s.vx || oy < 1) return {0, 0, 0, 0, 0, 0};
    o.ntx = one_x ? 1 : (p.nx + ox - 1) / ox;
    o.sx = one_x ? C : ((p.nx + o.ntx - 1) / o.ntx + s.vx - 1) / s.vx * s.vx;
    o.nty = one_y ? 1 : (interior + oy - 1) / oy;
    o.sy = (interior + o.nty - 1) / o.nty;
    return o;
}

// Estimated microseconds of one pass of `depth` sweeps; what the terms stand for was measured on
// MI355X:
//   * a wavefront's row costs its vector instructions (4 cycles each at 2.4 GHz): 12 per 2 FP64
//     points and 18 per 4 FP32 points, 16 and 22 where faces are masked, on 4 SIMDs;
//   * a sweep's workgroup barrier and LDS rows: 0.2 us for 16 wavefronts, 0.05 where a second
//     workgroup on the CU fills the wait;
//   * a pass's device-wide barrier, first loads and last stores: 5.5 us past the L2, 9 us with the
//     barrier's two fences, 2 us if one workgroup does it all;
//   * the part of the field's traffic (at 5 TB/s) that a second workgroup on the CU does not hide.
// At 16384^2 FP64 in 14-row, 8-wavefront tiles it gives 890, 1330 and 1800 us for depths 8, 12 and
// 16, measured 900, 1322 and 1780; at 1024^2 in 6-row tiles 16.1 and 23.2 for depths 12 and 20,
// measured 17.2 and 24.9.
double pass_us(const cfm_jacobi_params &p, const Shape2D &s, int depth, double cus) {
    const Split2D o = split2d(p, s, depth);
    if (o.ntx < 1) return 1e30;
    const bool f64 = p.prec == CFM_F64;
    const double tiles = (double)o.ntx * o.nty;
    const bool pairs = s.waves <= 8;  // two workgroups per CU
    const double rounds = std::ceil(tiles / cus);
    const bool at_once = rounds <= (pairs ? 2 : 1);  // a pass then lasts as long as its tiles with faces
    const double row = (f64 ? (at_once ? 64 : 48) : (at_once ? 88 : 72)) / 2400.0;
    const double traffic = 2.0 * (f64 ? 8 : 4) * p.nx * (double)p.ny / 5.0e6;
    return (tiles > 1 ? (pairs ? 9.0 : 5.5) : 2.0) + 1.07 * rounds * depth * (s.r * s.waves / 4) * row +
           (pairs ? 0.05 * std::ceil(rounds / 2) : 0.2 * rounds) * depth + (pairs ? 0.5 : 0.75) * traffic;
}

// Estimated microseconds of `sweeps` sweeps from the start of a run: its passes, with what large, flat and
// narrow fields and norms add to them (measured, too):
//   * a pass that moves more than the caches hold takes at least its traffic at 4.2 TB/s;
//   * each round of tiles beyond the first its loads and stores: 1.2 us, 2.2 for pairs of workgroups (16 and
//     fewer rows of 2,000,000), 3 more where every tile has a face in x (8 to 64 columns);
//   * a pass with a norm masks all its tiles, and each norm sums up every point.
double run_us(const cfm_jacobi_params &p, const Shape2D &s, int depth, double cus, int sweeps) {
    const Split2D o = split2d(p, s, depth);
    const bool f64 = p.prec == CFM_F64, pairs = s.waves <= 8;
    const double rounds = std::ceil((double)o.ntx * o.nty / cus), rows = rounds * (s.r * s.waves / 4);
    const double moved = 2.0 * (f64 ? 8 : 4) * p.nx * (double)p.ny;
    const double tiles = (rounds - 1) * ((pairs ? 2.2 : 1.2) + (o.ntx <= 2 ? 3.0 : 0.0));
    const bool masked = rounds <= (pairs ? 2 : 1);  // (as in pass_us)
    double us = 0.0;
    for (int k = 0; k < sweeps;) {
        const int steps = p.bc == CFM_BC_PERIODIC && k == 0 ? 1 : std::min(depth, sweeps - k);
        const int ne = p.norm_every, norms = ne > 0 ? (k + steps + ne - 1) / ne - (k + ne - 1) / ne : 0;
        double pass = pass_us(p, s, steps, cus) + tiles + norms * rows * (f64 ? 0.025 : 0.052);
        if (norms > 0 && !masked) pass += 1.07 * rows * steps * (f64 ? 16 : 30) / 2400.0;
        us += moved > 2.5e8 ? std::max(pass, moved / 4.2e6) : pass;
        k += steps;
    }
    return us;
}

// The same of the streaming kernels (jacobi.hip), as configured in c: a row after another of a chunk, one and
// two more at each end for every further sweep of the pass, for each round of wavefronts; norms cost them
// nothing.  Microseconds of a row for 1 to 4 sweeps a pass, more the fuller the chip is (half as much again for FP32 rows that
// are not whole vectors), and TB/s; 9 us between passes.  At 16384^2 and 1024^2 FP64 this gives 1202 and 156
// us for four sweeps, 904 and 91 for two of periodic rows, measured 1124 and 144, 863 and 89.
double streaming_us(const cfm_jacobi_params &p, const JacobiConfig &c, int sweeps) {
    static const double row64[] = {0.85, 1.0, 1.5, 1.9}, row32[] = {1.0, 1.4, 1.6, 2.4}, periodic[] = {0.9, 1.15};
    static const double tb64[] = {4.8, 4.8, 4.0, 3.6}, tb32[] = {4.6, 4.5, 4.0, 3.1};
    const bool f64 = p.prec == CFM_F64, per = p.bc == CFM_BC_PERIODIC;
    const bool ragged = !f64 && (size_t)p.nx * 4 % 16 != 0;
    const double fill = (double)c.ntx * c.chunks / ((double)c.grid * (c.block / 64)), rounds = std::max(1.0, fill);
    const double moved = 2.0 * c.elem_size * p.nx * (double)p.ny;
    const auto pass = [&](int s) {
        double row = (per ? periodic : f64 ? row64 : row32)[s - 1];
        if (fill <= 1.0) row *= 1.0 + (s == 1 ? 0.7 : 0.3) * fill;
        const double tb = per ? 4.8 : (f64 ? tb64 : tb32)[s - 1];
        return (sweeps == 1 ? 2.0 : 9.0) +
               std::max(rounds * (c.chunk_len + 2 * (s - 1)) * row * (ragged ? 1.5 : 1.0), moved / (tb * 1e6));
    };
    const int whole = c.sweeps_per_pass, rest = sweeps % whole;
    return (sweeps / whole ? sweeps / whole * pass(whole) : 0.0) + (rest ? pass(rest) : 0.0);
}

}  // namespace

bool jacobi_tile_configure(const cfm_jacobi_params &p, JacobiConfig *c) {
    const bool f64 = p.prec == CFM_F64;
    // a row's byte offsets are 32-bit, and a buffer's range check drops what lies beyond 2 GiB
    if (p.nz >= 3 || (double)p.nx * (f64 ? 8 : 4) > 0x7fffffff) return false;
    // 16-wavefront shapes for fields of few tiles (short rows of work per wavefront, one
    // workgroup per CU); 14 (FP32: 13, 14 spills when timed) rows in 8 wavefronts, two workgroups per CU that hide each other's
    // loads, for fields of many (16384^2 FP64 x 48 sweeps: 5.3 ms against 5.7 for 8 x 16).
    static const Shape2D s64[] = {shape2d<double, 2, 4, 16>(), shape2d<double, 2, 6, 16>(),
                                  shape2d<double, 2, 8, 16>(), shape2d<double, 2, 14, 8>()};
    static const Shape2D s32[] = {shape2d<float, 4, 4, 16>(), shape2d<float, 4, 6, 16>(), shape2d<float, 4, 8, 16>(),
                                  shape2d<float, 4, 13, 8>()};
    // a run of n sweeps: whole passes and a shorter last one (periodic rows: the first sweep alone)
    const int sweeps = std::max(p.niter - (p.bc == CFM_BC_PERIODIC ? 1 : 0), 1);
    const Shape2D *best = nullptr;
    int depth = 0;
    double best_us = 1e30;
    const int most = jacobi_norm_workgroups(*c);
    const auto cus_of = [&](const Shape2D &s) {  // as many as `most` workgroups fill
        const double per_cu = s.waves <= 8 ? 2.0 : 1.0;
        return std::min(per_cu * c->dev.cus, (double)most) / per_cu;
    };
    for (const Shape2D &s : f64 ? s64 : s32) {
        const double cus = cus_of(s);
        const Split2D whole = split2d(p, s, 1);
        if (whole.ntx * whole.nty == 1 && p.bc == CFM_BC_DIRICHLET) {  // one workgroup holds the field
            const double us = pass_us(p, s, sweeps, cus);
            if (us < best_us) best_us = us, best = &s, depth = sweeps;
            continue;
        }
        for (int d = std::min(2, sweeps); d <= std::min(24, sweeps); ++d) {
            double us = sweeps / d * pass_us(p, s, d, cus);
            if (sweeps % d) us += pass_us(p, s, sweeps % d, cus);
            if (us < best_us) best_us = us, best = &s, depth = d;
        }
    }
    if (!best) return false;
    // The streaming kernels walk the rows of a field of any shape at the memory's rate, with or without norms:
    // they are the faster ones for a few sweeps of a large field, and for fields of few rows, most of
    // which a tile's rows lie outside.  FP64, us, streaming / tiles: 16384^2 1 sweep 893 / 987, 2 of periodic rows 921 /
    // 1977, 4 1331 / 923, 40 with every norm 11,614 / 9886; 4,000,000 x 5, 40 sweeps 1054 / 4365, 1,000,000 x 32
    // 1643 / 1295.  (Within the estimates' spread of 8 % the streaming kernels keep a run.)
    const int few = std::min(p.niter, 4096);
    if (1.08 * run_us(p, *best, depth, cus_of(*best), few) > streaming_us(p, *c, few)) return false;
    KernelFn fn = best->fn[p.phase_timers != 0];
    const int block = 64 * best->waves;
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void *)fn, block, 0) != hipSuccess || per_cu < 1)
        return false;
    const Split2D o = split2d(p, *best, depth);
    c->kernel = fn;
    c->block = block;
    c->tile_hx = o.hx;
    c->tile_hy = o.hy;
    c->tile_sx = o.sx;
    c->tile_sy = o.sy;
    c->ntx = o.ntx;
    c->nty = o.nty;
    c->depth = depth;
    c->grid = (int)std::min((long long)std::min(per_cu * c->dev.cus, most), (long long)o.ntx * o.nty);
    return true;
}

}  // namespace cfm
