// 3D Jacobi sweeps as a register pipeline: four sweeps per pass over the field.
//
// A workgroup owns a box of the field: a tile of columns and rows and a chunk of
// planes.  It walks the planes from the top down; at each step one plane of the
// tile comes in, each of the four levels (the fields after 0, 1, 2 and 3 sweeps)
// advances by one plane, and one plane of the field four sweeps on goes out.
// Level j lags one plane behind level j - 1, so level j's newest plane, the two
// before it, and nothing else is needed of it: two planes a level stay in
// registers, and the third goes from one level's result straight into the next
// level's sum.  The tile loads four more columns and rows on every side that has a
// neighbour, and the chunk four more planes at each end.  Every value comes from
// the single-sweep expression, (E + W + (y+1) + (y-1) + (z+1) + (z-1)) / 6 in that
// order: walking down makes z-1, the value that has just been made, the last term.
//
// What bounds it: small fields, the latency of a step (barrier, LDS, four dependent
// levels: 0.8 us for two rows a wavefront) and of the 9 to 12 steps that a pass is at least;
// large fields, vector instructions (10 for an FP64 update, 8 in pairs of columns, 1.5 us of
// the 2.2 us that a step of 4096 columns takes) and then memory (4.1 TB/s at 512^3).  The
// streaming kernels (jacobi.hip) make two sweeps a pass and need long chunks of planes for
// every wavefront: 64^3 FP64 25 us a sweep, here 3.3; 317 x 251 x 190 FP32 78 and 11.6;
// 512^3 FP64 229 and 130.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "jacobi_dev.hpp"
#include "jacobi_host.hpp"

namespace cfm {

namespace {

constexpr int L = 4;        // levels, sweeps of a pass
constexpr unsigned kNowhere = 0xf0000000u;  // an offset beyond every plane: a store that is dropped

template <typename T, int N>
struct VecOf {
    typedef T type __attribute__((ext_vector_type(N)));
};

// `bytes` of memory from p on; accesses beyond them read zeros and write nothing.
template <typename T>
__device__ __forceinline__ auto plane_rsrc(const T *p, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc((void *)p, (short)0, bytes, 0x00020000);
}

// Keeps a uniform value in its scalar register: the compiler would rather work out anew for every row,
// or hold a register for each, what a step's rows share.
template <typename T>
__device__ __forceinline__ void keep(T &v) {
    static_assert(sizeof(T) == 4 || sizeof(T) == 8, "one or two registers");
    unsigned u[sizeof(T) / 4];
    __builtin_memcpy(u, &v, sizeof(T));
#pragma unroll
    for (auto &w : u) {
        w = __builtin_amdgcn_readfirstlane(w);
        asm volatile("" : "+s"(w));
    }
    __builtin_memcpy(&v, u, sizeof(T));
}

template <int AUX, typename T, int VX, typename RSRC>
__device__ __forceinline__ void load_lane(RSRC p, unsigned off, T (&v)[VX]) {
    if constexpr (VX * sizeof(T) == 16) {
        const auto u = __builtin_amdgcn_raw_buffer_load_b128(p, (int)off, 0, AUX);
        __builtin_memcpy(&v, &u, 16);
    } else if constexpr (VX * sizeof(T) == 8) {
        const auto u = __builtin_amdgcn_raw_buffer_load_b64(p, (int)off, 0, AUX);
        __builtin_memcpy(&v, &u, 8);
    } else {
        const unsigned u = __builtin_amdgcn_raw_buffer_load_b32(p, (int)off, 0, AUX);
        __builtin_memcpy(&v, &u, 4);
    }
}
template <int AUX, typename T, int VX, typename RSRC>
__device__ __forceinline__ void store_lane(RSRC p, unsigned off, const T (&v)[VX]) {
    typedef unsigned U2 __attribute__((ext_vector_type(2)));
    typedef unsigned U4 __attribute__((ext_vector_type(4)));
    if constexpr (VX * sizeof(T) == 16) {
        U4 u;
        __builtin_memcpy(&u, &v, 16);
        __builtin_amdgcn_raw_buffer_store_b128(u, p, (int)off, 0, AUX);
    } else if constexpr (VX * sizeof(T) == 8) {
        U2 u;
        __builtin_memcpy(&u, &v, 8);
        __builtin_amdgcn_raw_buffer_store_b64(u, p, (int)off, 0, AUX);
    } else {
        unsigned u;
        __builtin_memcpy(&u, &v, 4);
        __builtin_amdgcn_raw_buffer_store_b32(u, p, (int)off, 0, AUX);
    }
}

// A copy that the compiler cannot see through.  Left to itself it keeps what was loaded where it is and
// loads the next plane elsewhere, and moves the loaded registers back at the end of the loop, which
// waits there for loads that are wanted two steps later.
template <typename T>
__device__ __forceinline__ T copied(T v) {
    T o;
    if constexpr (sizeof(T) == 8)
        asm volatile("v_mov_b64 %0, %1" : "=v"(o) : "v"(v));
    else
        asm volatile("v_mov_b32 %0, %1" : "=v"(o) : "v"(v));
    return o;
}

// What a step looks out for: nothing (all points of the wavefront are updated), columns and rows that
// are on a face or outside the field, or planes and levels too.
enum Kind { kPlain, kFaces, kEnds };

// In the lanes of `lanes`, to[j] becomes from[j].  (A select costs two instructions for each FP64 value
// in every lane; with the moves under another EXEC mask it is one, and the mask changes once a row.)
template <typename T>
__device__ __forceinline__ void hold(unsigned long long lanes, T &t0, T &t1, T &t2, T &t3, T f0, T f1, T f2, T f3) {
    static_assert(L == 4, "a value a level");
    if constexpr (sizeof(T) == 8)
        asm volatile("s_mov_b64 exec, %8\n\tv_mov_b64 %0, %4\n\tv_mov_b64 %1, %5\n\tv_mov_b64 %2, %6\n\tv_mov_b64 %3, %7\n\t"
                     "s_mov_b64 exec, -1"
                     : "+&v"(t0), "+&v"(t1), "+&v"(t2), "+&v"(t3)
                     : "v"(f0), "v"(f1), "v"(f2), "v"(f3), "s"(lanes));
    else
        asm volatile("s_mov_b64 exec, %8\n\tv_mov_b32 %0, %4\n\tv_mov_b32 %1, %5\n\tv_mov_b32 %2, %6\n\tv_mov_b32 %3, %7\n\t"
                     "s_mov_b64 exec, -1"
                     : "+&v"(t0), "+&v"(t1), "+&v"(t2), "+&v"(t3)
                     : "v"(f0), "v"(f1), "v"(f2), "v"(f3), "s"(lanes));
}

// Plane that a wrapped plane index stands for: the interior planes 1..nz-2 repeat.
__device__ __forceinline__ int wrap_plane(int z, int nz) {
    const int p = nz - 2;
    int m = (z - 1) % p;
    if (m < 0) m += p;
    return 1 + m;
}

// What a workgroup works on, the same for all of it.
struct Box {
    int x0, xo, xo_end;  // first column; owned columns
    int y0, yo, yo_end;  // first row; owned rows
    int zo, zo_end;      // owned planes, interior ones only
    bool wrap;           // planes repeat beyond the interior
};

// WAVES wavefronts one above the other, R rows of 64 VX columns each.  The rows just outside a
// wavefront's own come from its neighbours through LDS (two buffers, one workgroup barrier a
// step); x-neighbours are DPP shifts.
template <typename T, int VX, int R, int WAVES>
struct Pipe3D {
    typedef typename VecOf<T, VX>::type V;
    static constexpr int C = 64 * VX, H = R * WAVES;
    // planes that are loaded ahead of their step
    static constexpr int AHEAD = R * VX * sizeof(T) >= 32 ? 2 : 4;
    typedef T Edge[2][L][WAVES][2][C];

    T a[2][L][R][VX];  // [step parity]: each level's newest plane, and at the other parity the one before
    T in[AHEAD][R][VX];
    // rows that are stored or not together: boxes own whole groups (a halo of L rows; rows beyond the
    // field's last are offsets beyond the plane)
    static constexpr int kGroup = R < L ? R : L;
    static_assert(R % kGroup == 0 && L % kGroup == 0, "a halo ends between two groups");

    unsigned ld, st, st1, pitch;  // the first row's offset in a plane (st: kNowhere where the lane stores nothing)
    int wave, lane;
    unsigned long long xin[VX], xown[VX];  // lanes whose column is updated; and is this box's
    unsigned long long fixed[VX];          // lanes whose column is a face
    unsigned live_rows;      // rows that are updated, a bit each
    int plain_lo, plain_hi;  // with top in [plain_lo, plain_hi] no level is at an end of the planes
    bool own[R / kGroup];    // the group's rows are this box's
    bool odd;

    // the plane z as a buffer to load from
    __device__ __forceinline__ auto from(const JacobiArgs &A, const T *src, size_t plane, int z) const {
        // A lane of two columns may start on a plane's last element and reach into the next plane.  (The
        // field's last plane has none; its last element, a corner, then reads as zero and is not used.)
        const int bytes = (int)(plane * sizeof(T)) + (VX > 1 && z < A.nz - 1 ? (VX - 1) * (int)sizeof(T) : 0);
        const bool there = z >= 0 && z < A.nz;
        return plane_rsrc(src + (there ? (size_t)z * plane : 0), there ? bytes : 0);
    }
    template <bool THROUGH, typename RSRC>
    __device__ __forceinline__ void load(RSRC p, int r, T (&v)[VX]) {
        load_lane<THROUGH ? kSc1 : 0, T, VX>(p, ld + r * pitch, v);
    }

    // The order of a step's rows: some inner rows first, which need nothing of the neighbours, then the
    // outer two, which are published at once, then the other inner rows.
    static constexpr int kOuter = (R - 2) / 2;
    static constexpr __device__ __forceinline__ int nth_row(int i) {
        return i < kOuter ? i + 1 : i == kOuter ? 0 : i == kOuter + 1 ? R - 1 : i - 1;
    }

    template <Kind KIND, bool THROUGH, typename RSRC>
    __device__ __forceinline__ void store(RSRC p, int r, const T (&v)[VX]) {
        constexpr int AUX = THROUGH ? kSc1 : 0;
        store_lane<AUX, T, VX>(p, st + r * pitch, v);
        if constexpr (KIND != kPlain && VX > 1) {
            if (odd) {  // the field's last column is a lane's first
                const T one[1] = {v[0]};
                store_lane<AUX, T, 1>(p, st1 + r * pitch, one);
            }
        }
    }

    // The neighbours' rows are read a row before they are used, which hides the LDS, but for the shape
    // whose registers do not allow it.
    static constexpr bool kEarly = kOuter > 0 && sizeof(V) < 16;

    // One step's sums and stores.  top: the plane index of level 0's incoming plane, fresh.
    template <int PAR, Kind KIND, bool NORM, bool THROUGH, typename RSRC>
    __device__ __forceinline__ void sums(const JacobiArgs &A, const Box &B, T *dst, size_t plane, int top, int steps,
                                         RSRC ahead, T (&fresh)[R][VX], Edge &edge, double &acc) {
        const T c = T(1) / T(6);
        T(&cur)[L][R][VX] = a[PAR];
        T(&old)[L][R][VX] = a[1 - PAR];
        const int zout = top + L;  // the plane that leaves
        const bool out = zout >= B.zo && zout < B.zo_end;
        const int whole = (int)(plane * sizeof(T));
        T *to = dst + (out ? (size_t)zout * plane : 0);
        keep(to);
        int bytes[R / kGroup];  // of the plane, for the rows that are stored
#pragma unroll
        for (int g = 0; g < R / kGroup; ++g) {
            bytes[g] = out && own[g] ? whole : 0;
            keep(bytes[g]);
        }
        V up[L], dn[L];
        unsigned long long live[L][VX];  // lanes whose column is updated, none where the level's plane is not
        unsigned rows = 0;               // rows that are updated, a bit each
        bool copy = false;               // with periodic planes: the plane that leaves is a halo plane too
        if constexpr (KIND == kFaces) {
            rows = live_rows;
            keep(rows);
        }
        if constexpr (KIND == kEnds) {
#pragma unroll
            for (int j = 0; j < L; ++j)
#pragma unroll
                for (int e = 0; e < VX; ++e) {
                    live[j][e] = j < steps && (B.wrap || (top + j + 1 >= 1 && top + j + 1 <= A.nz - 2)) ? xin[e] : 0;
                    keep(live[j][e]);
                }
            rows = live_rows;
            keep(rows);
            copy = A.bc == CFM_BC_PERIODIC && out && (zout == 1 || zout == A.nz - 2);
        }
#pragma unroll
        for (int i = 0; i < R; ++i) {
            const int r = nth_row(i);
            // (constant conditions; the tile's own outer rows have no neighbour: any value does, they are
            // stale already)
            if (i == (kEarly ? kOuter - 1 : kOuter))
#pragma unroll
                for (int j = 0; j < L; ++j)
                    up[j] = *reinterpret_cast<const V *>(&edge[PAR][j][wave > 0 ? wave - 1 : 0][1][lane * VX]);
            if (i == (kEarly ? kOuter : kOuter + 1))
#pragma unroll
                for (int j = 0; j < L; ++j)
                    dn[j] = *reinterpret_cast<const V *>(&edge[PAR][j][wave < WAVES - 1 ? wave + 1 : wave][0][lane * VX]);
            T sum[L][VX];
#pragma unroll
            for (int j = 0; j < L; ++j) {
                const T west = lane_up1z(cur[j][r][VX - 1]);
                const T east = lane_dn1z(cur[j][r][0]);
#pragma unroll
                for (int e = 0; e < VX; ++e) {
                    const T E = e < VX - 1 ? cur[j][r][e < VX - 1 ? e + 1 : e] : east;
                    const T W = e > 0 ? cur[j][r][e > 0 ? e - 1 : e] : west;
                    const T N = r < R - 1 ? cur[j][r < R - 1 ? r + 1 : r][e] : dn[j][e];
                    const T S = r > 0 ? cur[j][r > 0 ? r - 1 : r][e] : up[j][e];
                    sum[j][e] = E + W + N + S + old[j][r][e];
                }
            }
            T t[VX];
#pragma unroll
            for (int e = 0; e < VX; ++e) t[e] = copied(fresh[r][e]);
            // the row of a later plane takes its place at once: spread over the step, the loads do not
            // hold up the wavefronts that issue them
            load<THROUGH>(ahead, r, fresh[r]);
            const unsigned long long row = rows >> r & 1 ? ~0ull : 0;  // uniform
#pragma unroll
            for (int j = 0; j < L; ++j) {
#pragma unroll
                for (int e = 0; e < VX; ++e) {
                    const T n = c * (sum[j][e] + t[e]);
                    const T v = KIND != kEnds || __builtin_amdgcn_inverse_ballot_w64(live[j][e] & row) ? n : cur[j][r][e];
                    if (NORM && j == 0) {
                        const double d = (double)n - (double)cur[j][r][e];
                        const bool count = own[r / kGroup] && top + 1 >= B.zo && top + 1 < B.zo_end;  // uniform
                        const double dd = __builtin_amdgcn_inverse_ballot_w64(count ? xown[e] & row : 0) ? d : 0.0;
                        acc += dd * dd;
                        asm volatile("" : "+v"(acc));  // (summed here: left free, the squares wait in registers)
                    }
                    old[j][r][e] = t[e];
                    t[e] = v;
                }
            }
            if constexpr (KIND == kFaces) {
#pragma unroll
                for (int e = 0; e < VX; ++e)
                    hold(fixed[e] | ~row, old[1][r][e], old[2][r][e], old[3][r][e], t[e], cur[0][r][e], cur[1][r][e],
                         cur[2][r][e], cur[3][r][e]);
            }
            store<KIND, THROUGH>(plane_rsrc(to, bytes[r / kGroup]), r, t);
            if (KIND == kEnds && copy) {
                if (zout == A.nz - 2) store<KIND, THROUGH>(plane_rsrc(dst, bytes[r / kGroup]), r, t);
                if (zout == 1)
                    store<KIND, THROUGH>(plane_rsrc(dst + (A.nz - 1) * plane, bytes[r / kGroup]), r, t);
            }
            if (i == kOuter + 1) {  // (constant)
#pragma unroll
                for (int j = 0; j < L; ++j) {
                    V lo, hi;
#pragma unroll
                    for (int e = 0; e < VX; ++e) {
                        lo[e] = old[j][0][e];
                        hi[e] = old[j][R - 1][e];
                    }
                    *reinterpret_cast<V *>(&edge[1 - PAR][j][wave][0][lane * VX]) = lo;
                    *reinterpret_cast<V *>(&edge[1 - PAR][j][wave][1][lane * VX]) = hi;
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    // One step.
    template <int PAR, Kind KIND, bool NORM, bool THROUGH>
    __device__ __forceinline__ void step(const JacobiArgs &A, const Box &B, const T *src, T *dst, size_t plane, int &top,
                                         int &next, int steps, T (&fresh)[R][VX], Edge &edge, double &acc) {
        // (beyond the chunk's last plane the pipeline only runs out: what is loaded is not used)
        sums<PAR, KIND, NORM, THROUGH>(A, B, dst, plane, top, steps, from(A, src, plane, next), fresh, edge, acc);
        __syncthreads();
        --top;
        --next;
        if (B.wrap && next <= 0) next = A.nz - 2;
    }

    // One box, one pass; KIND: what the steps away from the ends look out for (kEnds: there are none).
    template <Kind KIND, bool NORM, bool THROUGH>
    __device__ __forceinline__ void pass(const JacobiArgs &A, const Box &B, const T *src, T *dst, int steps, Edge &edge,
                                         double &acc) {
        const int nx = A.nx, ny = A.ny;
        const size_t plane = (size_t)nx * ny;
        lane = threadIdx.x & 63;
        wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        const int x = B.x0 + lane * VX, y = B.y0 + wave * R;
        const int row_lo = min(max(1 - y, 0), R), row_hi = min(max(ny - 1 - y, 0), R);
        live_rows = (1u << row_hi) - (1u << min(row_lo, row_hi));
#pragma unroll
        for (int g = 0; g < R / kGroup; ++g) own[g] = y + g * kGroup >= B.yo && y + g * kGroup < B.yo_end;
#pragma unroll
        for (int e = 0; e < VX; ++e) {
            xin[e] = __ballot(x + e >= 1 && x + e <= nx - 2);
            fixed[e] = __ballot(x + e == 0 || x + e == nx - 1);
            xown[e] = xin[e] & __ballot(x + e >= B.xo && x + e < B.xo_end);
        }
        // with top, ends among the levels' planes top + 1 .. top + L
        plain_lo = B.wrap ? 2 - L : 0;  // (wrapped, only the copies of planes 1 and nz - 2 need the masked steps)
        plain_hi = A.nz - 3 - (B.wrap ? L : L - 1);
        // (rows beyond the field's last are offsets beyond the plane; no box starts before its first)
        pitch = (unsigned)nx * sizeof(T);
        ld = (unsigned)y * pitch + (unsigned)x * sizeof(T);
        const bool mine = x >= B.xo && x < B.xo_end, cut = VX > 1 && x == nx - 1;
        st = mine && !cut ? ld : kNowhere;
        st1 = mine && cut ? ld : kNowhere;
        odd = VX > 1 && B.xo_end == nx && nx % VX != 0;
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
            for (int j = 0; j < L; ++j)
#pragma unroll
                for (int r = 0; r < R; ++r)
#pragma unroll
                    for (int e = 0; e < VX; ++e) a[p][j][r][e] = T(0);
        int top = B.zo_end - 1 + L;                       // level 0's incoming plane
        int next = B.wrap ? wrap_plane(top, A.nz) : top;  // the plane to load
        const int n = B.zo_end - B.zo + 2 * L;
#pragma unroll
        for (int s = 0; s < AHEAD; ++s) {
            const auto p = from(A, src, plane, next);
#pragma unroll
            for (int i = 0; i < R; ++i) {
                load<THROUGH>(p, nth_row(i), in[s][nth_row(i)]);
                // (in this order: the loop's waits count on it, and take the shorter count of its entries)
                __builtin_amdgcn_sched_barrier(0);
            }
            --next;
            if (B.wrap && next == 0) next = A.nz - 2;
        }
        // Steps [k1, k2) look out for no ends, in whole rounds of the loads' ring.  (Loops, not a choice within one:
        // two bodies on one set of registers would not fit.)
        int k = 0, k1 = n, k2 = n;
        if (KIND != kEnds) {
            const int lo = (max(top - plain_hi, 0) + AHEAD - 1) / AHEAD * AHEAD;
            const int hi = min(n, top - plain_lo + 1) / AHEAD * AHEAD;
            if (lo < hi) k1 = lo, k2 = hi;
        }
        for (int part = 0; part < 2; ++part) {
            steps_to<kEnds, NORM, THROUGH>(A, B, src, dst, plane, top, next, steps, k, k1, n, edge, acc);
            if constexpr (KIND != kEnds)
                steps_to<KIND, NORM, THROUGH>(A, B, src, dst, plane, top, next, steps, k, k2, n, edge, acc);
            k1 = n;
        }
    }

    // steps k .. to - 1, of n
    template <Kind KIND, bool NORM, bool THROUGH>
    __device__ __forceinline__ void steps_to(const JacobiArgs &A, const Box &B, const T *src, T *dst, size_t plane,
                                             int &top, int &next, int steps, int &k, int to, int n, Edge &edge,
                                             double &acc) {
        for (; k < to; k += AHEAD) {
#pragma unroll
            for (int s = 0; s < AHEAD; s += 2) {
                if (s > 0 && k + s >= n) break;
                step<0, KIND, NORM, THROUGH>(A, B, src, dst, plane, top, next, steps, in[s], edge, acc);
                step<1, KIND, NORM, THROUGH>(A, B, src, dst, plane, top, next, steps, in[s + 1], edge, acc);
            }
        }
    }
};

// THROUGH: past the L2 on both sides, for fields of few boxes, whose passes are short enough for the
// barrier's fences to count.
template <typename T, int VX, int R, int WAVES, bool THROUGH, bool TIMED>
__global__ void __launch_bounds__(64 * WAVES, R >= 4 && WAVES <= 8 ? 2 : 4) jacobi3d_pipe_kernel(JacobiArgs A) {
    typedef Pipe3D<T, VX, R, WAVES> Pipe;
    __shared__ typename Pipe::Edge edge;
    __shared__ double lds[WAVES];
    __shared__ unsigned long long clk_lds[kClockWords];
    PhaseClock<TIMED> clk{clk_lds};
    clk.start();
    const bool periodic = A.bc == CFM_BC_PERIODIC;
    const int tiles = A.ntx * A.nty, units = tiles * A.chunks;
    const int first = xcd_block_id();
    unsigned int epoch = 0;
    int turn = 0;
    for (int k = 0; k < A.niter; ++turn) {
        // Periodic planes: the first sweep reads the caller's halo planes, which need not be copies
        // of the opposite ends yet; from the second on the planes simply repeat.
        Box B;
        B.wrap = periodic && k > 0;
        const int steps = jacobi_pipe_steps(k, A.niter, A.depth, A.norm_every, periodic);
        const bool norm = A.norm_every > 0 && k % A.norm_every == 0;
        const T *src = static_cast<const T *>((turn & 1) ? A.buf1 : A.buf0);
        T *dst = static_cast<T *>((turn & 1) ? A.buf0 : A.buf1);
        double acc = 0.0;
        for (int u = first; u < units; u += gridDim.x) {
            const int ch = u / tiles, t = u - ch * tiles;
            const int ty = t / A.ntx, tx = t - ty * A.ntx;
            B.x0 = tx * A.tile_sx;
            B.xo = tx > 0 ? B.x0 + A.tile_hx : 0;
            B.xo_end = tx < A.ntx - 1 ? B.x0 + Pipe::C - A.tile_hx : A.nx;
            B.y0 = ty * A.tile_sy;
            B.yo = ty > 0 ? B.y0 + A.tile_hy : 0;
            B.yo_end = ty < A.nty - 1 ? B.y0 + Pipe::H - A.tile_hy : A.ny;
            B.zo = 1 + ch * A.chunk_len;
            B.zo_end = min(B.zo + A.chunk_len, A.nz - 1);
            Pipe p;
            // (the wavefronts of a box may take different ones: they do the same number of steps)
            const int y = B.y0 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * R;
            if (norm)
                p.template pass<kEnds, true, THROUGH>(A, B, src, dst, steps, edge, acc);
            else if (steps < L)
                p.template pass<kEnds, false, THROUGH>(A, B, src, dst, steps, edge, acc);
            else if (B.x0 < 1 || B.x0 + Pipe::C > A.nx - 1 || y < 1 || y + R > A.ny - 1)
                p.template pass<kFaces, false, THROUGH>(A, B, src, dst, steps, edge, acc);
            else
                p.template pass<kPlain, false, THROUGH>(A, B, src, dst, steps, edge, acc);
        }
        if (norm) {
            const double sum = block_sum_waves<WAVES>(acc, lds);
            if (threadIdx.x == 0) A.norm_part[(size_t)(k / A.norm_every) * gridDim.x + blockIdx.x] = sum;
        }
        k += steps;
        if (k < A.niter) {
            if (!pass_barrier<THROUGH>(A, epoch, clk)) return;
        }
    }
    clk.mark(CFM_PHASE_SPMV);
    clk.flush(A.timers);
}

// A shape and what it measured: microseconds of a step with one workgroup on a CU and with as many as
// fit, the rate at which it moves fields (each pass reads one array and writes the other) that
// the 256 MB of memory-side cache do not hold, and how much longer the steps of a pass with a norm, and of
// one of fewer than L sweeps, take than a plain pass's (both are masked throughout).
struct Shape3D {
    int vx, r, waves, per_cu;
    bool through;
    double step_us, full_us, tb_s, norm, part;
    KernelFn fn[2];  // [timed]
};

template <typename T, int VX, int R, int WAVES, bool THROUGH>
Shape3D shape3d(int per_cu, double step_us, double full_us, double tb_s, double norm, double part) {
    return {VX, R, WAVES, per_cu, THROUGH, step_us, full_us, tb_s, norm, part,
            {(KernelFn)jacobi3d_pipe_kernel<T, VX, R, WAVES, THROUGH, false>,
             (KernelFn)jacobi3d_pipe_kernel<T, VX, R, WAVES, THROUGH, true>}};
}

// tiles of `span` columns (or rows) that n of them need, neighbours overlapping by a halo each
int tiles_along(int n, int span) { return n <= span ? 1 : (n - span + span - 2 * L - 1) / (span - 2 * L) + 1; }

// Estimated microseconds of one pass: the chunk's planes and 2 L more to fill and empty the pipeline,
// for each round of boxes on `most` workgroups or as many as fit; the device-wide barrier, the first loads and
// the last stores, 5 us.
double pass_us(const cfm_jacobi_params &p, const Shape3D &s, int tiles, int chunks, int cus, int most,
               double longer = 1.0) {
    const int len = (p.nz - 2 + chunks - 1) / chunks;
    const double units = (double)tiles * chunks;
    const double rounds = std::ceil(units / std::min(cus * s.per_cu, most));
    const double moved = 2.0 * (p.prec == CFM_F64 ? 8 : 4) * p.nx * (double)p.ny * p.nz;
    return 5.0 + std::max(rounds * (len + 2 * L) * (units > cus ? s.full_us : s.step_us) * longer,
                          moved > 2.0e8 ? moved / (s.tb_s * 1e6) : 0.0);
}

// Estimated microseconds of `sweeps` sweeps from the start of a run.
double run_us(const cfm_jacobi_params &p, const Shape3D &s, int tiles, int chunks, int cus, int most, int sweeps) {
    const double plain = pass_us(p, s, tiles, chunks, cus, most), norm = pass_us(p, s, tiles, chunks, cus, most, s.norm),
                 part = pass_us(p, s, tiles, chunks, cus, most, s.part);
    double us = 0.0;
    for (int k = 0; k < sweeps;) {
        const int steps = jacobi_pipe_steps(k, sweeps, L, p.norm_every, p.bc == CFM_BC_PERIODIC);
        us += p.norm_every > 0 && k % p.norm_every == 0 ? norm : steps < L ? part : plain;
        k += steps;
    }
    return us;
}

// The same of the streaming kernels (jacobi.hip), as configured in c: a step a plane and two more to warm
// up, for each round of units; norms cost them nothing.  Microseconds of a step as measured, FP64 and FP32:
// two sweeps a pass 1.75 and 2.1 (rows of whole vectors), 2.1 and 2.4 (x tiles), 2.55 and 5.9 (other rows),
// 1.25, 1.6, 2.0 and 1.45, 1.7, 4.8 where a run's last pass has one; the one-sweep kernels 2.45 and 3.75
// (FP32 rows that are not whole vectors: 7.3 a tile of 1024 columns).
// At 512^3, 300^3, 128^3 and 317 x 251 x 190 FP64 this gives 473, 179, 40 and 130 us for two sweeps, measured 468,
// 173, 41 and 125.
double streaming_us(const cfm_jacobi_params &p, const JacobiConfig &c, int sweeps) {
    const bool f64 = p.prec == CFM_F64, periodic = p.bc == CFM_BC_PERIODIC;
    const bool aligned = (size_t)p.nx * c.elem_size % 16 == 0, tiles_x = c.ntx > 1;
    const double units = (double)c.ntx * c.nty * c.chunks, rounds = std::ceil(units / c.grid);
    const double steps = rounds * (c.chunk_len + 2), moved = 2.0 * c.elem_size * p.nx * (double)p.ny * p.nz;
    if (!c.t2) {
        const double step = f64 ? 2.45 : aligned ? 3.75 : 7.3 * std::min(1.0, p.nx / 1024.0);
        return sweeps * (3.0 + std::max(steps * step, moved / 4.6e6));
    }
    const double slow = periodic ? 1.06 : 1.0;  // (the copies of the opposite planes)
    const double two = slow * (!aligned ? (f64 ? 2.55 : 5.9) : tiles_x ? (f64 ? 2.1 : 2.4) : (f64 ? 1.75 : 2.1));
    const double one = slow * (!aligned ? (f64 ? 2.0 : 4.8) : tiles_x ? (f64 ? 1.6 : 1.7) : (f64 ? 1.25 : 1.45));
    return sweeps / 2 * ((periodic ? 12.0 : 5.0) + std::max(steps * two, moved / 4.6e6)) +
           sweeps % 2 * ((sweeps > 1 ? 5.0 : 0.0) + std::hypot(steps * one, moved / 5.5e6));
}

}  // namespace

bool jacobi_pipe_configure(const cfm_jacobi_params &p, JacobiConfig *c) {
    const bool f64 = p.prec == CFM_F64;
    // 32-bit offsets within a plane and a tile's rows beyond it, and a wavefront's rows beyond kNowhere
    const double pitch = (double)p.nx * (f64 ? 8 : 4);
    if (p.nz < 3 || pitch * p.ny >= 2.0e9 || pitch >= 1.6e7) return false;
    // Few rows a wavefront for small fields (a step is then shorter, and more boxes share the field),
    // many for large ones (less halo).  FP64: 16-byte lanes move a large field faster than 8-byte
    // ones (512^3: 130 us a sweep against 141 for 4 rows of 8-byte lanes and 165 for 8, whose 64
    // rows at a pitch of 4096 bytes fall on few of the caches' channels), but waste half their
    // columns on rows of up to 64 points.  Going past the L2 costs nothing where a field's boxes are read once a
    // pass, and the barrier is then 3.6 us shorter.
    static const Shape3D s64[] = {shape3d<double, 1, 2, 8, true>(2, 0.83, 1.22, 3.1, 1.3, 1.0),
                                  shape3d<double, 1, 4, 8, true>(1, 1.22, 1.22, 3.8, 1.3, 1.0),
                                  shape3d<double, 1, 8, 8, false>(1, 2.2, 2.2, 3.1, 1.3, 1.0),
                                  shape3d<double, 2, 4, 8, false>(1, 2.2, 2.2, 4.1, 1.15, 1.15)};
    static const Shape3D s32[] = {shape3d<float, 1, 2, 8, true>(3, 0.6, 1.05, 3.1, 1.65, 1.0),
                                  shape3d<float, 2, 2, 8, true>(2, 0.8, 1.23, 3.1, 1.65, 1.0),
                                  shape3d<float, 2, 4, 8, true>(1, 1.2, 1.2, 3.3, 1.65, 1.0),
                                  shape3d<float, 2, 8, 8, false>(1, 2.4, 2.4, 3.4, 1.65, 1.0)};
    const Shape3D *best = nullptr;
    int chunks = 0, ntx = 0, nty = 0;
    double best_us = 1e30;
    const int interior = p.nz - 2, most = jacobi_norm_workgroups(*c);
    for (const Shape3D &s : f64 ? s64 : s32) {
        const int tx = tiles_along(p.nx, 64 * s.vx), ty = tiles_along(p.ny, s.r * s.waves);
        if ((double)tx * ty * interior > 1e9) continue;
        for (int ch = 1; ch <= std::min(interior, 2048); ++ch) {  // (some rounds of what fits at once, at any size)
            const double us = pass_us(p, s, tx * ty, ch, c->dev.cus, most);
            if (us < best_us) best_us = us, best = &s, chunks = ch, ntx = tx, nty = ty;
        }
    }
    if (!best) return false;
    // The streaming kernels make two sweeps a pass whatever the run: they are the faster ones where a run is
    // short, where norms are frequent (a sweep whose norm is wanted starts a pass) and where planes are
    // few.  512^3 FP64, us, streaming / pipeline: 2 sweeps 542 / 657, 4 of periodic planes 1122 / 1305, 40 with a
    // norm every 5 9416 / 9312, every 4 9368 / 6215; 3 x 512 x 512, 40 sweeps 251 / 181, with a norm every 3
    // 255 / 277.  (Within the estimates' spread of 5 % the streaming kernels keep a run.)
    const int sweeps = std::min(p.niter, 4096);
    if (1.05 * run_us(p, *best, ntx * nty, chunks, c->dev.cus, most, sweeps) > streaming_us(p, *c, sweeps)) return false;
    KernelFn fn = best->fn[p.phase_timers != 0];
    const int block = 64 * best->waves;
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void *)fn, block, 0) != hipSuccess || per_cu < 1)
        return false;
    c->kernel = fn;
    c->block = block;
    c->tile_hx = c->tile_hy = L;
    c->tile_sx = 64 * best->vx - 2 * L;
    c->tile_sy = best->r * best->waves - 2 * L;
    c->ntx = ntx;
    c->nty = nty;
    c->chunk_len = (interior + chunks - 1) / chunks;
    c->chunks = (interior + c->chunk_len - 1) / c->chunk_len;
    c->depth = L;
    c->pipe = true;
    c->grid = (int)std::min((long long)std::min(per_cu * c->dev.cus, most), (long long)ntx * nty * c->chunks);
    return true;
}

}  // namespace cfm
