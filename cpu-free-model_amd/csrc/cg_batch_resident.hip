// Batched CG with every system resident: while a system is solved, its matrix and vectors are in the
// registers of its own team of workgroups, one 1024-row chunk each.
//
// The general batch kernel (cg_batch.hip) streams every active system through memory once per
// iteration under one device-wide barrier.  The systems are independent, so here a team iterates at
// its own pace under a barrier of its own, and when its system is done its workgroups go on to their
// next one.  Same recurrences, row map and trees, so a member has the bits of its solo solve.
//
// A workgroup of 256 threads holds 232 registers a lane: two to a CU, whose latencies overlap.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <numeric>

#include "cg_batch_args.hpp"
#include "cg_resident.hpp"

namespace cfm {

__global__ void reset_team_kernel(TeamSync *t, unsigned long long limit_ticks) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) {
        t->abort = 0;
        t->spin_limit_ticks = limit_ticks;
    }
    if (i < kMaxTeamGrid) {
        t->arrive[i] = 0;
        t->go[16 * i] = 0;
    }
}

namespace {

// A team: workgroups base .. base + size - 1, this one is `me`.  The epoch's upper half is the round,
// so a workgroup's words only ever grow, whichever team it is in.
struct Team {
    TeamSync *s;
    int me, base, size;
    unsigned long long epoch;
};

// The sum of the launch's arrival words (zeros beyond its workgroups).  They only grow, and do as long as
// any team of several workgroups iterates.
__device__ __forceinline__ unsigned long long arrivals(const TeamSync *s) {
    unsigned long long sum = 0;
    for (int b = 0; b < kMaxTeamGrid; ++b)
        sum += __hip_atomic_load(&s->arrive[b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return sum;
}

// grid_barrier_through for one team: arrivals to its first workgroup, which releases every member on a
// line of its own (a line that only that member reads: no release of an earlier team can be late).
// At the first barrier of a later round members may still be at their previous systems, which have several
// workgroups (batch_resident_schedule), for as long as those take: that wait's clock starts anew while the
// launch makes progress.  (All others wait for at most an iteration.  A word of a workgroup alone in its team
// would cost it 3 to 6 % of an iteration.)
__device__ __forceinline__ bool team_barrier(Team &T) {
    __shared__ int s_abort;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    const unsigned long long e = ++T.epoch;
    if (T.size == 1) return true;
    TeamSync *s = T.s;
    const unsigned long long limit = s->spin_limit_ticks;
    const bool patient = (unsigned)e == 1 && (e >> 32) > 1;
    int ab = 0;
    if (threadIdx.x == 0) {
        s_abort = 0;
        __hip_atomic_store(&s->arrive[T.me], e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    const bool gather = T.me == T.base;
    if (gather) __syncthreads();
    if (gather || threadIdx.x == 0) {
        unsigned long long t0 = __builtin_amdgcn_s_memrealtime(), seen = 0;
        const unsigned long long *first = gather ? &s->arrive[T.base + threadIdx.x] : &s->go[16 * T.me];
        const int count = gather ? T.size - (int)threadIdx.x : 1;
        for (int b = 0; b < count && !ab; b += blockDim.x) {
            while (__hip_atomic_load(first + b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < e) {
                const bool stop = __hip_atomic_load(&s->abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                const bool late = spin_expired(t0, limit);
                if (late && patient && !stop) {
                    const unsigned long long now = arrivals(s);
                    if (now != seen) {
                        seen = now;
                        t0 = __builtin_amdgcn_s_memrealtime();
                        continue;
                    }
                }
                if (late || stop) {
                    __hip_atomic_store(&s->abort, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    ab = 1;
                    break;
                }
                __builtin_amdgcn_s_sleep(1);
            }
        }
        if (ab) s_abort = 1;
    }
    if (gather) {
        __syncthreads();
        if (!s_abort)
            for (int b = threadIdx.x; b < T.size; b += blockDim.x)
                __hip_atomic_store(&s->go[16 * (T.base + b)], e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    asm volatile("" ::: "memory");
    return s_abort == 0;
}

// The system a team solves, as buffers of its own rows (offset 0 is its first row).
struct System {
    int sy, rows, chunk, first_chunk, chunks;
    int off;  // byte offset of this thread's first row
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_of(const System &Y, const double *v) {
    return __builtin_amdgcn_make_buffer_rsrc((void *)(v + (size_t)Y.first_chunk * kChunk), (short)0, Y.rows * 8,
                                             0x00020000);
}
__device__ __forceinline__ void read_rows(const System &Y, const double *from, double (&v)[kRows]) {
    const auto rsrc = rows_of(Y, from);
#pragma unroll
    for (int i = 0; i < kRows; ++i)
        v[i] = __builtin_bit_cast(double,
                                  __builtin_amdgcn_raw_buffer_load_b64(rsrc, Y.off + i * kThreads * 8, 0, kSc1));
}
__device__ __forceinline__ void write_rows(const System &Y, double *to, const double (&v)[kRows]) {
    typedef unsigned int U2 __attribute__((ext_vector_type(2)));
    const auto rsrc = rows_of(Y, to);
#pragma unroll
    for (int i = 0; i < kRows; ++i)
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(U2, v[i]), rsrc, Y.off + i * kThreads * 8, 0, kSc1);
}
template <int W>
__device__ __forceinline__ void gather(const System &Y, const Entries<double, double, W> &M, const double *x,
                                       double (&g)[kRows][W]) {
    M.gather(x + (size_t)Y.first_chunk * kChunk, Y.rows, g);
}

template <int K>
__device__ __forceinline__ void put(const BatchArgs &A, const System &Y, double (&v)[K], const int (&which)[K],
                                    double *lds) {
    sub_sums<1, K>(v, lds);
    if (threadIdx.x == 0)
#pragma unroll
        for (int k = 0; k < K; ++k) store_wt(&A.part[which[k] * A.total_chunks + Y.chunk], v[k]);
}
template <int K>
__device__ __forceinline__ void get(const BatchArgs &A, const System &Y, const int (&which)[K], double (&v)[K],
                                    double *lds) {
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] = 0.0;
    for (int j = threadIdx.x; j < Y.chunks; j += kThreads)
#pragma unroll
        for (int k = 0; k < K; ++k)
            v[k] = v[k] + load_through(&A.part[which[k] * A.total_chunks + Y.first_chunk + j]);
    sub_sums<1, K>(v, lds);
}

// One system to its end; false when the launch is aborting.  Rows of the last chunk beyond the system
// take part as zeros.  part: [0,1] delta, [2,3] gamma by iteration parity, [4] <b,b>.
template <int W>
__device__ __forceinline__ bool solve_system(const BatchArgs &A, const System &Y, Team &T, double *lds) {
    Entries<double, double, W> M;
    M.load(A.A, Y.chunk, threadIdx.x, true, Y.first_chunk * kChunk);
    const bool owner = Y.chunk == Y.first_chunk && threadIdx.x == 0;
    double x[kRows], r[kRows], z[kRows], s[kRows], p[kRows], w[kRows], g[kRows][W];
    double two[2];
    {
        double b[kRows];
        read_rows(Y, A.x0, x);
        read_rows(Y, A.b, b);
        gather(Y, M, A.x0, g);
        two[0] = two[1] = 0.0;
#pragma unroll
        for (int i = 0; i < kRows; ++i) {
            r[i] = fma(-1.0, M.row_sum(i, g), b[i]);
            two[0] = fma(r[i], r[i], two[0]);
            two[1] = fma(b[i], b[i], two[1]);
        }
    }
    write_rows(Y, A.r, r);
    put<2>(A, Y, two, {1, 4}, lds);  // (delta buffer 1 is free until iteration 0 writes it)
    if (!team_barrier(T)) return false;
    get<2>(A, Y, {1, 4}, two, lds);
    const double bb = two[1];
    const double *from = A.r;
    if (A.x0_guard) {
        const bool reject = !(two[0] <= bb);  // a non-finite residual is rejected too
        if (owner) A.x0_rejected[Y.sy] = reject ? 1 : 0;
        if (reject) {
            from = A.b;
            read_rows(Y, A.b, r);
#pragma unroll
            for (int i = 0; i < kRows; ++i) x[i] = 0.0;
        }
    }
    // (one gather from a pointer that the compiler knows to be uniform)
    const unsigned long long fp = (unsigned long long)from;
    gather(Y, M,
           (const double *)((unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(fp >> 32)) << 32 |
                            (unsigned)__builtin_amdgcn_readfirstlane((int)fp)),
           g);
    two[0] = two[1] = 0.0;
#pragma unroll
    for (int i = 0; i < kRows; ++i) {
        w[i] = M.row_sum(i, g);
        z[i] = s[i] = p[i] = 0.0;
        two[0] = fma(r[i], r[i], two[0]);
        two[1] = fma(r[i], w[i], two[1]);
    }
    write_rows(Y, A.w[0], w);
    put<2>(A, Y, two, {0, 2}, lds);
    if (!team_barrier(T)) return false;
    const double thr = A.tol > 0.0 ? A.tol * A.tol * bb : 0.0;
    double alpha = 0.0, beta = 0.0, delta_prev = 0.0;
    int k = 0, st = kActive;
    for (;;) {
        const int buf = __builtin_amdgcn_readfirstlane(k & 1);
        gather(Y, M, A.w[buf], g);
        get<2>(A, Y, {0 + buf, 2 + buf}, two, lds);
        const double delta = two[0], gam = two[1];
        if (owner && A.hist && k < A.hist_cap) A.hist[(size_t)Y.sy * A.hist_cap + k] = delta;
        if (delta <= thr) {
            st = kConverged;
            break;
        }
        if (k >= A.max_iter) {
            st = kMaxIter;
            break;
        }
        double denom;
        if (A.quirk ? (k > 1) : (k > 0)) {
            beta = delta / delta_prev;
            denom = gam - (beta / alpha) * delta;
        } else {
            beta = 0.0;
            denom = gam;
        }
        if (!(denom > 0.0) || !is_finite(denom)) {
            st = kBreakdown;
            break;
        }
        alpha = delta / denom;
        two[0] = two[1] = 0.0;
#pragma unroll
        for (int i = 0; i < kRows; ++i) {
            z[i] = fma(beta, z[i], M.row_sum(i, g));
            s[i] = fma(beta, s[i], w[i]);
            p[i] = fma(beta, p[i], r[i]);
            x[i] = fma(alpha, p[i], x[i]);
            r[i] = fma(-alpha, s[i], r[i]);
            w[i] = fma(-alpha, z[i], w[i]);
            two[0] = fma(r[i], r[i], two[0]);
            two[1] = fma(r[i], w[i], two[1]);
        }
        write_rows(Y, A.w[1 - buf], w);
        put<2>(A, Y, two, {1 - buf, 3 - buf}, lds);
        if (!team_barrier(T)) return false;
        delta_prev = delta;
        ++k;
    }
    write_rows(Y, A.x, x);
    if (owner) {
        A.fin[Y.sy] = k;
        A.status[Y.sy] = st;
        A.iters[Y.sy] = k;
    }
    return true;
}

template <int W>
__global__ void __launch_bounds__(kThreads, 2) cg_batch_resident(BatchResidentArgs R) {
    __shared__ double lds[8];
    const BatchArgs &A = R.B;
    const int me = xcd_block_id();
    for (int round = 0; round < R.rounds; ++round) {
        const TeamSlot slot = R.slots[(size_t)round * gridDim.x + me];  // the same for the whole workgroup
        System Y;
        Y.sy = __builtin_amdgcn_readfirstlane(slot.sys);
        if (Y.sy < 0) continue;
        const int base = __builtin_amdgcn_readfirstlane(slot.base);
        Y.rows = A.sys_rows[Y.sy];
        Y.first_chunk = A.sys_chunk0[Y.sy];
        Y.chunks = A.sys_chunk0[Y.sy + 1] - Y.first_chunk;
        Y.chunk = Y.first_chunk + me - base;
        Y.off = ((me - base) * kChunk + (int)threadIdx.x) * 8;
        Team T{R.team, me, base, Y.chunks, (unsigned long long)(round + 1) << 32};
        if (!solve_system<W>(A, Y, T, lds)) return;
    }
}

}  // namespace

BatchResidentFn batch_resident_kernel(int max_width, const DeviceProps &dev, int *grid) {
    if (max_width > 7) return nullptr;
    const BatchResidentFn fn = max_width <= 3 ? cg_batch_resident<3> : cg_batch_resident<7>;
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void *)fn, kThreads, 0) != hipSuccess ||
        per_cu < 1)
        return nullptr;
    *grid = std::min(per_cu * dev.cus, kMaxTeamGrid);
    return fn;
}

// Largest systems first (they also need the most iterations), each into the first round with room: a
// round then holds systems of about the same length, with small ones in what the large ones leave.
// Systems of one chunk go where no larger one comes after them: the members of a team wait for each other
// as long as arrival words grow, and a workgroup alone in its team has none.
std::vector<TeamSlot> batch_resident_schedule(const std::vector<int> &chunk0, int grid, int *rounds) {
    const int nsys = (int)chunk0.size() - 1;
    std::vector<int> order(nsys);
    std::iota(order.begin(), order.end(), 0);
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) {
        return chunk0[a + 1] - chunk0[a] > chunk0[b + 1] - chunk0[b];
    });
    std::vector<TeamSlot> slots;
    std::vector<int> used;  // workgroups taken, per round
    bool alone = false;     // the systems of one chunk have begun
    for (const int s : order) {
        const int need = chunk0[s + 1] - chunk0[s];
        if (need > grid) return {};
        if (need == 1 && !alone) {
            alone = true;
            for (int k = (int)used.size() - 2; k >= 0; --k) used[k] = std::max(used[k], used[k + 1]);
        }
        size_t r = 0;
        while (r < used.size() && used[r] + need > grid) ++r;
        if (r == used.size()) {
            used.push_back(0);
            slots.resize(slots.size() + grid, TeamSlot{-1, 0});
        }
        for (int j = 0; j < need; ++j) slots[r * grid + used[r] + j] = TeamSlot{s, used[r]};
        used[r] += need;
    }
    *rounds = (int)used.size();
    return slots;
}

}  // namespace cfm
