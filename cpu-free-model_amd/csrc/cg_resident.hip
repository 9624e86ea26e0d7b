// Resident CG: the whole solve of a system that the chip can hold, with every
// vector and the matrix in registers.
//
// Same recurrences, row-to-thread map and summation trees as cg.hip (so the
// same bits); what changes is where things live.  A sub-block of 256 threads
// owns one 1024-row chunk for the whole solve, four rows a thread; the rows'
// entries, x, r, p, ... stay in its registers.  Only the vector that the SpMV
// gathers and the chunk partials go through memory, past the L2 on both sides,
// so the device barrier needs no L2 write-back or invalidate
// (grid_barrier_through).
//
// Standard CG and the refinement keep the gathered entries of p as well: a row
// gathers r after each update of r and forms its neighbours' p = r + beta p itself,
// the owner's expression on the owner's values.  p is never published, and an
// iteration has two barriers instead of three.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "cg_resident.hpp"

namespace cfm {

namespace {

// This thread's place: chunk c, rows c*1024 + i*256 + t.
template <int SUB>
struct Place {
    int t, c;
    bool in[kRows];
    __device__ __forceinline__ explicit Place(const CgArgs &A) {
        t = threadIdx.x & (kThreads - 1);
        c = blockIdx.x * SUB + (threadIdx.x >> 8);
#pragma unroll
        for (int i = 0; i < kRows; ++i) in[i] = c < A.nchunks && row(i) < A.n;
    }
    __device__ __forceinline__ int row(int i) const { return c * kChunk + i * kThreads + t; }
    __device__ __forceinline__ int slice(int i) const { return c * kSlicesPerChunk + i * 4 + (t >> 6); }
};

// Chunk sums of K per-thread values into part[which[k]].
template <int SUB, int K>
__device__ __forceinline__ void put_partials(const CgArgs &A, const Place<SUB> &P, double (&v)[K], const int (&which)[K],
                                             double *lds) {
    sub_sums<SUB, K>(v, lds);
    if (P.t == 0 && P.c < A.nchunks)
#pragma unroll
        for (int k = 0; k < K; ++k) store_wt(&A.part[which[k] * A.nchunks + P.c], v[k]);
}

// reduce_partials of K partial arrays at once (the same order of additions).
template <int SUB, int K>
__device__ __forceinline__ void get_partials(const CgArgs &A, const int (&which)[K], double (&v)[K], double *lds) {
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] = 0.0;
#pragma unroll
    for (int u = 0; u < SUB; ++u) {  // (a grid of SUB chunks a workgroup is at most 256 workgroups)
        const int j = (threadIdx.x & (kThreads - 1)) + u * kThreads;
        if (j < A.nchunks)
#pragma unroll
            for (int k = 0; k < K; ++k) v[k] = v[k] + load_through(&A.part[which[k] * A.nchunks + j]);
    }
    sub_sums<SUB, K>(v, lds);
}

// r = b - A x0 of this thread's rows, <b,b> and <r,r> along the way.
template <int SUB, int W>
__device__ __forceinline__ void first_residual(const CgArgs &A, const Place<SUB> &P, const Entries<double, double, W> &M,
                                               double (&x)[kRows], double (&r)[kRows], double &rr, double &bb) {
    double g[kRows][W];
    M.gather(A.x0, A.n, g);
    rr = bb = 0.0;
#pragma unroll
    for (int i = 0; i < kRows; ++i) {
        x[i] = r[i] = 0.0;
        if (P.in[i]) {
            const double bi = A.b[P.row(i)];
            x[i] = A.x0[P.row(i)];
            r[i] = fma(-1.0, M.row_sum(i, g), bi);
            rr = fma(r[i], r[i], rr);
            bb = fma(bi, bi, bb);
        }
    }
}

// Buffer stores past the L2: the range check drops rows beyond the system, and one offset a thread
// serves all its rows.
template <int SUB, typename T>
__device__ __forceinline__ void publish(const CgArgs &A, const Place<SUB> &P, T *to, const T (&v)[kRows]) {
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)to, (short)0, A.n * (int)sizeof(T), 0x00020000);
#pragma unroll
    for (int i = 0; i < kRows; ++i) {
        const int off = P.row(i) * (int)sizeof(T);
        if constexpr (sizeof(T) == 8) {
            typedef unsigned int U2 __attribute__((ext_vector_type(2)));
            __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(U2, v[i]), rsrc, off, 0, kSc1);
        } else {
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v[i]), rsrc, off, 0, kSc1);
        }
    }
}

// This thread's rows of a vector it published itself.
template <int SUB>
__device__ __forceinline__ void own_rows(const CgArgs &A, const Place<SUB> &P, const double *from, double (&v)[kRows]) {
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)from, (short)0, A.n * 8, 0x00020000);
#pragma unroll
    for (int i = 0; i < kRows; ++i)
        v[i] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rsrc, P.row(i) * 8, 0, kSc1));
}

// Standard CG.  part: [0]=gamma, [1]=delta, [2]=bb; v[0]: r as the others gather it.  With two
// sub-blocks (256 registers a lane) x stays in memory, where only its own thread touches it.
template <int SUB, int W, bool TIMED>
__global__ void __launch_bounds__(256 * SUB) cg_standard_resident(CgArgs A) {
    __shared__ double lds[8 * SUB];
    __shared__ unsigned long long clk_lds[kClockWords];
    PhaseClock<TIMED> clk{clk_lds};
    clk.start();
    unsigned int epoch = 0;
    const Place<SUB> P(A);
    Entries<double, double, W> M;
    M.load(A.A64, P.c, P.t, P.c < A.nchunks, 0);
    double x[kRows], r[kRows], p[kRows], pg[kRows][W];
    double two[2];
    first_residual(A, P, M, x, r, two[0], two[1]);
    if (SUB > 1) publish(A, P, A.x, x);
    publish(A, P, A.v[0], r);
    put_partials<SUB, 2>(A, P, two, {0, 2}, lds);
    clk.mark(CFM_PHASE_OTHER);
    if (!grid_barrier_through(A.sync, epoch)) return;
    clk.mark(CFM_PHASE_BARRIER);
    M.gather(A.v[0], A.n, pg);  // p starts as r
#pragma unroll
    for (int i = 0; i < kRows; ++i) p[i] = r[i];
    get_partials<SUB, 2>(A, {0, 2}, two, lds);
    double gamma = two[0];
    const double thr = A.tol > 0.0 ? A.tol * A.tol * two[1] : 0.0;
    write_hist(A, 0, gamma);
    clk.mark(CFM_PHASE_REDUCE);
    int k = 0, status = CFM_OK;
    bool converged = gamma <= thr;
    while (!converged && k < A.max_iter) {
        double s[kRows], one[1] = {0.0};
#pragma unroll
        for (int i = 0; i < kRows; ++i) {
            s[i] = M.row_sum(i, pg);
            if (P.in[i]) one[0] = fma(p[i], s[i], one[0]);
        }
        put_partials<SUB, 1>(A, P, one, {1}, lds);
        clk.mark(CFM_PHASE_SPMV);
        if (!grid_barrier_through(A.sync, epoch)) return;
        clk.mark(CFM_PHASE_BARRIER);
        get_partials<SUB, 1>(A, {1}, one, lds);
        const double delta = one[0];
        clk.mark(CFM_PHASE_REDUCE);
        if (!(delta > 0.0) || !is_finite(delta)) {
            status = CFM_EBREAKDOWN;
            break;
        }
        const double alpha = gamma / delta;
        one[0] = 0.0;
        if (SUB > 1) own_rows(A, P, A.x, x);
#pragma unroll
        for (int i = 0; i < kRows; ++i) {
            x[i] = fma(alpha, p[i], x[i]);
            r[i] = fma(-alpha, s[i], r[i]);
            if (P.in[i]) one[0] = fma(r[i], r[i], one[0]);
        }
        if (SUB > 1) publish(A, P, A.x, x);
        publish(A, P, A.v[0], r);
        put_partials<SUB, 1>(A, P, one, {0}, lds);
        clk.mark(CFM_PHASE_UPDATE);
        if (!grid_barrier_through(A.sync, epoch)) return;
        clk.mark(CFM_PHASE_BARRIER);
        double rg[kRows][W];
        M.gather(A.v[0], A.n, rg);  // on its way while the partials are summed
        get_partials<SUB, 1>(A, {0}, one, lds);
        const double gamma_new = one[0];
        ++k;
        write_hist(A, k, gamma_new);
        clk.mark(CFM_PHASE_REDUCE);
        if (gamma_new <= thr) {
            converged = true;
            break;
        }
        const double beta = gamma_new / gamma;
#pragma unroll
        for (int i = 0; i < kRows; ++i) {
            p[i] = fma(beta, p[i], r[i]);
#pragma unroll
            for (int j = 0; j < W; ++j) pg[i][j] = fma(beta, pg[i][j], rg[i][j]);
        }
        gamma = gamma_new;
    }
    if (status == CFM_OK && !converged && A.tol > 0.0) status = CFM_ENOTCONV;
    if (SUB == 1)
#pragma unroll
        for (int i = 0; i < kRows; ++i)
            if (P.in[i]) A.x[P.row(i)] = x[i];
    write_info(A, status, k, 0);
    clk.mark(CFM_PHASE_OTHER);
    clk.flush(A.timers);
}

// Pipelined CG.  part as in cg.hip: [0,1] = delta, [2,3] = gamma (by iteration parity), [4] = bb.
// v[0]: r (for w0 only), v[4], v[5]: w by iteration parity.
template <int SUB, int W, bool TIMED>
__global__ void __launch_bounds__(256 * SUB) cg_pipelined_resident(CgArgs A) {
    __shared__ double lds[8 * SUB];
    __shared__ unsigned long long clk_lds[kClockWords];
    PhaseClock<TIMED> clk{clk_lds};
    clk.start();
    unsigned int epoch = 0;
    const Place<SUB> P(A);
    Entries<double, double, W> M;
    M.load(A.A64, P.c, P.t, P.c < A.nchunks, 0);
    double x[kRows], r[kRows], z[kRows], s[kRows], p[kRows], w[kRows], g[kRows][W];
    double one[1], two[2];
    first_residual(A, P, M, x, r, two[0], one[0]);
    publish(A, P, A.v[0], r);
    put_partials<SUB, 1>(A, P, one, {4}, lds);
    clk.mark(CFM_PHASE_OTHER);
    if (!grid_barrier_through(A.sync, epoch)) return;
    clk.mark(CFM_PHASE_BARRIER);
    M.gather(A.v[0], A.n, g);
    two[0] = two[1] = 0.0;
#pragma unroll
    for (int i = 0; i < kRows; ++i) {
        w[i] = M.row_sum(i, g);
        z[i] = s[i] = p[i] = 0.0;
        if (P.in[i]) {
            two[0] = fma(r[i], r[i], two[0]);
            two[1] = fma(r[i], w[i], two[1]);
        }
    }
    publish(A, P, A.v[4], w);
    put_partials<SUB, 2>(A, P, two, {0, 2}, lds);
    clk.mark(CFM_PHASE_OTHER);
    if (!grid_barrier_through(A.sync, epoch)) return;
    clk.mark(CFM_PHASE_BARRIER);
    get_partials<SUB, 1>(A, {4}, one, lds);
    const double thr = A.tol > 0.0 ? A.tol * A.tol * one[0] : 0.0;
    double alpha = 0.0, beta = 0.0, delta_prev = 0.0;
    int k = 0, status = CFM_OK;
    bool converged = false;
    for (;;) {
        const int buf = __builtin_amdgcn_readfirstlane(k & 1);  // (uniform, which the compiler loses over the loop)
        M.gather(A.v[4 + buf], A.n, g);  // on its way while the partials are summed
        get_partials<SUB, 2>(A, {0 + buf, 2 + buf}, two, lds);
        const double delta = two[0], gam = two[1];
        write_hist(A, k, delta);
        clk.mark(CFM_PHASE_REDUCE);
        if (delta <= thr) {
            converged = true;
            break;
        }
        if (k >= A.max_iter) break;
        double denom;
        if (A.quirk ? (k > 1) : (k > 0)) {
            beta = delta / delta_prev;
            denom = gam - (beta / alpha) * delta;
        } else {
            beta = 0.0;
            denom = gam;
        }
        if (!(denom > 0.0) || !is_finite(denom)) {
            status = CFM_EBREAKDOWN;
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
            if (P.in[i]) {
                two[0] = fma(r[i], r[i], two[0]);
                two[1] = fma(r[i], w[i], two[1]);
            }
        }
        publish(A, P, A.v[5 - buf], w);
        put_partials<SUB, 2>(A, P, two, {1 - buf, 3 - buf}, lds);
        clk.mark(CFM_PHASE_SPMV);
        if (!grid_barrier_through(A.sync, epoch)) return;
        clk.mark(CFM_PHASE_BARRIER);
        delta_prev = delta;
        ++k;
    }
    if (status == CFM_OK && !converged && A.tol > 0.0) status = CFM_ENOTCONV;
#pragma unroll
    for (int i = 0; i < kRows; ++i)
        if (P.in[i]) A.x[P.row(i)] = x[i];
    write_info(A, status, k, 0);
    clk.mark(CFM_PHASE_OTHER);
    clk.flush(A.timers);
}

// Row i of A x in FP64 for the refinement: the FP64 values are read again each time (there are few
// refinements), the columns are the ones at hand.
template <int SUB, int W>
__device__ __forceinline__ double row_sum64(const CgArgs &A, const Place<SUB> &P, const Entries<float, float, W> &M,
                                            int i, const double *x) {
    const auto rv = __builtin_amdgcn_make_buffer_rsrc((void *)A.A64.val, (short)0, A.entries * 8, 0x00020000);
    const auto rx = __builtin_amdgcn_make_buffer_rsrc((void *)x, (short)0, A.n * 8, 0x00020000);
    const int e = (P.in[i] ? A.A64.slice_ptr[P.slice(i)] : 0) + (P.t & 63);
    double v[W], g[W], acc = 0.0;
#pragma unroll
    for (int j = 0; j < W; ++j) {
        const bool ok = M.off[i][j] >= 0;
        v[j] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rv, ok ? (e + 64 * j) * 8 : -1, 0, 0));
        g[j] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rx, ok ? M.off[i][j] * 2 : -1, 0, kSc1));
    }
#pragma unroll
    for (int j = 0; j < W; ++j) acc = fma(v[j], g[j], acc);
    return acc;
}

// FP32 inner CG inside FP64 refinement.  part: [0]=rr (outer), [1]=g, [2]=delta, [3]=bb.
// f[0]: the inner residual as the others gather it; A.x likewise between refinements.
template <int SUB, int W, bool TIMED>
__global__ void __launch_bounds__(256 * SUB) cg_ir_resident(CgArgs A) {
    __shared__ double lds[12 * SUB];
    __shared__ unsigned long long clk_lds[kClockWords];
    PhaseClock<TIMED> clk{clk_lds};
    clk.start();
    unsigned int epoch = 0;
    const Place<SUB> P(A);
    Entries<float, float, W> M;
    M.load(A.A32, P.c, P.t, P.c < A.nchunks, 0);
    double thr = 0.0;
    int outer = 0, inner_total = 0, status = CFM_ENOTCONV;
    for (;;) {
        const bool first = __builtin_amdgcn_readfirstlane(outer == 0);  // (uniform)
        float rf[kRows], p[kRows], d[kRows], pg[kRows][W];
        double three[3];
        {
            double r[kRows];
            three[0] = three[2] = 0.0;
#pragma unroll
            for (int i = 0; i < kRows; ++i) {
                const double ax = row_sum64(A, P, M, i, first ? A.x0 : A.x);
                r[i] = 0.0;
                if (P.in[i]) {
                    const double bi = A.b[P.row(i)];
                    r[i] = fma(-1.0, ax, bi);
                    three[0] = fma(r[i], r[i], three[0]);
                    three[2] = fma(bi, bi, three[2]);
                }
            }
            if (first) {
                double x[kRows];
                own_rows(A, P, A.x0, x);
                publish(A, P, A.x, x);
            }
            three[1] = 0.0;
#pragma unroll
            for (int i = 0; i < kRows; ++i) {
                rf[i] = p[i] = (float)r[i];
                d[i] = 0.0f;
                if (P.in[i]) three[1] = fma((double)rf[i], (double)rf[i], three[1]);
            }
        }
        publish(A, P, A.f[0], rf);
        put_partials<SUB, 3>(A, P, three, {0, 1, 3}, lds);
        clk.mark(CFM_PHASE_OTHER);
        if (!grid_barrier_through(A.sync, epoch)) return;
        clk.mark(CFM_PHASE_BARRIER);
        M.gather(A.f[0], A.n, pg);  // p starts as the residual
        get_partials<SUB, 3>(A, {0, 1, 3}, three, lds);
        if (first) thr = A.tol * A.tol * three[2];
        const double rr = three[0];
        write_hist(A, outer, rr);
        clk.mark(CFM_PHASE_REDUCE);
        if (rr <= thr) {
            status = CFM_OK;
            break;
        }
        if (outer == A.max_outer) break;
        double g = three[1];
        // no refinement is solved beyond half the outer target
        const double thr_in = fmax(A.inner_tol * A.inner_tol * g, 0.25 * thr);
        int j = 0;
        bool brk = false;
        while (j < A.max_iter) {
            float s[kRows];
            double one[1] = {0.0};
#pragma unroll
            for (int i = 0; i < kRows; ++i) {
                s[i] = M.row_sum(i, pg);
                if (P.in[i]) one[0] = fma((double)p[i], (double)s[i], one[0]);
            }
            put_partials<SUB, 1>(A, P, one, {2}, lds);
            clk.mark(CFM_PHASE_SPMV);
            if (!grid_barrier_through(A.sync, epoch)) return;
            clk.mark(CFM_PHASE_BARRIER);
            get_partials<SUB, 1>(A, {2}, one, lds);
            const double delta = one[0];
            clk.mark(CFM_PHASE_REDUCE);
            if (!(delta > 0.0) || !is_finite(delta)) {
                brk = true;
                break;
            }
            const float af = (float)(g / delta);
            one[0] = 0.0;
#pragma unroll
            for (int i = 0; i < kRows; ++i) {
                d[i] = fmaf(af, p[i], d[i]);
                rf[i] = fmaf(-af, s[i], rf[i]);
                if (P.in[i]) one[0] = fma((double)rf[i], (double)rf[i], one[0]);
            }
            publish(A, P, A.f[0], rf);
            put_partials<SUB, 1>(A, P, one, {1}, lds);
            clk.mark(CFM_PHASE_UPDATE);
            if (!grid_barrier_through(A.sync, epoch)) return;
            clk.mark(CFM_PHASE_BARRIER);
            float rg[kRows][W];
            M.gather(A.f[0], A.n, rg);
            get_partials<SUB, 1>(A, {1}, one, lds);
            const double gn = one[0];
            clk.mark(CFM_PHASE_REDUCE);
            ++j;
            if (gn <= thr_in) break;
            const float bf = (float)(gn / g);
#pragma unroll
            for (int i = 0; i < kRows; ++i) {
                p[i] = fmaf(bf, p[i], rf[i]);
#pragma unroll
                for (int e = 0; e < W; ++e) pg[i][e] = fmaf(bf, pg[i][e], rg[i][e]);
            }
            g = gn;
        }
        inner_total += j;
        double x[kRows];
        own_rows(A, P, A.x, x);
#pragma unroll
        for (int i = 0; i < kRows; ++i) x[i] = x[i] + (double)d[i];
        publish(A, P, A.x, x);
        clk.mark(CFM_PHASE_UPDATE);
        if (!grid_barrier_through(A.sync, epoch)) return;
        clk.mark(CFM_PHASE_BARRIER);
        ++outer;
        if (brk && j == 0) {
            status = CFM_EBREAKDOWN;
            break;
        }
    }
    write_info(A, status, inner_total, outer);
    clk.flush(A.timers);
}

// ------------------------------------------------- vectors resident only --
// Larger systems: the vectors stay in registers, the matrix is streamed.  1024 threads, four
// sub-blocks of NCH chunks each: up to 1024 x NCH chunks on 256 CUs.  The gathered vector is written
// past the L2 and read through it (a row's neighbours are read about seven times), so the barrier
// before a gather invalidates; the others only carry partials and do not.  A workgroup's chunks
// follow each other and consecutive workgroups share an XCD, so most of a gather stays in its L2.
constexpr int kSub = 4;
constexpr int kStreamWidth = kResidentDiag;  // entries a row at most (SELL-64), diagonals at most (DIA)

template <int NCH>
struct PlaceN {
    int t, c0;  // chunks c0 .. c0 + NCH - 1
    __device__ __forceinline__ PlaceN() {
        t = threadIdx.x & (kThreads - 1);
        c0 = __builtin_amdgcn_readfirstlane((xcd_block_id() * kSub + (int)(threadIdx.x >> 8)) * NCH);
    }
    __device__ __forceinline__ int row(int q, int i) const { return (c0 + q) * kChunk + i * kThreads + t; }
    __device__ __forceinline__ int slice(int q, int i) const {  // the same for a whole wavefront
        return __builtin_amdgcn_readfirstlane((c0 + q) * kSlicesPerChunk + i * 4 + (t >> 6));
    }
};

template <typename T>
__device__ __forceinline__ T buffer_at(__amdgpu_buffer_rsrc_t rsrc, int off, int soff) {
    if constexpr (sizeof(T) == 8)
        return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(rsrc, off, soff, 0));
    else
        return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(rsrc, off, soff, 0));
}

// The matrix and the vectors it is applied to, read through buffers: one offset a lane serves all
// entries of a row, and what lies outside reads as zero (entries beyond a row's end, columns outside
// the system), so that every load goes out unconditionally.
template <typename T, bool DIA>
struct Stream {
    const Sell &S;
    __amdgpu_buffer_rsrc_t val, col;
    int n;
    __device__ __forceinline__ Stream(const CgArgs &A, const Sell &s) : S(s), n(A.n) {
        const int count = DIA ? s.ndiag * s.npad : A.entries;
        val = __builtin_amdgcn_make_buffer_rsrc((void *)s.val, (short)0, count * (int)sizeof(T), 0x00020000);
        col = __builtin_amdgcn_make_buffer_rsrc((void *)s.col, (short)0, DIA ? 0 : count * 4, 0x00020000);
    }
    // sell_row's chain for one row (its slice, this lane); live: the row's chunk is the system's (both
    // uniform over the wavefront).  kOff moves an offset out of every buffer.
    // GUESS: x is the caller's and may hold infinities.  What is read for entries that the row does not
    // have (a diagonal's zeros, x[0] beyond a SELL-64 slice's width) is then left out, so that they reach
    // only the rows that have their columns.
    template <bool GUESS = false>
    __device__ __forceinline__ T row(const T *x, int row, int slice, int lane, bool live) const {
        constexpr int kOff = (int)0x80000000u;
        const auto rx = __builtin_amdgcn_make_buffer_rsrc((void *)x, (short)0, n * (int)sizeof(T), 0x00020000);
        T v[kStreamWidth], g[kStreamWidth], acc = T(0);
        bool there[kStreamWidth];
        // (opaque: hoisted out of the solve's loop, every entry's offset of every row would hold a register)
        asm volatile("" : "+v"(row), "+v"(lane));
        if constexpr (DIA) {
#pragma unroll
            for (int d = 0; d < kStreamWidth; ++d) {
                const int out = live && d < S.ndiag ? 0 : kOff;
                const int e = min(d, S.ndiag - 1);
                v[d] = buffer_at<T>(val, row * (int)sizeof(T) | out, e * S.npad * (int)sizeof(T));
                g[d] = buffer_at<T>(rx, (row + S.doff[e]) * (int)sizeof(T) | out, 0);
                there[d] = v[d] != T(0);
            }
        } else {
            const int beg = S.slice_ptr[live ? slice : 0];
            const int width = live ? (S.slice_ptr[slice + 1] - beg) >> 6 : 0;
            int c[kStreamWidth];
#pragma unroll
            for (int j = 0; j < kStreamWidth; ++j) {
                const int out = j < width ? 0 : kOff;
                c[j] = __builtin_amdgcn_raw_buffer_load_b32(col, lane * 4 | out, (beg + 64 * j) * 4, 0);
                v[j] = buffer_at<T>(val, lane * (int)sizeof(T) | out, (beg + 64 * j) * (int)sizeof(T));
            }
#pragma unroll
            for (int j = 0; j < kStreamWidth; ++j) {
                g[j] = buffer_at<T>(rx, c[j] * (int)sizeof(T), 0);
                there[j] = j < width;
            }
        }
#pragma unroll
        for (int j = 0; j < kStreamWidth; ++j) acc = GUESS && !there[j] ? acc : fma(v[j], g[j], acc);
        asm volatile("" : "+v"(acc));  // (the next row's loads come after it)
        return acc;
    }
};

// The statements for each of this thread's rows (q, i, row, slice, live), unrolled in one straight
// line.  Rows beyond the system take part: all they read is zero, they change no sum, and what they
// publish is dropped.
#define CFM_FOR_RESIDENT_ROWS(...)                            \
    _Pragma("unroll") for (int q = 0; q < NCH; ++q) {         \
        const bool live = P.c0 + q < A.nchunks;               \
        (void)live;                                           \
        _Pragma("unroll") for (int i = 0; i < kRows; ++i) {   \
            const int row = P.row(q, i);                      \
            const int slice = P.slice(q, i);                  \
            (void)slice;                                      \
            (void)row;                                        \
            __VA_ARGS__                                       \
            __builtin_amdgcn_sched_barrier(0);                \
        }                                                     \
    }

// A thread's element of a vector of the system: through the caches, past the L2, and written past it.
template <typename T>
__device__ __forceinline__ T own(const CgArgs &A, const T *from, int row) {
    asm volatile("" : "+v"(row));
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)from, (short)0, A.n * (int)sizeof(T), 0x00020000);
    return buffer_at<T>(rsrc, row * (int)sizeof(T), 0);
}
__device__ __forceinline__ double own_through(const CgArgs &A, const double *from, int row) {
    asm volatile("" : "+v"(row));
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)from, (short)0, A.n * 8, 0x00020000);
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rsrc, row * 8, 0, kSc1));
}
template <typename T>
__device__ __forceinline__ void put(const CgArgs &A, T *to, int row, T v) {
    asm volatile("" : "+v"(row));
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)to, (short)0, A.n * (int)sizeof(T), 0x00020000);
    if constexpr (sizeof(T) == 8) {
        typedef unsigned int U2 __attribute__((ext_vector_type(2)));
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(U2, v), rsrc, row * 8, 0, kSc1);
    } else {
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), rsrc, row * 4, 0, kSc1);
    }
}

// One of a thread's vectors, a value per row: in registers, or (LDS) in the workgroup's LDS, where
// only the thread itself touches them: with two chunks a sub-block the registers hold about three FP64
// vectors beside a row's loads.
template <typename T, int NCH, bool LDS>
struct Held;
template <typename T, int NCH>
struct Held<T, NCH, false> {
    T v[NCH * kRows];
    struct Store {};
    __device__ __forceinline__ explicit Held(Store &) {}
    __device__ __forceinline__ T get(int q, int i) const { return v[q * kRows + i]; }
    __device__ __forceinline__ void set(int q, int i, T x) { v[q * kRows + i] = x; }
};
template <typename T, int NCH>
struct Held<T, NCH, true> {
    struct Store {
        T v[NCH * kRows][256 * kSub];
    };
    Store &s;
    __device__ __forceinline__ explicit Held(Store &st) : s(st) {}
    __device__ __forceinline__ T get(int q, int i) const { return s.v[q * kRows + i][threadIdx.x]; }
    __device__ __forceinline__ void set(int q, int i, T x) { s.v[q * kRows + i][threadIdx.x] = x; }
};

template <int NCH, int K>
__device__ __forceinline__ void put_partials_n(const CgArgs &A, const PlaceN<NCH> &P, double (&v)[NCH * K],
                                               const int (&which)[K], double *lds) {
    sub_sums<kSub, NCH * K>(v, lds);
#pragma unroll
    for (int q = 0; q < NCH; ++q)
        if (P.t == 0 && P.c0 + q < A.nchunks)
#pragma unroll
            for (int k = 0; k < K; ++k) store_wt(&A.part[which[k] * A.nchunks + P.c0 + q], v[q * K + k]);
}

// reduce_partials of K partial arrays at once, eight loads at least on their way together (beyond the
// last partial a zero is added, which changes no sum)
template <int K>
__device__ __forceinline__ void get_partials_n(const CgArgs &A, const int (&which)[K], double (&v)[K], double *lds) {
    constexpr int E = K > 1 ? 4 : 8;
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] = 0.0;
    for (int j0 = 0; j0 < A.nchunks; j0 += E * kThreads) {
        const int off = (j0 + (int)(threadIdx.x & (kThreads - 1))) * 8;
        double u[K][E];
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const auto rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)(A.part + which[k] * A.nchunks), (short)0,
                                                                A.nchunks * 8, 0x00020000);
#pragma unroll
            for (int e = 0; e < E; ++e)
                u[k][e] = __builtin_bit_cast(
                    double, __builtin_amdgcn_raw_buffer_load_b64(rsrc, off + e * kThreads * 8, 0, kSc1));
        }
#pragma unroll
        for (int k = 0; k < K; ++k)
#pragma unroll
            for (int e = 0; e < E; ++e) v[k] = v[k] + u[k][e];
    }
    sub_sums<kSub, K>(v, lds);
}

template <int NCH, bool DIA, bool TIMED>
__global__ void __launch_bounds__(256 * kSub) cg_standard_streamed(CgArgs A) {
    __shared__ double lds[8 * kSub * NCH];
    __shared__ unsigned long long clk_lds[kClockWords];
    PhaseClock<TIMED> clk{clk_lds};
    clk.start();
    unsigned int epoch = 0;
    const PlaceN<NCH> P;
    const Stream<double, DIA> M(A, A.A64);
    __shared__ typename Held<double, NCH, (NCH > 1)>::Store xs, ss;
    Held<double, NCH, (NCH > 1)> x(xs), s(ss);
    double r[NCH][kRows], p[NCH][kRows];
    double two[2 * NCH], one[NCH], sum2[2], sum1[1];
#pragma unroll
    for (int e = 0; e < 2 * NCH; ++e) two[e] = 0.0;
    CFM_FOR_RESIDENT_ROWS({
        const double ax = M.template row<true>(A.x0, row, slice, P.t & 63, live);
        const double bi = own(A, A.b, row);
        x.set(q, i, own(A, A.x0, row));
        p[q][i] = r[q][i] = fma(-1.0, ax, bi);
        put(A, A.v[1], row, p[q][i]);
        two[2 * q] = fma(r[q][i], r[q][i], two[2 * q]);
        two[2 * q + 1] = fma(bi, bi, two[2 * q + 1]);
    })
    put_partials_n<NCH, 2>(A, P, two, {0, 2}, lds);
    clk.mark(CFM_PHASE_OTHER);
    if (!grid_barrier_through<true>(A.sync, epoch)) return;
    clk.mark(CFM_PHASE_BARRIER);
    get_partials_n<2>(A, {0, 2}, sum2, lds);
    double gamma = sum2[0];
    const double thr = A.tol > 0.0 ? A.tol * A.tol * sum2[1] : 0.0;
    write_hist(A, 0, gamma);
    clk.mark(CFM_PHASE_REDUCE);
    int k = 0, status = CFM_OK;
    bool converged = gamma <= thr;
    while (!converged && k < A.max_iter) {
#pragma unroll
        for (int q = 0; q < NCH; ++q) one[q] = 0.0;
        CFM_FOR_RESIDENT_ROWS({
            const double si = M.row(A.v[1], row, slice, P.t & 63, live);
            s.set(q, i, si);
            one[q] = fma(p[q][i], si, one[q]);
        })
        put_partials_n<NCH, 1>(A, P, one, {1}, lds);
        clk.mark(CFM_PHASE_SPMV);
        if (!grid_barrier_through(A.sync, epoch)) return;
        clk.mark(CFM_PHASE_BARRIER);
        get_partials_n<1>(A, {1}, sum1, lds);
        const double delta = sum1[0];
        clk.mark(CFM_PHASE_REDUCE);
        if (!(delta > 0.0) || !is_finite(delta)) {
            status = CFM_EBREAKDOWN;
            break;
        }
        const double alpha = gamma / delta;
#pragma unroll
        for (int q = 0; q < NCH; ++q) one[q] = 0.0;
        CFM_FOR_RESIDENT_ROWS({
            x.set(q, i, fma(alpha, p[q][i], x.get(q, i)));
            r[q][i] = fma(-alpha, s.get(q, i), r[q][i]);
            one[q] = fma(r[q][i], r[q][i], one[q]);
        })
        put_partials_n<NCH, 1>(A, P, one, {0}, lds);
        clk.mark(CFM_PHASE_UPDATE);
        if (!grid_barrier_through(A.sync, epoch)) return;
        clk.mark(CFM_PHASE_BARRIER);
        get_partials_n<1>(A, {0}, sum1, lds);
        const double gamma_new = sum1[0];
        ++k;
        write_hist(A, k, gamma_new);
        clk.mark(CFM_PHASE_REDUCE);
        if (gamma_new <= thr) {
            converged = true;
            break;
        }
        const double beta = gamma_new / gamma;
        CFM_FOR_RESIDENT_ROWS({
            p[q][i] = fma(beta, p[q][i], r[q][i]);
            put(A, A.v[1], row, p[q][i]);
        })
        clk.mark(CFM_PHASE_UPDATE);
        if (!grid_barrier_through<true>(A.sync, epoch)) return;
        clk.mark(CFM_PHASE_BARRIER);
        gamma = gamma_new;
    }
    if (status == CFM_OK && !converged && A.tol > 0.0) status = CFM_ENOTCONV;
    CFM_FOR_RESIDENT_ROWS({ put(A, A.x, row, x.get(q, i)); })
    write_info(A, status, k, 0);
    clk.mark(CFM_PHASE_OTHER);
    clk.flush(A.timers);
}

template <int NCH, bool DIA, bool TIMED>
__global__ void __launch_bounds__(256 * kSub) cg_pipelined_streamed(CgArgs A) {
    __shared__ double lds[8 * kSub * NCH];
    __shared__ unsigned long long clk_lds[kClockWords];
    PhaseClock<TIMED> clk{clk_lds};
    clk.start();
    unsigned int epoch = 0;
    const PlaceN<NCH> P;
    const Stream<double, DIA> M(A, A.A64);
    // two chunks: s in LDS, and x too where the registers then suffice, else p and x stays in memory
    constexpr bool X_MEM = NCH > 1 && (!DIA || TIMED);
    __shared__ typename Held<double, NCH, (NCH > 1)>::Store ss;
    __shared__ typename Held<double, NCH, (NCH > 1 && !X_MEM)>::Store xs;
    __shared__ typename Held<double, NCH, X_MEM>::Store ps;
    Held<double, NCH, (NCH > 1)> s(ss);
    Held<double, NCH, (NCH > 1 && !X_MEM)> x(xs);
    Held<double, NCH, X_MEM> p(ps);
    double r[NCH][kRows], z[NCH][kRows];
    double two[2 * NCH], one[NCH], sum2[2], sum1[1];
#pragma unroll
    for (int q = 0; q < NCH; ++q) one[q] = 0.0;
    CFM_FOR_RESIDENT_ROWS({
        const double ax = M.template row<true>(A.x0, row, slice, P.t & 63, live);
        const double bi = own(A, A.b, row);
        if (X_MEM)
            put(A, A.x, row, own(A, A.x0, row));
        else
            x.set(q, i, own(A, A.x0, row));
        r[q][i] = fma(-1.0, ax, bi);
        asm volatile("" : "+v"(r[q][i]));  // (waits for this row's loads before the next row's)
        put(A, A.v[0], row, r[q][i]);
        one[q] = fma(bi, bi, one[q]);
    })
    put_partials_n<NCH, 1>(A, P, one, {4}, lds);
    clk.mark(CFM_PHASE_OTHER);
    if (!grid_barrier_through<true>(A.sync, epoch)) return;
    clk.mark(CFM_PHASE_BARRIER);
#pragma unroll
    for (int e = 0; e < 2 * NCH; ++e) two[e] = 0.0;
    CFM_FOR_RESIDENT_ROWS({
        const double w = M.row(A.v[0], row, slice, P.t & 63, live);
        put(A, A.v[4], row, w);
        two[2 * q] = fma(r[q][i], r[q][i], two[2 * q]);
        two[2 * q + 1] = fma(r[q][i], w, two[2 * q + 1]);
    })
    put_partials_n<NCH, 2>(A, P, two, {0, 2}, lds);
    clk.mark(CFM_PHASE_OTHER);
    if (!grid_barrier_through<true>(A.sync, epoch)) return;
    clk.mark(CFM_PHASE_BARRIER);
    get_partials_n<1>(A, {4}, sum1, lds);
    const double thr = A.tol > 0.0 ? A.tol * A.tol * sum1[0] : 0.0;
    CFM_FOR_RESIDENT_ROWS({
        z[q][i] = 0.0;
        p.set(q, i, 0.0);
        s.set(q, i, 0.0);
    })
    double alpha = 0.0, beta = 0.0, delta_prev = 0.0;
    int k = 0, status = CFM_OK;
    bool converged = false;
    for (;;) {
        const int buf = __builtin_amdgcn_readfirstlane(k & 1);  // (uniform, which the compiler loses over the loop)
        get_partials_n<2>(A, {0 + buf, 2 + buf}, sum2, lds);
        const double delta = sum2[0], gam = sum2[1];
        write_hist(A, k, delta);
        clk.mark(CFM_PHASE_REDUCE);
        if (delta <= thr) {
            converged = true;
            break;
        }
        if (k >= A.max_iter) break;
        double denom;
        if (A.quirk ? (k > 1) : (k > 0)) {
            beta = delta / delta_prev;
            denom = gam - (beta / alpha) * delta;
        } else {
            beta = 0.0;
            denom = gam;
        }
        if (!(denom > 0.0) || !is_finite(denom)) {
            status = CFM_EBREAKDOWN;
            break;
        }
        alpha = delta / denom;
        const double *wc = A.v[4 + buf];
        double *wn = A.v[5 - buf];
#pragma unroll
        for (int e = 0; e < 2 * NCH; ++e) two[e] = 0.0;
        CFM_FOR_RESIDENT_ROWS({
            const double qi = M.row(wc, row, slice, P.t & 63, live);
            const double wi = own(A, wc, row);
            z[q][i] = fma(beta, z[q][i], qi);
            const double si = fma(beta, s.get(q, i), wi);
            s.set(q, i, si);
            const double pi = fma(beta, p.get(q, i), r[q][i]);
            p.set(q, i, pi);
            if (X_MEM)
                put(A, A.x, row, fma(alpha, pi, own_through(A, A.x, row)));
            else
                x.set(q, i, fma(alpha, pi, x.get(q, i)));
            r[q][i] = fma(-alpha, si, r[q][i]);
            const double wn_i = fma(-alpha, z[q][i], wi);
            asm volatile("" : "+v"(z[q][i]), "+v"(r[q][i]));
            put(A, wn, row, wn_i);
            two[2 * q] = fma(r[q][i], r[q][i], two[2 * q]);
            two[2 * q + 1] = fma(r[q][i], wn_i, two[2 * q + 1]);
        })
        put_partials_n<NCH, 2>(A, P, two, {1 - buf, 3 - buf}, lds);
        clk.mark(CFM_PHASE_SPMV);
        if (!grid_barrier_through<true>(A.sync, epoch)) return;
        clk.mark(CFM_PHASE_BARRIER);
        delta_prev = delta;
        ++k;
    }
    if (status == CFM_OK && !converged && A.tol > 0.0) status = CFM_ENOTCONV;
    if (!X_MEM) CFM_FOR_RESIDENT_ROWS({ put(A, A.x, row, x.get(q, i)); })
    write_info(A, status, k, 0);
    clk.mark(CFM_PHASE_OTHER);
    clk.flush(A.timers);
}

template <int NCH, bool DIA, bool TIMED>
__global__ void __launch_bounds__(256 * kSub) cg_ir_streamed(CgArgs A) {
    __shared__ double lds[12 * kSub * NCH];
    __shared__ unsigned long long clk_lds[kClockWords];
    PhaseClock<TIMED> clk{clk_lds};
    clk.start();
    unsigned int epoch = 0;
    const PlaceN<NCH> P;
    const Stream<double, DIA> M(A, A.A64);
    const Stream<float, DIA> M32(A, A.A32);
    __shared__ typename Held<float, NCH, (NCH > 1)>::Store ds;
    double thr = 0.0;
    int outer = 0, inner_total = 0, status = CFM_ENOTCONV;
    for (;;) {
        const bool first = __builtin_amdgcn_readfirstlane(outer == 0);  // (uniform)
        Held<float, NCH, (NCH > 1)> d(ds);
        float rf[NCH][kRows], p[NCH][kRows], s[NCH][kRows];
        double three[3 * NCH], one[NCH], sum3[3], sum1[1];
#pragma unroll
        for (int e = 0; e < 3 * NCH; ++e) three[e] = 0.0;
        CFM_FOR_RESIDENT_ROWS({
            const double ax = M.template row<true>(first ? A.x0 : A.x, row, slice, P.t & 63, live);
            const double bi = own(A, A.b, row);
            const double ri = fma(-1.0, ax, bi);
            if (first) put(A, A.x, row, own(A, A.x0, row));
            rf[q][i] = p[q][i] = (float)ri;
            d.set(q, i, 0.0f);
            put(A, A.f[1], row, p[q][i]);
            three[3 * q] = fma(ri, ri, three[3 * q]);
            three[3 * q + 1] = fma((double)rf[q][i], (double)rf[q][i], three[3 * q + 1]);
            three[3 * q + 2] = fma(bi, bi, three[3 * q + 2]);
        })
        put_partials_n<NCH, 3>(A, P, three, {0, 1, 3}, lds);
        clk.mark(CFM_PHASE_OTHER);
        if (!grid_barrier_through<true>(A.sync, epoch)) return;
        clk.mark(CFM_PHASE_BARRIER);
        get_partials_n<3>(A, {0, 1, 3}, sum3, lds);
        if (first) thr = A.tol * A.tol * sum3[2];
        const double rr = sum3[0];
        write_hist(A, outer, rr);
        clk.mark(CFM_PHASE_REDUCE);
        if (rr <= thr) {
            status = CFM_OK;
            break;
        }
        if (outer == A.max_outer) break;
        double g = sum3[1];
        // no refinement is solved beyond half the outer target
        const double thr_in = fmax(A.inner_tol * A.inner_tol * g, 0.25 * thr);
        int j = 0;
        bool brk = false;
        while (j < A.max_iter) {
#pragma unroll
            for (int q = 0; q < NCH; ++q) one[q] = 0.0;
            CFM_FOR_RESIDENT_ROWS({
                s[q][i] = M32.row(A.f[1], row, slice, P.t & 63, live);
                one[q] = fma((double)p[q][i], (double)s[q][i], one[q]);
            })
            put_partials_n<NCH, 1>(A, P, one, {2}, lds);
            clk.mark(CFM_PHASE_SPMV);
            if (!grid_barrier_through(A.sync, epoch)) return;
            clk.mark(CFM_PHASE_BARRIER);
            get_partials_n<1>(A, {2}, sum1, lds);
            const double delta = sum1[0];
            clk.mark(CFM_PHASE_REDUCE);
            if (!(delta > 0.0) || !is_finite(delta)) {
                brk = true;
                break;
            }
            const float af = (float)(g / delta);
#pragma unroll
            for (int q = 0; q < NCH; ++q) one[q] = 0.0;
            CFM_FOR_RESIDENT_ROWS({
                d.set(q, i, fmaf(af, p[q][i], d.get(q, i)));
                rf[q][i] = fmaf(-af, s[q][i], rf[q][i]);
                one[q] = fma((double)rf[q][i], (double)rf[q][i], one[q]);
            })
            put_partials_n<NCH, 1>(A, P, one, {1}, lds);
            clk.mark(CFM_PHASE_UPDATE);
            if (!grid_barrier_through(A.sync, epoch)) return;
            clk.mark(CFM_PHASE_BARRIER);
            get_partials_n<1>(A, {1}, sum1, lds);
            const double gn = sum1[0];
            clk.mark(CFM_PHASE_REDUCE);
            ++j;
            if (gn <= thr_in) break;
            const float bf = (float)(gn / g);
            CFM_FOR_RESIDENT_ROWS({
                p[q][i] = fmaf(bf, p[q][i], rf[q][i]);
                put(A, A.f[1], row, p[q][i]);
            })
            clk.mark(CFM_PHASE_UPDATE);
            if (!grid_barrier_through<true>(A.sync, epoch)) return;
            clk.mark(CFM_PHASE_BARRIER);
            g = gn;
        }
        inner_total += j;
        CFM_FOR_RESIDENT_ROWS({ put(A, A.x, row, own_through(A, A.x, row) + (double)d.get(q, i)); })
        clk.mark(CFM_PHASE_UPDATE);
        if (!grid_barrier_through<true>(A.sync, epoch)) return;
        clk.mark(CFM_PHASE_BARRIER);
        ++outer;
        if (brk && j == 0) {
            status = CFM_EBREAKDOWN;
            break;
        }
    }
    write_info(A, status, inner_total, outer);
    clk.flush(A.timers);
}

template <int NCH, bool DIA>
CgKernelFn streamed_fn(int method, bool timed) {
    switch (method) {
        case CFM_CG_STANDARD:
            return timed ? cg_standard_streamed<NCH, DIA, true> : cg_standard_streamed<NCH, DIA, false>;
        case CFM_CG_PIPELINED:
            return timed ? cg_pipelined_streamed<NCH, DIA, true> : cg_pipelined_streamed<NCH, DIA, false>;
        default: return timed ? cg_ir_streamed<NCH, DIA, true> : cg_ir_streamed<NCH, DIA, false>;
    }
}

template <int SUB, int W>
CgKernelFn resident_fn(int method, bool timed) {
    switch (method) {
        case CFM_CG_STANDARD: return timed ? cg_standard_resident<SUB, W, true> : cg_standard_resident<SUB, W, false>;
        case CFM_CG_PIPELINED:
            return timed ? cg_pipelined_resident<SUB, W, true> : cg_pipelined_resident<SUB, W, false>;
        default: return timed ? cg_ir_resident<SUB, W, true> : cg_ir_resident<SUB, W, false>;
    }
}

}  // namespace

bool cg_resident_streams(int nchunks, const DeviceProps &dev) {
    const int cus = std::min(dev.cus, kThreads);
    return nchunks > 2 * cus && nchunks <= 2 * kSub * cus;
}

CgResident cg_resident(int method, int nchunks, int max_width, bool dia, bool timed, const DeviceProps &dev) {
    CgResident o;
    const int cus = std::min(dev.cus, kThreads);  // (get_partials reads one partial a thread and sub-block)
    if (!dia && max_width <= 7 && nchunks <= 2 * cus) {
        // one chunk per workgroup while there is a CU for each, else two
        o.sub = nchunks <= cus ? 1 : 2;
        if (o.sub == 1)
            o.fn = max_width <= 3 ? resident_fn<1, 3>(method, timed) : resident_fn<1, 7>(method, timed);
        else
            o.fn = max_width <= 3 ? resident_fn<2, 3>(method, timed) : resident_fn<2, 7>(method, timed);
        o.grid = (nchunks + o.sub - 1) / o.sub;
    } else if (cg_resident_streams(nchunks, dev) && max_width <= kStreamWidth) {
        const int per = nchunks <= kSub * cus ? 1 : 2;
        o.sub = kSub;
        if (dia)
            o.fn = per == 1 ? streamed_fn<1, true>(method, timed) : streamed_fn<2, true>(method, timed);
        else
            o.fn = per == 1 ? streamed_fn<1, false>(method, timed) : streamed_fn<2, false>(method, timed);
        o.grid = (nchunks + kSub * per - 1) / (kSub * per);
    }
    return o;
}

}  // namespace cfm
