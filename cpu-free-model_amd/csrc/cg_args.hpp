// Pieces shared by the single-system CG kernels: their argument block, the
// write-through stores and the result words.
#pragma once

#include "cg_common.hpp"

namespace cfm {

struct CgArgs {
    int n;
    int nchunks;
    int entries;  // stored entries of the SELL-64 matrix, padding included
    Sell A64;  // FP64 values
    Sell A32;  // FP32 values (IR only)
    const double *b;
    const double *x0;
    double *x;
    double *v[6];        // work vectors (meaning depends on the method)
    float *f[4];         // FP32 work vectors (IR)
    double *part;        // partial sums, [8][nchunks]
    double *hist;
    int hist_cap;
    int max_iter;
    double tol;
    int quirk;
    int max_outer;
    double inner_tol;
    int *info;           // [0] status, [1] iterations, [2] outer iterations
    GridSync *sync;
    unsigned long long *timers;  // phase-timer build: [workgroup][kTimerSlots] ticks
};

// Store that writes through the XCD's L2 (a relaxed agent-scope atomic store:
// a vector store with scope bit sc1 on gfx950) instead of leaving a dirty
// line there for the next device barrier's release to write back.  Measured
// on the 128^3 Poisson system: Standard CG (s, x, r, p; three barriers per
// iteration) 82.1 -> 76.4 us per iteration; the refinement's FP32 inner
// iteration (s, d, r, p) 60.6 -> 59.7 us; Pipelined CG (one barrier per
// iteration) gains only for w, the vector the next SpMV gathers (71.6 -> 70.7
// us), and runs slower with its other vectors written through.  Being a
// compiler-visible store, it is counted in the compiler's own wait counters.
// Ordering against other workgroups comes only from the device barrier (a
// workgroup barrier, then one thread's agent-scope release, which the HIP
// memory model makes cumulative over the workgroup's earlier stores; an
// agent-scope acquire on exit); the relaxed atomic adds no ordering of its own.
__device__ __forceinline__ void store_wt(double *p, double v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void store_wt(float *p, float v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void write_info(const CgArgs &A, int status, int iters, int outer) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        A.info[0] = status;
        A.info[1] = iters;
        A.info[2] = outer;
    }
}
__device__ __forceinline__ void write_hist(const CgArgs &A, int k, double v) {
    if (blockIdx.x == 0 && threadIdx.x == 0 && A.hist && k < A.hist_cap) A.hist[k] = v;
}

using CgKernelFn = void (*)(CgArgs);

// The resident kernel (cg_resident.hip) for a system of this method, stored as DIA or as SELL-64
// with at most max_width diagonals or entries a row, with its workgroup and grid; null where it does not apply.
struct CgResident {
    CgKernelFn fn = nullptr;
    int sub = 0, grid = 0;
};
constexpr int kResidentDiag = 8;  // diagonals they take at most
// whether a system of nchunks chunks is one whose matrix they stream
bool cg_resident_streams(int nchunks, const DeviceProps &dev);
CgResident cg_resident(int method, int nchunks, int max_width, bool dia, bool timed, const DeviceProps &dev);

}  // namespace cfm
