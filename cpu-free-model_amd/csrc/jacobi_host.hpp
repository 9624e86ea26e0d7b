// Host-side pieces of the Jacobi sweeps shared by the plan entry points and
// the no-allocation entry point: the kernel argument block, the launch
// configuration of one parameter set, and the enqueue of one run.
#pragma once

#include <algorithm>

#include "cfm_common.hpp"

namespace cfm {

struct JacobiArgs {
    void *buf0;
    void *buf1;
    int nx, ny, nz;
    int niter;        // sweeps in this launch
    int it0;          // index of the first sweep (parity and norm slots)
    int bc;
    int norm_every;
    int chunks;       // chunks along the streamed axis
    int chunk_len;
    int ntx, nty;     // tiles along x and y (nty = 1 in 2D)
    int tile_sx, tile_sy;  // register tiles: columns and rows a tile owns
    int tile_hx, tile_hy;  // and loads beyond them on each side
    int depth;             // sweeps per pass of the register tiles
    int no_compute;
    double *norm_part;  // [slot][gridDim.x]
    GridSync *sync;
    unsigned long long *timers;  // phase timers: [workgroup][kTimerSlots] ticks, or null
};

using KernelFn = void (*)(JacobiArgs);

// Launch configuration of one parameter set: kernel, workgroup, grid and the
// work split.  Computed without allocating anything (device queries only).
struct JacobiConfig {
    DeviceProps dev{};
    size_t elems = 0;
    size_t elem_size = 0;
    int norm_slots = 0;
    size_t norm_doubles = 0;  // set before: what the workgroups' sums of all norms have to fit in (0: no limit)
    KernelFn kernel = nullptr;
    bool t2 = false;  // more than one sweep per pass (the two-/three-/four-sweep kernels)
    int sweeps_per_pass = 1;
    bool tile = false;  // the register-tile and pipeline kernels (jacobi_tile.hip, jacobi_pipe.hip)
    bool pipe = false;  // the latter
    int tile_sx = 0, tile_sy = 0, tile_hx = 0, tile_hy = 0, depth = 0;
    int grid = 0;
    int norm_grid = 0;  // the streaming kernel's grid, which the no-allocation entry point's limit goes by
    int chunks = 0, chunk_len = 0, ntx = 0, nty = 0, rows = 0, block = 256;
    unsigned long long spin_ticks = 0;
};

// Validates p and fills c for the current device.
cfm_status jacobi_configure(const cfm_jacobi_params *p, JacobiConfig *c);
// Sweeps of the pipeline kernels' pass that starts with sweep k (jacobi_swaps counts the passes): a sweep whose update norm is wanted
// is the first of its pass, and with periodic planes the run's first sweep is a pass of its own.
__host__ __device__ inline int jacobi_pipe_steps(int k, int niter, int depth, int norm_every, bool periodic) {
    int steps = niter - k < depth ? niter - k : depth;
    if (norm_every > 0 && norm_every - k % norm_every < steps) steps = norm_every - k % norm_every;
    return periodic && k == 0 ? 1 : steps;
}
// The workgroups' partial sums of squares in workgroup order, with what each addition rounds off kept
// and added last: more workgroups share a field in the tile kernels than in the streaming ones, and
// their norms are as accurate for it.
__host__ __device__ inline double jacobi_norm_sum(const double *part, int n) {
    double sum = 0.0, lost = 0.0;
    for (int b = 0; b < n; ++b) {
        const double next = sum + part[b], from_part = next - sum;
        lost += (sum - (next - from_part)) + (part[b] - from_part);
        sum = next;
    }
    return lost == lost ? sum + lost : sum;  // (an infinite sum has no meaningful rest)
}
// Workgroups whose sums of the run's norms, and the norms themselves, fit.
inline int jacobi_norm_workgroups(const JacobiConfig &c) {
    if (c.norm_doubles == 0 || c.norm_slots == 0) return kMaxGrid;
    return (int)std::min((size_t)kMaxGrid, std::max(c.norm_doubles / c.norm_slots, (size_t)2) - 1);
}
// Takes c to a register-tile kernel where that is the faster one; false leaves it as it is.
bool jacobi_tile_configure(const cfm_jacobi_params &p, JacobiConfig *c);  // 2D
bool jacobi_pipe_configure(const cfm_jacobi_params &p, JacobiConfig *c);  // 3D
// Enqueues one run of p.niter sweeps on `stream` (barrier reset, then the
// persistent launch or one launch per sweep) over b0 (current field) and b1;
// timers (may be null): per-workgroup phase ticks; *coop as launch_persistent
// reports it (-1 without a persistent launch).
cfm_status jacobi_enqueue(const cfm_jacobi_params &p, const JacobiConfig &c, void *b0, void *b1, GridSync *sync,
                          double *norm_part, unsigned long long *timers, hipStream_t stream, int *coop);
// Passes of one run, as time_block counts them.
int jacobi_passes(const cfm_jacobi_params &p, const JacobiConfig &c);
// Times that one run changes arrays (its parity says which array holds the result): its passes,
// or the register tiles' own trips through memory.
int jacobi_swaps(const cfm_jacobi_params &p, const JacobiConfig &c);
void jacobi_fill_timing(cfm_timing *t, const cfm_jacobi_params &p, const JacobiConfig &c, float ms, double wall_ms,
                        int coop);

}  // namespace cfm
