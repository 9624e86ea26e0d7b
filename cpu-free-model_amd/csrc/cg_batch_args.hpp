// Argument blocks of the batched CG kernels.
#pragma once

#include <vector>

#include "cg_common.hpp"

namespace cfm {

enum { kActive = 0, kConverged = 1, kBreakdown = 2, kMaxIter = 3 };

struct BatchArgs {
    int nsys;
    int total_chunks;
    const int *sys_chunk0;  // [nsys+1] first chunk of each system
    const int *sys_rows;    // [nsys] real rows of each system
    Sell A;                 // SELL-64 over the padded global rows
    const double *b;
    const double *x0;
    double *x, *r, *z, *s, *p;
    double *w[2];
    double *part;      // [5][total_chunks]: delta buf0/1, gamma buf0/1, <b,b>
    double *st_alpha;  // [2][nsys]
    double *st_delta;  // [2][nsys]
    int *fin;          // [nsys] iteration at which the system finished (INT_MAX: running)
    int *status;       // [nsys] final state (kConverged, kBreakdown, kMaxIter)
    int *iters;        // [nsys]
    double *hist;      // [nsys][hist_cap] or null
    int hist_cap;
    int max_iter;
    double tol;
    int quirk;
    int x0_guard;      // restart a system from x0 = 0 when <r0,r0> > <b,b>
    int *x0_rejected;  // [nsys] 1 where the guard restarted the system
    // DIA storage (dmax > 0): a(row, row + doff[sy*dmax + d]) at dval[d*dpad + row]
    const double *dval;
    const int *doff;
    int dmax;
    long long dpad;
    GridSync *sync;
};

// Resident batch (cg_batch_resident.hip): a team of workgroups, one for each chunk of a system, solves
// it; slots[round][workgroup] says which system's team a workgroup is in, round after round.
struct TeamSlot {
    int sys;   // -1: none in this round
    int base;  // the team's first workgroup (one per chunk, in chunk order)
};
constexpr int kMaxTeamGrid = 1024;
struct TeamSync {
    unsigned int abort;
    unsigned int pad0[31];
    unsigned long long spin_limit_ticks;
    unsigned long long pad1[15];
    unsigned long long arrive[kMaxTeamGrid];
    unsigned long long go[kMaxTeamGrid * 16];  // workgroup w polls go[16 w], on a line of its own
};
struct BatchResidentArgs {
    BatchArgs B;
    const TeamSlot *slots;
    int rounds;
    TeamSync *team;
};
using BatchResidentFn = void (*)(BatchResidentArgs);
// The kernel for systems whose rows hold at most max_width entries, and the workgroups of 256 threads
// that run at once; null where it does not apply.
BatchResidentFn batch_resident_kernel(int max_width, const DeviceProps &dev, int *grid);
// Rounds for systems of chunk0[s+1] - chunk0[s] chunks on `grid` workgroups; empty where one is too large.
std::vector<TeamSlot> batch_resident_schedule(const std::vector<int> &chunk0, int grid, int *rounds);
__global__ void reset_team_kernel(TeamSync *t, unsigned long long limit_ticks);

}  // namespace cfm
