// Device pieces shared by the streaming and the register-tile Jacobi kernels.
#pragma once

#include "jacobi_host.hpp"

namespace cfm {

// ------------------------------------------------------------ pass clock --
// Phase timers of the Jacobi kernels (TIMED builds, A.timers set): the time
// between barriers goes to the sweeps, the wait at the device-wide barrier to
// the barrier.
template <bool THROUGH = false, bool TIMED>
__device__ __forceinline__ bool pass_barrier(const JacobiArgs &A, unsigned int &epoch, PhaseClock<TIMED> &clk) {
    clk.mark(CFM_PHASE_SPMV);
    const bool ok = THROUGH ? grid_barrier_through(A.sync, epoch) : grid_barrier(A.sync, epoch);
    clk.mark(CFM_PHASE_BARRIER);
    return ok;
}

// The same shifts with zeros shifted in at lane 0 / lane 63 (bound_ctrl): no copy
// of the old value into the destination first, for callers that replace those
// two lanes anyway.
template <typename T>
__device__ __forceinline__ T lane_up1z(T v) {
    static_assert(sizeof(T) == 8 || sizeof(T) == 4, "4- or 8-byte values");
    if constexpr (sizeof(T) == 8) {
        union {
            T t;
            int i[2];
        } a, r;
        a.t = v;
        r.i[0] = __builtin_amdgcn_mov_dpp(a.i[0], 0x138 /* wave_shr:1 */, 0xf, 0xf, true);
        r.i[1] = __builtin_amdgcn_mov_dpp(a.i[1], 0x138, 0xf, 0xf, true);
        return r.t;
    } else {
        return __builtin_bit_cast(T, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x138, 0xf, 0xf, true));
    }
}
template <typename T>
__device__ __forceinline__ T lane_dn1z(T v) {
    static_assert(sizeof(T) == 8 || sizeof(T) == 4, "4- or 8-byte values");
    if constexpr (sizeof(T) == 8) {
        union {
            T t;
            int i[2];
        } a, r;
        a.t = v;
        r.i[0] = __builtin_amdgcn_mov_dpp(a.i[0], 0x130 /* wave_shl:1 */, 0xf, 0xf, true);
        r.i[1] = __builtin_amdgcn_mov_dpp(a.i[1], 0x130, 0xf, 0xf, true);
        return r.t;
    } else {
        return __builtin_bit_cast(T, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x130, 0xf, 0xf, true));
    }
}

// The global wavefront index under the same map.
__device__ __forceinline__ int xcd_wave_id() { return xcd_block_id() * (blockDim.x >> 6) + (threadIdx.x >> 6); }

}  // namespace cfm
