// Device pieces of the resident CG kernels (cg_resident.hip, cg_batch_resident.hip): a chunk's matrix
// entries in registers, gathers past the L2, and sums of several values at once.
#pragma once

#include "cg_args.hpp"

namespace cfm {

constexpr int kRows = 4;  // rows per thread: a chunk over a sub-block

template <typename T>
__device__ __forceinline__ T load_through(const T *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The rows' entries in stored order.  Columns are kept as byte offsets into a vector of XT, -1 beyond
// a row's end.  The gather is buffer loads (scope bit sc1: past the L2): their range check turns -1
// into a zero, so all loads go out in one straight line, and they take the offset as it is, where
// plain loads would hold a 64-bit address for every entry.
template <typename VT, typename XT, int W>
struct Entries {
    VT v[kRows][W];
    int off[kRows][W];

    // chunk's rows of this thread (none if the chunk is not live); columns count from col0
    __device__ __forceinline__ void load(const Sell &S, int chunk, int t, bool live, int col0) {
        const int *sp = S.slice_ptr + (live ? chunk * kSlicesPerChunk : 0);
        const int first = sp[0], count = live ? sp[kSlicesPerChunk] - first : 0;
        const auto rc = __builtin_amdgcn_make_buffer_rsrc((void *)(S.col + first), (short)0, count * 4, 0x00020000);
        const auto rv = __builtin_amdgcn_make_buffer_rsrc((void *)(static_cast<const VT *>(S.val) + first), (short)0,
                                                          count * (int)sizeof(VT), 0x00020000);
#pragma unroll
        for (int i = 0; i < kRows; ++i) {
            const int s = i * 4 + (t >> 6);
            const int beg = live ? sp[s] - first : 0;
            const int width = live ? (sp[s + 1] - first - beg) >> 6 : 0;
#pragma unroll
            for (int j = 0; j < W; ++j) {
                const int e = beg + 64 * j + (t & 63);
                const int c = __builtin_amdgcn_raw_buffer_load_b32(rc, j < width ? e * 4 : -1, 0, 0);
                if constexpr (sizeof(VT) == 8)
                    v[i][j] = __builtin_bit_cast(
                        VT, __builtin_amdgcn_raw_buffer_load_b64(rv, j < width ? e * 8 : -1, 0, 0));
                else
                    v[i][j] = __builtin_bit_cast(
                        VT, __builtin_amdgcn_raw_buffer_load_b32(rv, j < width ? e * 4 : -1, 0, 0));
                off[i][j] = j < width && c >= 0 ? (c - col0) * (int)sizeof(XT) : -1;
            }
        }
    }
    // x: n elements (a resident system is far below 2 GiB)
    __device__ __forceinline__ void gather(const XT *x, int n, XT (&g)[kRows][W]) const {
        const auto rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)x, (short)0, n * (int)sizeof(XT), 0x00020000);
#pragma unroll
        for (int i = 0; i < kRows; ++i)
#pragma unroll
            for (int j = 0; j < W; ++j)
                if constexpr (sizeof(XT) == 8)
                    g[i][j] = __builtin_bit_cast(XT, __builtin_amdgcn_raw_buffer_load_b64(rsrc, off[i][j], 0, kSc1));
                else
                    g[i][j] = __builtin_bit_cast(XT, __builtin_amdgcn_raw_buffer_load_b32(rsrc, off[i][j], 0, kSc1));
    }
    // The row sum over gathered entries: sell_row's chain.  Entries beyond a row's end are 0 * 0,
    // which leaves the sum as it is (skipping them instead held a lane mask per entry).
    __device__ __forceinline__ XT row_sum(int i, const XT (&g)[kRows][W]) const {
        XT acc = XT(0);
#pragma unroll
        for (int j = 0; j < W; ++j) acc = fma((XT)v[i][j], g[i][j], acc);
        return acc;
    }
};

// sub_sum of K values with one pair of workgroup barriers; lds holds K * 4 * SUB doubles.
template <int SUB, int K>
__device__ __forceinline__ void sub_sums(double (&v)[K], double *lds) {
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] = wave_butterfly(v[k]);
    __syncthreads();  // lds may still be read from a previous call
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int k = 0; k < K; ++k) lds[k * 4 * SUB + (threadIdx.x >> 6)] = v[k];
    __syncthreads();
    const int w0 = (threadIdx.x >> 8) * 4;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const double *l = lds + k * 4 * SUB + w0;
        v[k] = (l[0] + l[1]) + (l[2] + l[3]);
    }
}

}  // namespace cfm
