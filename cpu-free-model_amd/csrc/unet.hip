// Learned warm start: a 3-level 3D U-Net (16/32/64 channels, 3x3x3 convs)
// with hand-written forward and backward kernels on BF16 MFMA (FP32
// accumulate), trained on the GPU with Adam.  No counterpart in the
// reference: it produces initial guesses x0 for the CG solvers.
//
// Tensors are channels-last (NDHWC) BF16; spatial index p = ((b*n+z)*n+y)*n+x.
// A 3x3x3 convolution is an implicit GEMM: Y[p][co] = sum_k W[co][k] Xs[p][k]
// with k = tap*Cin + ci and Xs[p][k] = X[p + offset(tap)][ci] (zero outside).
// One v_mfma_f32_16x16x32_bf16 handles 16 output channels x 16 points x 32
// k; lane l holds A[l%16][8(l/16)..+7], B[8(l/16)..+7][l%16] and
// D[4(l/16)+i][l%16] (layout checked on the device).  Channel counts are
// multiples of 8, so a lane's 8 k-values are 8 consecutive channels of one
// tap: one 16-byte read from the workgroup's input block, which is staged in
// LDS with its one-point halo.
//
// Backward data is the same kernel with the weights flipped in space and
// transposed in channels; backward weights is a split-K MFMA GEMM over point
// slabs (one workgroup per slab, all taps, point blocks staged transposed in
// LDS) followed by a fixed-order reduction of the slab partials.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <vector>

#include "cfm_common.hpp"
#include "unet.hpp"

namespace cfm {
namespace unet {

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float bf2f(bf16 v) { return (float)v; }
__device__ __forceinline__ bf16 f2bf(float v) { return (bf16)v; }  // round to nearest even

// The decoder's convolutions (48 and 96 input channels) read the concatenation of an upsampled
// tensor and a skip connection; it is not stored: the channels below upsampled_channels(CIN) come from the
// points of a grid of half the edge (nearest upsampling), the others from the skip connection's tensor.
constexpr __host__ __device__ int upsampled_channels(int cin) { return cin == 48 ? 32 : cin == 96 ? 64 : 0; }

// channels 8 cv .. 8 cv + 7 of point (x, y, z) of batch element b
template <int CIN>
__device__ __forceinline__ bf16x8 input8(const bf16 *__restrict__ X, const bf16 *__restrict__ Xup, int n, int b, int z,
                                         int y, int x, int cv) {
    constexpr int UP = upsampled_channels(CIN), OWN = CIN - UP;
    if (UP > 0 && cv < UP / 8) {
        const int m = n / 2;
        return *reinterpret_cast<const bf16x8 *>(Xup + ((((size_t)b * m + z / 2) * m + y / 2) * m + x / 2) * UP + cv * 8);
    }
    return *reinterpret_cast<const bf16x8 *>(X + ((((size_t)b * n + z) * n + y) * n + x) * OWN + (cv - UP / 8) * 8);
}

// ------------------------------------------------------------- conv fwd ---
// Y = conv3x3x3(X) + bias, optional ReLU.  W is [Cout][Kp] BF16 (k = tap*Cin+ci,
// zero padded to Kp, a multiple of 32).
// LDS-staged forward conv for the layer shapes of the network.  A workgroup
// owns 16 (x) x TY (y) x TZ (z) output points of one batch element; the input
// block with its one-point halo and all CIN channels is staged in LDS once
// (zeros outside the grid), so a lane's B fragment (8 channels of one tap at
// one point) is a single ds_read_b128 with no bounds checks.  Each of the
// four wavefronts computes NT = TY*TZ/4 rows of 16 points (rows w*NT .. of the
// tile, y fastest) for all MT channel tiles: every weight fragment (read from
// the L1/L2-resident weights) feeds NT MFMAs and every input fragment MT.
// The four accumulators of a lane (output channels 4g..4g+3 of one point) are
// biased, rectified, rounded to BF16 and written as one 8-byte store.
template <int MT, int CIN, int TY, int TZ>
__global__ void __launch_bounds__(256) conv3_fwd_lds_kernel(const bf16 *__restrict__ X, const bf16 *__restrict__ Xup,
                                                            const bf16 *__restrict__ W,
                                                            int Kp, const float *__restrict__ bias,
                                                            bf16 *__restrict__ Y, int n, int nbx, int nby, int nbz,
                                                            int relu, const bf16 *__restrict__ mask) {
    constexpr int HX = 18, HY = TY + 2, HZ = TZ + 2, NV = CIN / 8;
    constexpr int NT = TY * TZ / 4;
    static_assert(CIN % 8 == 0 && (TY * TZ) % 4 == 0, "shape");
    __shared__ bf16x8 blk[HZ * HY * HX * NV];
    int bid = blockIdx.x;
    const int bx = bid % nbx;
    bid /= nbx;
    const int by = bid % nby;
    bid /= nby;
    const int bz = bid % nbz;
    const int b = bid / nbz;
    const int x0 = bx * 16, y0 = by * TY, z0 = bz * TZ;
    const bf16x8 zero8 = {(bf16)0.0f, (bf16)0.0f, (bf16)0.0f, (bf16)0.0f,
                          (bf16)0.0f, (bf16)0.0f, (bf16)0.0f, (bf16)0.0f};
    // (the loads of U vectors go out before the first of them is stored: one after the other they would
    // each wait out the latency of the memory)
    constexpr int TOTAL = HZ * HY * HX * NV, TURNS = (TOTAL + 255) / 256, U = TURNS < 6 ? TURNS : 6;
#pragma unroll
    for (int i0 = 0; i0 < TURNS; i0 += U) {
        bf16x8 val[U];
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const int v = threadIdx.x + (i0 + i) * 256;
            const int cv = v % NV, cx = v / NV % HX, cy = v / (NV * HX) % HY, cz = v / (NV * HX * HY);
            const int gx = x0 - 1 + cx, gy = y0 - 1 + cy, gz = z0 - 1 + cz;
            val[i] = zero8;
            if (v < TOTAL && gx >= 0 && gx < n && gy >= 0 && gy < n && gz >= 0 && gz < n)
                val[i] = input8<CIN>(X, Xup, n, b, gz, gy, gx, cv);
        }
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const int v = threadIdx.x + (i0 + i) * 256;
            if (v < TOTAL) blk[v] = val[i];
        }
    }
    __syncthreads();
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int nl = lane & 15, g = lane >> 4;
    int ty[NT], tz[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        ty[t] = (w * NT + t) % TY;
        tz[t] = (w * NT + t) / TY;
    }
    constexpr int K = 27 * CIN, KPC = (K + 31) / 32 * 32;  // Kp == KPC (checked by the host)
    f32x4 acc[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    // a compile-time trip count, unrolled by eight: the weight loads of eight k steps go out
    // together instead of one L2 round trip per k step
#pragma unroll 8
    for (int kb = 0; kb < KPC; kb += 32) {
        const int k = kb + 8 * g;
        bf16x8 av[MT];
#pragma unroll
        for (int m = 0; m < MT; ++m) av[m] = *reinterpret_cast<const bf16x8 *>(W + (size_t)(m * 16 + nl) * Kp + k);
        const bool kin = k < K;
        const int tap = kin ? k / CIN : 26;  // the zero-padded tail of K reads a valid slot, then discards it
        const int ci8 = kin ? (k % CIN) / 8 : 0;
        const int dz = tap / 9, dy = (tap / 3) % 3, dx = tap % 3;  // offsets + 1
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            bf16x8 bv = blk[(((tz[t] + dz) * HY + (ty[t] + dy)) * HX + (nl + dx)) * NV + ci8];
            if (!kin) bv = zero8;
#pragma unroll
            for (int m = 0; m < MT; ++m) acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[m], bv, acc[m][t], 0, 0, 0);
        }
    }
    // D[4g+i][nl]: output channel m*16 + 4g + i of point (x0 + nl, y0 + ty[t], z0 + tz[t])
    constexpr int Cout = MT * 16;
    const int x = x0 + nl;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int y = y0 + ty[t], z = z0 + tz[t];
        if (x >= n || y >= n || z >= n) continue;
        const size_t p = (((size_t)b * n + z) * n + y) * n + x;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            bf16x4 o;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float v = acc[m][t][i] + (bias ? bias[m * 16 + 4 * g + i] : 0.f);
                if (relu && v < 0.f) v = 0.f;
                o[i] = f2bf(v);
            }
            if (mask) {  // ReLU backward: zero where the forward activation was not positive
                const bf16x4 mk = *reinterpret_cast<const bf16x4 *>(mask + p * Cout + m * 16 + 4 * g);
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (!(bf2f(mk[i]) > 0.f)) o[i] = (bf16)0.0f;
            }
            *reinterpret_cast<bf16x4 *>(Y + p * Cout + m * 16 + 4 * g) = o;
        }
    }
}

// Forward conv with the three x taps in three accumulators, for rows of at
// most 64 points.  A workgroup owns whole x rows (NXT 16-point tiles, zeros
// beyond n) of TY x TZ (y, z) rows of one batch element and stages their
// (TY+2) x (TZ+2) input rows, all CIN channels, in LDS; no x halo is needed.
// K runs over the nine (dz, dy) taps and the channels, k = (3 dz + dy) CIN + ci
// (a lane's 8 values: 8 channels of one tap).  Per 32-wide k block a lane reads
// ONE input fragment, X at its own point x, rows y + dy, z + dz, and feeds it to
// the three dx taps with their own weight fragments W[co][(3 (3 dz + dy) + dx) CIN
// + ci]: acc[dx] at x collects the terms of X[x] that belong to output
// Y[x + 1 - dx].  After the k loop Y[x] = acc[1][x] + acc[0][x - 1] + acc[2][x + 1]
// (zero past the row ends: the padding there is zero): a DPP row shift per value,
// the lane across a 16-point tile edge taken from the neighbouring tile by a row
// rotation.  Per input fragment read from LDS the wavefront issues 3 MT MFMAs,
// against MT when the x taps are separate k values.  RPW rows per wavefront; the
// k loop unrolled by KU.
template <int MT, int CIN, int TY, int TZ, int NXT, int NW, int KU>
__global__ void __launch_bounds__(64 * NW) conv3_fwd_xacc_kernel(const bf16 *__restrict__ X,
                                                                 const bf16 *__restrict__ Xup,
                                                                 const bf16 *__restrict__ W, int Kp,
                                                                 const float *__restrict__ bias,
                                                                 bf16 *__restrict__ Y, int n, int nby, int nbz,
                                                                 int relu, const bf16 *__restrict__ mask) {
    constexpr int XW = NXT * 16, HY = TY + 2, HZ = TZ + 2, NV = CIN / 8;
    constexpr int RPW = TY * TZ / NW;
    constexpr int K9 = 9 * CIN, KB = (K9 + 31) / 32;
    static_assert(CIN % 8 == 0 && (TY * TZ) % NW == 0, "shape");
    __shared__ bf16x8 blk[HZ * HY * XW * NV];
    int bid = blockIdx.x;
    const int by = bid % nby;
    bid /= nby;
    const int bz = bid % nbz;
    const int b = bid / nbz;
    const int y0 = by * TY, z0 = bz * TZ;
    const bf16x8 zero8 = {(bf16)0.0f, (bf16)0.0f, (bf16)0.0f, (bf16)0.0f,
                          (bf16)0.0f, (bf16)0.0f, (bf16)0.0f, (bf16)0.0f};
    constexpr int TOTAL = HZ * HY * XW * NV, TURNS = (TOTAL + 64 * NW - 1) / (64 * NW), U = TURNS < 6 ? TURNS : 6;
#pragma unroll
    for (int i0 = 0; i0 < TURNS; i0 += U) {  // (U loads in flight)
        bf16x8 val[U];
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const int v = threadIdx.x + (i0 + i) * 64 * NW;
            const int cv = v % NV, cx = v / NV % XW, cy = v / (NV * XW) % HY, cz = v / (NV * XW * HY);
            const int gy = y0 - 1 + cy, gz = z0 - 1 + cz;
            val[i] = zero8;
            if (v < TOTAL && cx < n && gy >= 0 && gy < n && gz >= 0 && gz < n)
                val[i] = input8<CIN>(X, Xup, n, b, gz, gy, cx, cv);
        }
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const int v = threadIdx.x + (i0 + i) * 64 * NW;
            if (v < TOTAL) blk[v] = val[i];
        }
    }
    __syncthreads();
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int nl = lane & 15, g = lane >> 4;
    int ry[RPW], rz[RPW];
#pragma unroll
    for (int r = 0; r < RPW; ++r) {
        ry[r] = (w * RPW + r) % TY;
        rz[r] = (w * RPW + r) / TY;
    }
    f32x4 acc[3][MT][RPW][NXT];
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int r = 0; r < RPW; ++r)
#pragma unroll
                for (int t = 0; t < NXT; ++t) acc[d][m][r][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    const bf16 *wrow = W + (size_t)nl * Kp;
#pragma unroll KU
    for (int kb = 0; kb < KB; ++kb) {
        const int k = kb * 32 + 8 * g;
        // (K9 not a multiple of 32: the tail lanes read tap 8's fragment, then zero it)
        const bool kin = K9 % 32 == 0 || k < K9;
        const int dzdy = kin ? k / CIN : 8;
        const int ci = kin ? k % CIN : 0;
        const int dz = dzdy / 3, dy = dzdy % 3;
        bf16x8 av[3][MT];
#pragma unroll
        for (int d = 0; d < 3; ++d)
#pragma unroll
            for (int m = 0; m < MT; ++m)
                av[d][m] = *reinterpret_cast<const bf16x8 *>(wrow + (size_t)m * 16 * Kp + (dzdy * 3 + d) * CIN + ci);
#pragma unroll
        for (int r = 0; r < RPW; ++r)
#pragma unroll
            for (int t = 0; t < NXT; ++t) {
                bf16x8 bv = blk[(((rz[r] + dz) * HY + (ry[r] + dy)) * XW + t * 16 + nl) * NV + ci / 8];
                if (!kin) bv = zero8;
#pragma unroll
                for (int d = 0; d < 3; ++d)
#pragma unroll
                    for (int m = 0; m < MT; ++m)
                        acc[d][m][r][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[d][m], bv, acc[d][m][r][t], 0, 0, 0);
            }
    }
    // D[4g+i][nl] of tile t: output channel m*16 + 4g + i at x = 16 t + nl
    constexpr int Cout = MT * 16;
#pragma unroll
    for (int r = 0; r < RPW; ++r) {
        const int y = y0 + ry[r], z = z0 + rz[r];
#pragma unroll
        for (int t = 0; t < NXT; ++t) {
            const int x = t * 16 + nl;
            const bool out = x < n && y < n && z < n;
            const size_t p = (((size_t)b * n + z) * n + y) * n + x;
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                bf16x4 o;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    // (each element copied to a float first: a bit cast of a vector element
                    // subscript reads element 0 in this compiler)
                    const float c0 = acc[0][m][r][t][i], c2 = acc[2][m][r][t][i];
                    const float p0 = t > 0 ? acc[0][m][r][t > 0 ? t - 1 : 0][i] : 0.f;
                    const float q2 = t + 1 < NXT ? acc[2][m][r][t + 1 < NXT ? t + 1 : t][i] : 0.f;
                    // acc[0] one point to the left: lane nl-1 of this tile (row_shr:1), lane 15 of
                    // tile t-1 for nl = 0 (row_ror:1 brings lane 15 of each 16-lane row to lane 0)
                    const int l0 = t > 0 ? __builtin_amdgcn_mov_dpp(__float_as_int(p0), 0x121 /* row_ror:1 */, 0xf, 0xf,
                                                                    false)
                                         : 0;
                    const int s0 = __builtin_amdgcn_update_dpp(l0, __float_as_int(c0), 0x111 /* row_shr:1 */, 0xf,
                                                               0xf, false);
                    // acc[2] one point to the right: lane nl+1 (row_shl:1), lane 0 of tile t+1 for
                    // nl = 15 (row_ror:15 brings lane 0 to lane 15)
                    const int l2 = t + 1 < NXT ? __builtin_amdgcn_mov_dpp(__float_as_int(q2), 0x12f /* row_ror:15 */,
                                                                          0xf, 0xf, false)
                                               : 0;
                    const int s2 = __builtin_amdgcn_update_dpp(l2, __float_as_int(c2), 0x101 /* row_shl:1 */, 0xf,
                                                               0xf, false);
                    float v = acc[1][m][r][t][i] + __int_as_float(s0) + __int_as_float(s2);
                    v += bias ? bias[m * 16 + 4 * g + i] : 0.f;
                    if (relu && v < 0.f) v = 0.f;
                    o[i] = f2bf(v);
                }
                if (out) {
                    if (mask) {  // ReLU backward: zero where the forward activation was not positive
                        const bf16x4 mk = *reinterpret_cast<const bf16x4 *>(mask + p * Cout + m * 16 + 4 * g);
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            if (!(bf2f(mk[i]) > 0.f)) o[i] = (bf16)0.0f;
                    }
                    *reinterpret_cast<bf16x4 *>(Y + p * Cout + m * 16 + 4 * g) = o;
                }
            }
        }
    }
}

// ------------------------------------------------------ conv weight grad ---
// Weight and bias gradients, every tap at once: workgroup s computes
// partial[s][co][tap*CIN + ci] (and the sums of dZ, partial[s][COUT*Kp + co]) over its blocks.
// A block is 64 points: R rows of at most 64 points of one plane, each padded to
// a multiple of 8 (rows longer than 64 points go in segments), with zero dZ where
// a point lies outside.  Per block it stages dZ once, transposed [co][point], and
// the 3 x (R+2) input rows around the block once, transposed [ci][x] with the
// columns x0 - 1 and x0 + W8 at the ends: the tap-shifted input of every tap is
// then a window of those rows, so nothing is staged per tap.  Wavefront w owns
// the taps of WROWS (dz, dy) rows; a lane's B fragment (8 consecutive points of
// one input channel, shifted by dx) comes from two aligned 16-byte LDS reads:
// dx = -1 is the first, dx = +1 the dwords 1..4, dx = 0 a 2-byte byte-align of
// the pair.  Input channels below 16 are padded with zero rows (the first layer's
// 8).  The bias gradient is one more product, with a B fragment of ones; every kBiasBlocks blocks its
// sums go to FP64 ones in LDS.
// blockIdx.y: the group of 16 input channels that the workgroup stages and computes.
// Bound by latency and by the vector instructions of the staging: blocks follow one another along y,
// the rows that the last block had stay in LDS, the new ones and the next dZ are loaded while a block is
// multiplied, and where an item comes from and goes to is worked out once.  At 4 x 64^3, 48 -> 16:
// 447 us with every block staged on its own, 261 with the rows kept, 161 us with the channels split and the items
// kept; 16 -> 16 102, 72 and 52.  Other row lengths than 16, 32 and 64 went through a kernel that
// staged the input anew for each of the 27 taps.
constexpr int kWgradRow = 72;  // a staged input row: 64 points, one at each end, and padding that keeps fragments 16-byte aligned
constexpr int kWgradRows16 = 16 * (kWgradRow + 1);  // and that of 16 channels
constexpr int kBiasBlocks = 8;
struct WgradShape {
    int n, nblk, per_slab;  // points along an edge; blocks, and blocks a workgroup takes
    int w8, rows, nyb, nseg;  // a row's padded points, rows of a block, blocks along y and x
    float inv_pairs;          // 1 / (w8 / 2 + 1)
};

template <int CIN, int COUT>
__global__ void __launch_bounds__(192, COUT == 16 ? 3 : 1) conv3_wgrad_rows_kernel(const bf16 *__restrict__ Xg,
                                                                        const bf16 *__restrict__ Xup,
                                                                        const bf16 *__restrict__ dZ, int Kp,
                                                                        float *__restrict__ partial, WgradShape S) {
    constexpr int UP = upsampled_channels(CIN), CINX = CIN - UP;  // channels per point of the input tensor(s)
    constexpr int CW = CIN < 16 ? CIN : 16;  // input channels of this workgroup
    constexpr int CINP = 16;                 // and as many rows as a fragment has
    constexpr int MT = COUT / 16, WROWS = 3, NTH = 192;
    static_assert(CIN % CW == 0, "channel split");
    const int ci0 = blockIdx.y * CW;
    const bool up = ci0 < UP;  // (uniform; UP is a multiple of 16)
    const bf16 *X = up ? Xup + ci0 : Xg + (ci0 - UP);
    constexpr int DS = 72;  // dZ row stride (64 points + 8: spreads the 16 rows of a fragment over the banks)
    static_assert(COUT % 16 == 0 && CW % 8 == 0, "shape");
    extern __shared__ __attribute__((aligned(16))) bf16 wg_lds[];
    const int n = S.n, W8 = S.w8, R = S.rows;
    bf16 *dzT = wg_lds;                 // [COUT][DS]
    // [3 planes][R + 2 rows][16 channels][W], x stored at column x - x0 + 1, with 8 elements more after
    // every 8 channels: the column pairs of the two groups, which one store writes together, then lie on
    // different banks
    bf16 *xT = wg_lds + COUT * DS;
    constexpr int W = kWgradRow, RSTR = CINP * (W + 1);
    static_assert(RSTR == kWgradRows16, "as the launch counts it");
    double *biasT = reinterpret_cast<double *>(xT + 3 * (R + 2) * RSTR);  // [COUT], a lane's own each
    const int s = blockIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int nl = lane & 15, g = lane >> 4;
    const bf16x8 one8 = {(bf16)1.0f, (bf16)1.0f, (bf16)1.0f, (bf16)1.0f,
                         (bf16)1.0f, (bf16)1.0f, (bf16)1.0f, (bf16)1.0f};
    if (CW < CINP) {  // padded input channels: zero once, never overwritten
        for (int v = threadIdx.x; v < 3 * (R + 2) * (CINP - CW) * W; v += NTH) {
            const int c = CW + (v / W) % (CINP - CW), r = v / (W * (CINP - CW));
            xT[r * RSTR + c * W + (c >> 3) * 8 + v % W] = (bf16)0.0f;
        }
    }
    f32x4 acc[WROWS][3][MT], accb[MT];
#pragma unroll
    for (int a = 0; a < WROWS; ++a)
#pragma unroll
        for (int d = 0; d < 3; ++d)
#pragma unroll
            for (int m = 0; m < MT; ++m) acc[a][d][m] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int m = 0; m < MT; ++m) accb[m] = f32x4{0.f, 0.f, 0.f, 0.f};
    const bool bias = w == 0 && blockIdx.y == 0;  // (uniform over the wavefront)
    if (bias && nl == 0)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int i = 0; i < 4; ++i) biasT[m * 16 + 4 * g + i] = 0.0;
    // this lane's first point in each of the two K steps: its row in the block and its column (a
    // group beyond the last row multiplies zeros of dZ with any staged row)
    int rq[2], xg[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int q = 32 * h + 8 * g;
        rq[h] = q / W8;
        xg[h] = q - rq[h] * W8;
        if (rq[h] >= R) rq[h] = 0;
    }
    // Two neighbouring points' 8 channels, transposed into LDS: each 4-byte store writes one channel's pair.
    struct Pair {
        u16x8 p[2];
    };
    const auto put = [](bf16 *to, int stride, const Pair &v) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            *reinterpret_cast<unsigned *>(to + i * stride) = (unsigned)v.p[0][i] | ((unsigned)v.p[1][i] << 16);
    };
    // 8 channels of a point that lies `off` bytes from `p`; zeros if it is not there
    const auto get = [](const bf16 *p, int bytes, int off, bool there) {
        const auto r = __builtin_amdgcn_make_buffer_rsrc((void *)p, (short)0, bytes, 0x00020000);
        return __builtin_bit_cast(u16x8, __builtin_amdgcn_raw_buffer_load_b128(r, there ? off : -16, 0, 0));
    };
    // dZ of a block: a pair of points of 8 channels an item
    constexpr int ZITEMS = 32 * (COUT / 8), NZ = (ZITEMS + NTH - 1) / NTH;
    struct ZItem {
        int lds, off, row, x;  // where it goes; where it comes from, from point (x0, y0) on; which point it is
    } zi[NZ];
#pragma unroll
    for (int i = 0; i < NZ; ++i) {
        const int v = threadIdx.x + i * NTH, j = 2 * (v / (COUT / 8)), c8 = v % (COUT / 8);
        const int row = j / W8, x = j - row * W8;
        zi[i] = {8 * c8 * DS + j, ((row * n + x) * COUT + 8 * c8) * 2, v < ZITEMS && row < R ? row : n, x};
    }
    const auto get_dz = [&](const ZItem &t, int x0, int y0, int z, int b) {
        const bf16 *from = dZ + ((((size_t)b * n + z) * n + y0) * n + x0) * COUT;
        const bool row = y0 + t.row < n;
        Pair o;
#pragma unroll
        for (int e = 0; e < 2; ++e)
            o.p[e] = get(from, 64 * n * COUT * 2, t.off + e * COUT * 2, row && x0 + t.x + e < n);
        return o;
    };
    const auto put_dz = [&](int i, const Pair &o) {
        if ((int)threadIdx.x + i * NTH < ZITEMS) put(dzT + zi[i].lds, DS, o);
    };
    // Input rows, 8 channels of a pair of columns an item.  Row y is kept at y + 1 modulo R + 2 of its
    // plane's rows, so a block needs only the R rows that the block before it did not have.
    const int pairs = W8 / 2 + 1;
    struct XItem {
        int lds, off, plane, row, x, c;  // as above, from (x0, first row, z) on; the plane's offset -1, 0, 1
    };
    const auto x_item = [&](int v, int rows) {
        const int c8 = v % (CW / 8), pr = v / (CW / 8);
        const int r = (int)(((float)pr + 0.5f) * S.inv_pairs);  // pr / pairs, exact below 2^20
        const int xj = 2 * (pr - r * pairs), dz = r >= 2 * rows ? 2 : r >= rows ? 1 : 0, row = r - dz * rows;
        return XItem{dz * (R + 2) * RSTR + c8 * (8 * W + 8) + xj, ((row * n + xj - 1) * CINX + 8 * c8) * 2,
                     v < 3 * rows * pairs * (CW / 8) ? dz - 1 : n + 1, row, xj - 1, 8 * c8};
    };
    const auto get_x = [&](const XItem &t, int x0, int y, int z, int b) {
        const bool there = z + t.plane >= 0 && z + t.plane < n && y + t.row >= 0 && y + t.row < n;
        Pair o;
        if (UP > 0 && up) {
            const int m = n / 2;
            const unsigned line = (unsigned)((b * m + ((z + t.plane) >> 1)) * m + ((y + t.row) >> 1)) * m;
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int x = x0 + t.x + e;
                o.p[e] = get(X, 0x7fffffff, (int)(((line + (x >> 1)) * UP + t.c) * 2), there && x >= 0 && x < n);
            }
            return o;
        }
        // (an offset below zero, the column before x0, is within the tensor wherever it is read)
        const bf16 *from = X + ((((size_t)b * n + z) * n + y) * n + x0 - 1) * CINX - n * n * CINX;
        const unsigned off = (unsigned)t.off + CINX * 2 + (unsigned)(t.plane + 1) * (unsigned)(n * n * CINX * 2);
#pragma unroll
        for (int e = 0; e < 2; ++e)
            o.p[e] = get(from, 0x7fffffff, (int)(off + e * CINX * 2), there && x0 + t.x + e >= 0 && x0 + t.x + e < n);
        return o;
    };
    const auto put_x = [&](const XItem &t, int base, const Pair &o) {
        const int slot = base + t.row >= R + 2 ? base + t.row - (R + 2) : base + t.row;
        if (t.plane <= 1) put(xT + t.lds + slot * RSTR, W, o);
    };
    // the next block's new rows and dZ wait in registers while this block is multiplied: R <= 8 rows of
    // R (W8 / 2 + 1) <= 40 pairs
    constexpr int NX = (3 * 40 * (CW / 8) + NTH - 1) / NTH;
    XItem xi[NX];
#pragma unroll
    for (int i = 0; i < NX; ++i) xi[i] = x_item(threadIdx.x + i * NTH, R);
    Pair pz[NZ], px[NX];
    const int blk_end = min(S.nblk, (s + 1) * S.per_slab);
    bool fresh = true;  // nothing of the block's rows is staged yet
    for (int blk = s * S.per_slab; blk < blk_end; ++blk) {
        int u = blk;
        const int yb = u % S.nyb, y0 = yb * R;
        u /= S.nyb;
        const int x0 = (u % S.nseg) * 64;
        u /= S.nseg;
        const int z = u % n, b = u / n;
        const int base = y0 % (R + 2);  // where row y0 - 1 is kept
        if (fresh) {
#pragma unroll
            for (int i = 0; i < NZ; ++i) put_dz(i, get_dz(zi[i], x0, y0, z, b));
            constexpr int U = 4;  // loads of four items in flight
            for (int v = threadIdx.x; v < 3 * (R + 2) * pairs * (CW / 8); v += U * NTH) {
                XItem t[U];
                Pair p[U];
#pragma unroll
                for (int i = 0; i < U; ++i) {
                    t[i] = x_item(v + i * NTH, R + 2);
                    p[i] = get_x(t[i], x0, y0 - 1, z, b);
                }
#pragma unroll
                for (int i = 0; i < U; ++i) put_x(t[i], base, p[i]);
            }
        }
        __syncthreads();
        fresh = yb + 1 == S.nyb;
        const bool more = !fresh && blk + 1 < blk_end;
        if (more) {
#pragma unroll
            for (int i = 0; i < NZ; ++i) pz[i] = get_dz(zi[i], x0, y0 + R, z, b);
#pragma unroll
            for (int i = 0; i < NX; ++i) px[i] = get_x(xi[i], x0, y0 + R + 1, z, b);
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {  // two K steps of 32 points
            const int q = 32 * h + 8 * g;  // this lane's first point in the block
            bf16x8 av[MT];
#pragma unroll
            for (int m = 0; m < MT; ++m) av[m] = *reinterpret_cast<const bf16x8 *>(&dzT[(m * 16 + nl) * DS + q]);
            if (bias) {
#pragma unroll
                for (int m = 0; m < MT; ++m)
                    accb[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[m], one8, accb[m], 0, 0, 0);
            }
#pragma unroll
            for (int a = 0; a < WROWS; ++a) {
                const int rw = w * WROWS + a;  // (dz, dy) row index 0..8
                const int dz = rw / 3, dy = rw % 3;  // offsets + 1
                int slot = base + rq[h] + dy;
                if (slot >= R + 2) slot -= R + 2;
                const bf16 *src = xT + (dz * (R + 2) + slot) * RSTR + nl * W + (nl >> 3) * 8 + xg[h];
                const bf16x8 lo = *reinterpret_cast<const bf16x8 *>(src);
                const bf16x8 hi = *reinterpret_cast<const bf16x8 *>(src + 8);
                typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
                const u32x4 l4 = __builtin_bit_cast(u32x4, lo), h4 = __builtin_bit_cast(u32x4, hi);
                const u32x4 mid = {__builtin_amdgcn_alignbyte(l4[1], l4[0], 2),
                                   __builtin_amdgcn_alignbyte(l4[2], l4[1], 2),
                                   __builtin_amdgcn_alignbyte(l4[3], l4[2], 2),
                                   __builtin_amdgcn_alignbyte(h4[0], l4[3], 2)};
                const u32x4 up = {l4[1], l4[2], l4[3], h4[0]};
                const bf16x8 bv[3] = {lo, __builtin_bit_cast(bf16x8, mid), __builtin_bit_cast(bf16x8, up)};
#pragma unroll
                for (int d = 0; d < 3; ++d)
#pragma unroll
                    for (int m = 0; m < MT; ++m)
                        acc[a][d][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[m], bv[d], acc[a][d][m], 0, 0, 0);
            }
        }
        if (bias && ((blk - s * S.per_slab) % kBiasBlocks == kBiasBlocks - 1 || blk + 1 == blk_end)) {
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                if (nl == 0)
#pragma unroll
                    for (int i = 0; i < 4; ++i) biasT[m * 16 + 4 * g + i] += (double)accb[m][i];
                accb[m] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
        }
        __syncthreads();  // the staged rows are rewritten next
        if (more) {
#pragma unroll
            for (int i = 0; i < NZ; ++i) put_dz(i, pz[i]);
            // (row y0 + R + 1 is row R + 2 from y0 - 1 on: kept where that was)
#pragma unroll
            for (int i = 0; i < NX; ++i) put_x(xi[i], base, px[i]);
        }
    }
    // D[4g+i][nl] = dW[m*16 + 4g + i][tap*CIN + ci0 + nl], tap = 9 dz + 3 dy + dx (offsets + 1)
    float *out = partial + (size_t)s * COUT * (Kp + 1);
#pragma unroll
    for (int a = 0; a < WROWS; ++a) {
        const int rw = w * WROWS + a;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const int tap = 3 * rw + d;
#pragma unroll
            for (int m = 0; m < MT; ++m)
                if (nl < CW)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        out[(size_t)(m * 16 + 4 * g + i) * Kp + tap * CIN + ci0 + nl] = acc[a][d][m][i];
        }
    }
    // (the K tail [27 CIN, Kp) is left as it is: nothing reads it)
    if (bias && nl == 0) {
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                out[(size_t)COUT * Kp + m * 16 + 4 * g + i] = (float)biasT[m * 16 + 4 * g + i];
    }
}

// The slabs' sums, part[s][i] in the fixed order s = 0, 1, ..., for i < COUT (Kp + 1), taken
// from the kernel layout (co, k = tap*Cin + ci; then the bias) to the master order [Cout][Cin_real][27]
// and [Cout].  In FP64: there may be thousands of slabs, and the sums are bound by the loads.  Eight
// loads are issued before their eight in-order adds, so the memory latency is
// paid once per eight slabs instead of once per slab.
template <typename T>
__global__ void reduce_slabs_kernel(const T *__restrict__ part, int nslab, int Cout, int Cin_real, int Cin, int Kp,
                                    float *__restrict__ g, float *__restrict__ gb) {
    const int count = Cout * (Kp + 1);
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    const bool bias = i >= Cout * Kp;
    const int co = i / Kp, k = i - co * Kp;
    const int tap = k / Cin, ci = k - tap * Cin;
    if (!bias && (tap >= 27 || ci >= Cin_real)) return;  // the K tail, padded input channels
    double a = 0.0;
    int s = 0;
    for (; s + 8 <= nslab; s += 8) {
        T v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = part[(size_t)(s + j) * count + i];
#pragma unroll
        for (int j = 0; j < 8; ++j) a += (double)v[j];
    }
    for (; s < nslab; ++s) a += (double)part[(size_t)s * count + i];
    if (bias)
        gb[i - Cout * Kp] = (float)a;
    else
        g[((size_t)co * Cin_real + ci) * 27 + tap] = (float)a;
}

// First pass of a two-pass slab reduction: part p of P sums slabs
// [p*nslab/P, (p+1)*nslab/P) in order into tmp[p][i], so P times more threads
// share the reads; reduce_slabs_kernel then adds the P parts in order (a fixed
// tree: the same bits on every call).
__global__ void reduce_slab_parts_kernel(const float *__restrict__ partial, int nslab, size_t count, int nparts,
                                         double *__restrict__ tmp) {
    const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    const int part = blockIdx.y;
    if (i >= count) return;
    const int s0 = (int)((long long)nslab * part / nparts), s1 = (int)((long long)nslab * (part + 1) / nparts);
    double a = 0.0;
    int s = s0;
    for (; s + 8 <= s1; s += 8) {
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = partial[(size_t)(s + j) * count + i];
#pragma unroll
        for (int j = 0; j < 8; ++j) a += (double)v[j];
    }
    for (; s < s1; ++s) a += (double)partial[(size_t)s * count + i];
    tmp[(size_t)part * count + i] = a;
}

// out[r] = sum of row r of part ([rows][nslab], row-major), one 1024-thread
// workgroup per row: thread t adds s = t, t + 1024, ... in order (eight loads in
// flight), then a fixed pairwise tree over the threads, so every call gives the
// same bits.  For the few-value sums (bias and head gradients) whose slab
// counts run to tens of thousands.
__global__ void __launch_bounds__(1024) reduce_rows_kernel(const float *__restrict__ part, int nslab,
                                                           float *__restrict__ out) {
    __shared__ float sh[1024];
    const float *row = part + (size_t)blockIdx.x * nslab;
    const int t = threadIdx.x;
    float a = 0.f;
    int s = t;
    for (; s + 7 * 1024 < nslab; s += 8 * 1024) {
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = row[s + j * 1024];
#pragma unroll
        for (int j = 0; j < 8; ++j) a += v[j];
    }
    for (; s < nslab; s += 1024) a += row[s];
    sh[t] = a;
    __syncthreads();
    for (int w = 512; w > 0; w >>= 1) {
        if (t < w) sh[t] += sh[t + w];
        __syncthreads();
    }
    if (t == 0) out[blockIdx.x] = sh[0];
}

// --------------------------------------------------------- elementwise ----
// The elementwise kernels below move 8 channels (one 16-byte vector) per
// thread; every channel count and offset of the network is a multiple of 8
// and points number fewer than 2^27, so 32-bit index math suffices.
__device__ __forceinline__ bf16x8 ld8(const bf16 *p) { return *reinterpret_cast<const bf16x8 *>(p); }
__device__ __forceinline__ void st8(bf16 *p, bf16x8 v) { *reinterpret_cast<bf16x8 *>(p) = v; }

// 2x2x2 average pooling: n -> n/2
__global__ void pool_fwd_kernel(const bf16 *__restrict__ X, bf16 *__restrict__ Y, int C, int n, int nb) {
    const unsigned m = n / 2, V = C / 8;
    const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (unsigned)nb * m * m * m * V) return;
    const unsigned cv = i % V, q = i / V;
    const unsigned x = q % m, y = (q / m) % m, z = (q / (m * m)) % m, b = q / (m * m * m);
    float a[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int dz = 0; dz < 2; ++dz)
        for (int dy = 0; dy < 2; ++dy)
            for (int dx = 0; dx < 2; ++dx) {
                const bf16x8 v = ld8(X + ((((size_t)b * n + 2 * z + dz) * n + 2 * y + dy) * n + 2 * x + dx) * C + 8 * cv);
#pragma unroll
                for (int j = 0; j < 8; ++j) a[j] += bf2f(v[j]);
            }
    bf16x8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = f2bf(a[j] * 0.125f);
    st8(Y + (size_t)q * C + 8 * cv, o);
}

// gradient of 2x2x2 average pooling, then (skip != null) plus the skip connection's gradient,
// channels [skip_off, skip_off + C) of a buffer with skip_ct channels, then (mask != null) the
// ReLU backward of the layer that produced the pooled tensor: zero where mask ([points][C]) is
// not positive.  Each step rounds to BF16 as separate kernels would.
__global__ void pool_bwd_kernel(const bf16 *__restrict__ dY, bf16 *__restrict__ dX, int C, int n, int nb,
                                const bf16 *__restrict__ skip, int skip_ct, int skip_off,
                                const bf16 *__restrict__ mask) {
    const unsigned V = C / 8, un = n, m = n / 2;
    const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (unsigned)nb * un * un * un * V) return;
    const unsigned cv = i % V, q = i / V;
    const unsigned x = q % un, y = (q / un) % un, z = (q / (un * un)) % un, b = q / (un * un * un);
    const bf16x8 v = ld8(dY + ((((size_t)b * m + z / 2) * m + y / 2) * m + x / 2) * C + 8 * cv);
    bf16x8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = f2bf(bf2f(v[j]) * 0.125f);
    if (skip) {
        const bf16x8 sk = ld8(skip + (size_t)q * skip_ct + skip_off + 8 * cv);
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j] = f2bf(bf2f(o[j]) + bf2f(sk[j]));
    }
    if (mask) {
        const bf16x8 mk = ld8(mask + (size_t)q * C + 8 * cv);
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (!(bf2f(mk[j]) > 0.f)) o[j] = (bf16)0.0f;
    }
    st8(dX + (size_t)q * C + 8 * cv, o);
}

// gradient of nearest upsampling: sum of the 8 children (from channels [off, off+C) of dY), then
// (mask != null) the ReLU backward of the layer that produced the upsampled tensor
__global__ void up_bwd_kernel(const bf16 *__restrict__ dY, bf16 *__restrict__ dX, int C, int Ct, int off, int m,
                              int nb, const bf16 *__restrict__ mask) {
    const unsigned n = 2 * m, V = C / 8, um = m;
    const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (unsigned)nb * um * um * um * V) return;
    const unsigned cv = i % V, q = i / V;
    const unsigned x = q % um, y = (q / um) % um, z = (q / (um * um)) % um, b = q / (um * um * um);
    float a[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int dz = 0; dz < 2; ++dz)
        for (int dy = 0; dy < 2; ++dy)
            for (int dx = 0; dx < 2; ++dx) {
                const bf16x8 v =
                    ld8(dY + ((((size_t)b * n + 2 * z + dz) * n + 2 * y + dy) * n + 2 * x + dx) * Ct + off + 8 * cv);
#pragma unroll
                for (int j = 0; j < 8; ++j) a[j] += bf2f(v[j]);
            }
    bf16x8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = f2bf(a[j]);
    if (mask) {
        const bf16x8 mk = ld8(mask + (size_t)q * C + 8 * cv);
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (!(bf2f(mk[j]) > 0.f)) o[j] = (bf16)0.0f;
    }
    st8(dX + (size_t)q * C + 8 * cv, o);
}

// input packing: host-order float planes [b][2][n^3] -> NDHWC BF16 with 8 channels (2 used)
__global__ void pack_input_kernel(const float *__restrict__ in, bf16 *__restrict__ X, int n3, int nb) {
    const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    if (i >= (size_t)nb * n3) return;
    const size_t b = i / n3, q = i % n3;
    bf16x8 v;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = (bf16)0.0f;
    v[0] = f2bf(in[(b * 2 + 0) * n3 + q]);
    v[1] = f2bf(in[(b * 2 + 1) * n3 + q]);
    *reinterpret_cast<bf16x8 *>(X + i * 8) = v;
}

// 1x1 head 16 -> 1: out[p] = sum_c w[c] X[p][c] + w[16] (FP32 out)
__global__ void head_fwd_kernel(const bf16 *__restrict__ X, const float *__restrict__ w, float *__restrict__ out,
                                size_t npts) {
    const size_t p = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    if (p >= npts) return;
    float a = w[16];
#pragma unroll
    for (int c = 0; c < 16; ++c) a += w[c] * bf2f(X[p * 16 + c]);
    out[p] = a;
}

// loss = mean((pred - target)^2); dpred = 2 (pred - target) / N  (partials per block)
__global__ void mse_kernel(const float *__restrict__ pred, const float *__restrict__ target, float *__restrict__ dpred,
                           double *__restrict__ lpart, size_t npts) {
    __shared__ double sh[256];
    const size_t p = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    double l = 0.0;
    if (p < npts) {
        const float d = pred[p] - target[p];
        dpred[p] = 2.0f * d / (float)npts;
        l = (double)d * d;
    }
    sh[threadIdx.x] = l;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) sh[threadIdx.x] += sh[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) lpart[blockIdx.x] = sh[0];
}

// head backward: dX[p][c] = dpred[p] w[c] (BF16), zero where X (the ReLU output the head reads)
// is not positive (the ReLU backward of the last conv); per-block partial grads of w (16) and
// b (1), gpart[c][block] (rows for reduce_rows_kernel)
__global__ void head_bwd_kernel(const bf16 *__restrict__ X, const float *__restrict__ w,
                                const float *__restrict__ dpred, bf16 *__restrict__ dX, float *__restrict__ gpart,
                                size_t npts) {
    __shared__ float sh[17][256];
    const size_t p = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    float gw[17];
#pragma unroll
    for (int c = 0; c < 17; ++c) gw[c] = 0.f;
    if (p < npts) {
        const float d = dpred[p];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const bf16x8 x = ld8(X + p * 16 + 8 * h);
            bf16x8 o;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                o[j] = bf2f(x[j]) > 0.f ? f2bf(d * w[8 * h + j]) : (bf16)0.0f;
                gw[8 * h + j] = d * bf2f(x[j]);
            }
            st8(dX + p * 16 + 8 * h, o);
        }
        gw[16] = d;
    }
#pragma unroll
    for (int c = 0; c < 17; ++c) sh[c][threadIdx.x] = gw[c];
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s)
#pragma unroll
            for (int c = 0; c < 17; ++c) sh[c][threadIdx.x] += sh[c][threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x < 17) gpart[(size_t)threadIdx.x * gridDim.x + blockIdx.x] = sh[threadIdx.x][0];
}

// Adam on FP32 master parameters
__global__ void adam_kernel(float *__restrict__ w, const float *__restrict__ g, float *__restrict__ m,
                            float *__restrict__ v, size_t count, float lr, float b1, float b2, float eps, float c1,
                            float c2) {
    const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    if (i >= count) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    w[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// FP32 master conv weights [Cout][Cin_real][27] -> forward layout [Cout][Kp] (k = tap*Cin + ci)
// and backward-data layout [Cin][Kp_t] (k = tap'*Cout + co, tap' = 26 - tap), BF16
// (the padding beyond 27 Cin and 27 Cout was cleared when the arrays were made); every layer in one
// launch, layer blockIdx.y
constexpr int kNConv = 10;
struct PackTable {
    struct Layer {
        const float *w;
        bf16 *Wf, *Wt;
        int Cout, Cin_real, Cin, Kp, Kp_t;
    } layer[kNConv];
};
__global__ void pack_weights_kernel(PackTable T) {
    const PackTable::Layer &L = T.layer[blockIdx.y];
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= L.Cout * L.Cin * 27) return;
    const int tap = i % 27, ci = (i / 27) % L.Cin, co = i / (27 * L.Cin);
    const float v = ci < L.Cin_real ? L.w[((size_t)co * L.Cin_real + ci) * 27 + tap] : 0.f;
    L.Wf[(size_t)co * L.Kp + tap * L.Cin + ci] = f2bf(v);
    if (L.Wt) L.Wt[(size_t)ci * L.Kp_t + (26 - tap) * L.Cout + co] = f2bf(v);
}

}  // namespace unet
}  // namespace cfm

using namespace cfm;
using namespace cfm::unet;

namespace {

// Layer table: 10 3x3x3 convolutions (+ReLU) and a 1x1 head.
struct ConvSpec {
    int cin_real, cin, cout, level;
};
constexpr ConvSpec kConv[kNConv] = {
    {2, 8, 16, 0},   {16, 16, 16, 0},  // encoder level 1 (input padded to 8 channels)
    {16, 16, 32, 1}, {32, 32, 32, 1},  // encoder level 2
    {32, 32, 64, 2}, {64, 64, 64, 2},  // bottleneck
    {96, 96, 32, 1}, {32, 32, 32, 1},  // decoder level 2 (64 upsampled + 32 skip)
    {48, 48, 16, 0}, {16, 16, 16, 0},  // decoder level 1 (32 upsampled + 16 skip)
};
constexpr int kHeadIn = 16;

inline int pad32(int k) { return (k + 31) / 32 * 32; }

constexpr int kReduceParts = 16;  // parts of the first pass of the slab reductions
// Blocks of 64 points that a weight gradient's workgroup adds up in FP32; the workgroups' sums are added
// in FP64.  Against the FP64 mean of single samples' gradients (rms, relative, the worst layer): 4 x 64^3
// 6.5e-8, 32 x 64^3 5.5e-8, 128 x 64^3 5.1e-8; with 512 workgroups at any batch and FP32 throughout
// 1.8e-7, 2.7e-7 and 8.6e-7.  Training steps 2.16 -> 2.15, 13.0 -> 12.2 ms at 4 and 32 x 64^3.
constexpr int kSlabBlocks = 64;

size_t param_count() {
    size_t c = 0;
    for (const auto &s : kConv) c += (size_t)s.cout * s.cin_real * 27 + s.cout;
    return c + kHeadIn + 1;
}

// Blocks of 64 points of a layer's weight gradient, and the workgroups that share them: 512, two a CU, with
// the groups of 16 input channels counted (a workgroup that goes on to the next rows stages a third of
// them anew, and more workgroups write and re-read more partials), or up to 1024 where 512 would take
// fewer than 8 blocks each.  Training steps, ms, for 512 / 1024 / 2048 workgroups: 4 x 64^3 2.15, 2.23, 2.28;
// 8 x 36^3 1.47, 1.50, 1.55; 16 x 12^3 0.80, 0.73, 0.73.  A workgroup adds up at most kSlabBlocks blocks in
// FP32, for the sums' precision; larger layers take a multiple of 512 workgroups.
WgradShape wgrad_shape(int n, int batch, int cin, int *nslab) {
    WgradShape S;
    S.n = n;
    S.w8 = n >= 64 ? 64 : (n + 7) / 8 * 8;
    S.rows = 64 / S.w8;
    S.nyb = (n + S.rows - 1) / S.rows;
    S.nseg = (n + 63) / 64;
    S.nblk = batch * n * S.nyb * S.nseg;
    S.inv_pairs = 1.0f / (float)(S.w8 / 2 + 1);
    const int groups = (cin + 15) / 16;
    const long long work = S.nblk * (long long)groups;
    const long long turns = (work + 512 * kSlabBlocks - 1) / (512 * kSlabBlocks);
    const int most = std::max(1, (int)((work >= 8 * 512 ? 512 * turns : 1024) / groups));
    S.per_slab = std::min((S.nblk + most - 1) / most, kSlabBlocks);
    *nslab = (S.nblk + S.per_slab - 1) / S.per_slab;
    return S;
}

inline dim3 blocks_for(size_t count, int threads = 256) { return dim3((unsigned)((count + threads - 1) / threads)); }

}  // namespace

struct cfm_unet {
    int n = 0, batch = 0;
    size_t P[3] = {0, 0, 0};  // points per level (batch included)
    hipStream_t stream = nullptr, copies = nullptr;  // kernels; transfers that run beside them
    hipEvent_t copied = nullptr, done[2] = {nullptr, nullptr};
    // parameters
    float *master = nullptr, *grad = nullptr, *adam_m = nullptr, *adam_v = nullptr;
    size_t nparam = 0;
    size_t woff[kNConv], boff[kNConv], head_off = 0;
    bf16 *Wf[kNConv] = {}, *Wt[kNConv] = {};
    int Kp[kNConv], Kpt[kNConv];
    double *rtmp = nullptr;  // two-pass slab reduction: [kReduceParts][largest layer]
    float *partial = nullptr;
    // activations
    bf16 *X0 = nullptr, *A0 = nullptr, *S1 = nullptr, *Q1 = nullptr, *A2 = nullptr, *S2 = nullptr, *Q2 = nullptr,
         *A4 = nullptr, *A5 = nullptr, *A6 = nullptr, *A7 = nullptr, *A8 = nullptr,
         *A9 = nullptr;
    float *pred = nullptr, *target = nullptr, *dpred = nullptr, *in_f = nullptr;
    double *lpart = nullptr;
    float *hpart = nullptr;
    // gradients of activations (BF16), sized for the largest of each level
    bf16 *g1a = nullptr, *g1b = nullptr, *g1c = nullptr;  // level 1, up to 48 channels
    bf16 *g2a = nullptr, *g2b = nullptr, *g2c = nullptr;  // level 2, up to 96 channels
    bf16 *g3a = nullptr, *g3b = nullptr;                                   // level 3, 64 channels
    long long step = 0;
    std::vector<void *> allocs;
};

static cfm_status unet_alloc(cfm_unet *u, void **p, size_t bytes) {
    if (hipMalloc(p, bytes ? bytes : 16) != hipSuccess) return CFM_ENOMEM;
    u->allocs.push_back(*p);
    return CFM_OK;
}

extern "C" void cfm_unet_destroy(cfm_unet *u) {
    if (!u) return;
    if (u->copies) (void)hipStreamSynchronize(u->copies);
    if (u->stream) (void)hipStreamSynchronize(u->stream);
    for (void *p : u->allocs) (void)hipFree(p);
    for (hipEvent_t e : {u->copied, u->done[0], u->done[1]})
        if (e) (void)hipEventDestroy(e);
    if (u->copies) (void)hipStreamDestroy(u->copies);
    if (u->stream) (void)hipStreamDestroy(u->stream);
    delete u;
}

extern "C" size_t cfm_unet_param_count(void) { return param_count(); }

extern "C" cfm_status cfm_unet_create(int n, int batch, cfm_unet **out) {
    if (!out) return CFM_EINVAL;
    *out = nullptr;
    // batch * n^3 <= 2^27 keeps the elementwise kernels' and the weight gradients' offsets within 32 bits
    if (n < 4 || n % 4 != 0 || batch < 1 || (long long)batch * n * n * n > (1LL << 27)) return CFM_EINVAL;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return CFM_EDEVICE;
    auto *u = new (std::nothrow) cfm_unet();
    if (!u) return CFM_ENOMEM;
    auto fail = [&](cfm_status s) {
        cfm_unet_destroy(u);
        return s;
    };
    u->n = n;
    u->batch = batch;
    for (int l = 0; l < 3; ++l) {
        const size_t m = (size_t)(n >> l);
        u->P[l] = (size_t)batch * m * m * m;
    }
    if (hipStreamCreate(&u->stream) != hipSuccess || hipStreamCreate(&u->copies) != hipSuccess) return fail(CFM_EDEVICE);
    for (hipEvent_t *e : {&u->copied, &u->done[0], &u->done[1]})
        if (hipEventCreateWithFlags(e, hipEventDisableTiming) != hipSuccess) return fail(CFM_EDEVICE);
    u->nparam = param_count();
    size_t off = 0;
    for (int i = 0; i < kNConv; ++i) {
        u->woff[i] = off;
        off += (size_t)kConv[i].cout * kConv[i].cin_real * 27;
        u->boff[i] = off;
        off += kConv[i].cout;
        u->Kp[i] = pad32(27 * kConv[i].cin);
        u->Kpt[i] = pad32(27 * kConv[i].cout);
    }
    u->head_off = off;
    cfm_status st = CFM_OK;
    auto A = [&](auto **p, size_t bytes) {
        if (st == CFM_OK) st = unet_alloc(u, (void **)p, bytes);
    };
    A(&u->master, 4 * u->nparam);
    A(&u->grad, 4 * u->nparam);
    A(&u->adam_m, 4 * u->nparam);
    A(&u->adam_v, 4 * u->nparam);
    size_t max_wk = 0, max_partial = 0;
    for (int i = 0; i < kNConv; ++i) {
        A(&u->Wf[i], 2 * (size_t)kConv[i].cout * u->Kp[i]);
        if (i > 0) A(&u->Wt[i], 2 * (size_t)kConv[i].cin * u->Kpt[i]);
        max_wk = std::max(max_wk, (size_t)kConv[i].cout * (u->Kp[i] + 1));
        int nslab;
        wgrad_shape(n >> kConv[i].level, batch, kConv[i].cin, &nslab);
        max_partial = std::max(max_partial, (size_t)nslab * kConv[i].cout * (u->Kp[i] + 1));
    }
    A(&u->rtmp, 8 * kReduceParts * max_wk);
    A(&u->partial, 4 * max_partial);
    const size_t P1 = u->P[0], P2 = u->P[1], P3 = u->P[2];
    A(&u->X0, 2 * P1 * 8);
    A(&u->A0, 2 * P1 * 16);
    A(&u->S1, 2 * P1 * 16);
    A(&u->Q1, 2 * P2 * 16);
    A(&u->A2, 2 * P2 * 32);
    A(&u->S2, 2 * P2 * 32);
    A(&u->Q2, 2 * P3 * 32);
    A(&u->A4, 2 * P3 * 64);
    A(&u->A5, 2 * P3 * 64);
    A(&u->A6, 2 * P2 * 32);
    A(&u->A7, 2 * P2 * 32);
    A(&u->A8, 2 * P1 * 16);
    A(&u->A9, 2 * P1 * 16);
    A(&u->pred, 4 * P1);
    A(&u->target, 4 * P1);
    A(&u->dpred, 4 * P1);
    A(&u->in_f, 4 * P1 * 2);
    A(&u->lpart, 8 * ((P1 + 255) / 256));
    A(&u->hpart, 4 * 17 * ((P1 + 255) / 256));
    for (bf16 **g : {&u->g1a, &u->g1b, &u->g1c}) A(g, 2 * P1 * 48);
    for (bf16 **g : {&u->g2a, &u->g2b, &u->g2c}) A(g, 2 * P2 * 96);
    for (bf16 **g : {&u->g3a, &u->g3b}) A(g, 2 * P3 * 64);
    if (st != CFM_OK) return fail(st);
    for (int i = 0; i < kNConv; ++i)  // the packed weights' padding stays zero
        if (hipMemset(u->Wf[i], 0, 2 * (size_t)kConv[i].cout * u->Kp[i]) != hipSuccess ||
            (i > 0 && hipMemset(u->Wt[i], 0, 2 * (size_t)kConv[i].cin * u->Kpt[i]) != hipSuccess))
            return fail(CFM_EDEVICE);
    if (hipMemset(u->master, 0, 4 * u->nparam) != hipSuccess || hipMemset(u->adam_m, 0, 4 * u->nparam) != hipSuccess ||
        hipMemset(u->adam_v, 0, 4 * u->nparam) != hipSuccess)
        return fail(CFM_EDEVICE);
    *out = u;
    return CFM_OK;
}

static cfm_status pack_all_weights(cfm_unet *u) {
    PackTable T;
    int most = 0;
    for (int i = 0; i < kNConv; ++i) {
        const ConvSpec &s = kConv[i];
        T.layer[i] = {u->master + u->woff[i], u->Wf[i], u->Wt[i], s.cout, s.cin_real, s.cin, u->Kp[i], u->Kpt[i]};
        most = std::max(most, s.cout * s.cin * 27);
    }
    hipLaunchKernelGGL(pack_weights_kernel, dim3((unsigned)((most + 255) / 256), kNConv), dim3(256), 0, u->stream, T);
    CFM_HIP(hipGetLastError());
    return CFM_OK;
}

extern "C" cfm_status cfm_unet_set_params(cfm_unet *u, const float *params) {
    if (!u || !params) return CFM_EINVAL;
    CFM_HIP(hipMemcpy(u->master, params, 4 * u->nparam, hipMemcpyHostToDevice));
    CFM_HIP(hipMemset(u->adam_m, 0, 4 * u->nparam));
    CFM_HIP(hipMemset(u->adam_v, 0, 4 * u->nparam));
    u->step = 0;
    cfm_status st = pack_all_weights(u);
    if (st != CFM_OK) return st;
    CFM_HIP(hipStreamSynchronize(u->stream));
    return CFM_OK;
}

extern "C" cfm_status cfm_unet_get_params(cfm_unet *u, float *params) {
    if (!u || !params) return CFM_EINVAL;
    CFM_HIP(hipMemcpy(params, u->master, 4 * u->nparam, hipMemcpyDeviceToHost));
    return CFM_OK;
}

template <int MT, int CIN>
static bool launch_conv_lds(int n, int batch, hipStream_t st, const bf16 *X, const bf16 *Xup, const bf16 *W, int kp,
                            const float *bias, bf16 *Y, int relu, const bf16 *mask) {
    if (kp != (27 * CIN + 31) / 32 * 32) return false;
    // tile 16 x TY x TZ points, the staged block at most 80 KiB of LDS (two workgroups per CU): up
    // to 48 input channels 16 x 8 x 2 (four rows per wavefront), 64 channels 16 x 4 x 2, 96
    // channels 16 x 4 x 1
    constexpr int TY = CIN <= 48 ? 8 : 4;
    constexpr int TZ = CIN <= 64 ? 2 : 1;
    static_assert((TZ + 2) * (TY + 2) * 18 * CIN * 2 <= 80 * 1024, "staged block above 80 KiB");
    const int nbx = (n + 15) / 16, nby = (n + TY - 1) / TY, nbz = (n + TZ - 1) / TZ;
    const dim3 grid((unsigned)(nbx * nby * nbz * batch));
    hipLaunchKernelGGL((conv3_fwd_lds_kernel<MT, CIN, TY, TZ>), grid, dim3(256), 0, st, X, Xup, W, kp, bias, Y, n, nbx, nby,
                       nbz, relu, mask);
    return true;
}

#ifndef CFM_UNET_XACC
#define CFM_UNET_XACC 1
#endif

// Rows of NXT 16-point tiles: eight (y, z) rows (4 x 2), two per wavefront, while the
// accumulators (3 MT x 2 x NXT tiles) stay within 24 tiles, else 2 x 2 rows, one per
// wavefront; eight wavefronts (one row each) when the eight-row block is too large for two
// workgroups per CU.
template <int MT, int CIN, int NXT>
static void launch_conv_xacc(int n, int batch, hipStream_t st, const bf16 *X, const bf16 *Xup, const bf16 *W, int kp,
                             const float *bias, bf16 *Y, int relu, const bf16 *mask) {
    constexpr bool two = MT * NXT <= 4;
    constexpr int lds8 = NXT * 16 * 6 * 4 * CIN * 2;
    constexpr int NW = two && lds8 > 80 * 1024 ? 8 : 4;
    constexpr int TY = two ? 4 : 2, TZ = 2;
    static_assert(NXT * 16 * (TY + 2) * (TZ + 2) * CIN * 2 <= 144 * 1024, "staged block above 144 KiB");
    const int nby = (n + TY - 1) / TY, nbz = (n + TZ - 1) / TZ;
    hipLaunchKernelGGL((conv3_fwd_xacc_kernel<MT, CIN, TY, TZ, NXT, NW, 2>), dim3((unsigned)(nby * nbz * batch)),
                       dim3(64 * NW), 0, st, X, Xup, W, kp, bias, Y, n, nby, nbz, relu, mask);
}

// The x-accumulator kernel where it measured faster than the per-tap one: the wide inputs of
// the decoder, 48 -> 16 channels (rows of 64 points at 32 x 64^3: 1.06 vs 1.17 ms) and 96 -> 32
// (rows of 32: 0.59 vs 0.93 ms).  With 8 to 32 input channels the per-tap kernel's smaller
// staged block keeps 3 to 7 workgroups per CU against 1 to 3 and won (16 -> 16: 0.33 vs 0.41
// ms), and the 16 -> 48 and 32 -> 96 data gradients need 3 x 3 and 3 x 6 accumulator tiles per
// row: one wavefront per SIMD, twice the time.
static bool conv_xacc(int cin, int mt, int n, int batch, hipStream_t st, const bf16 *X, const bf16 *Xup, const bf16 *W, int kp,
                      const float *bias, bf16 *Y, int relu, const bf16 *mask) {
    if (!CFM_UNET_XACC || n > 64 || kp < 27 * cin) return false;
    const int nxt = n <= 16 ? 1 : n <= 32 ? 2 : 4;
#define CFM_CONV_XACC(C, M, T)                                               \
    if (cin == C && mt == M && nxt == T) {                                   \
        launch_conv_xacc<M, C, T>(n, batch, st, X, Xup, W, kp, bias, Y, relu, mask); \
        return true;                                                         \
    }
    CFM_CONV_XACC(48, 1, 4)
    CFM_CONV_XACC(48, 1, 2)
    CFM_CONV_XACC(48, 1, 1)
    CFM_CONV_XACC(96, 2, 2)
    CFM_CONV_XACC(96, 2, 1)
#undef CFM_CONV_XACC
    return false;
}

// the (input channels, output channel tiles) pairs of the network's forward and data-gradient convs
static bool conv_lds(int cin, int mt, int n, int batch, hipStream_t st, const bf16 *X, const bf16 *Xup, const bf16 *W, int kp,
                     const float *bias, bf16 *Y, int relu, const bf16 *mask) {
#define CFM_CONV_LDS(C, M)                                                  \
    if (cin == C && mt == M) {                                              \
        return launch_conv_lds<M, C>(n, batch, st, X, Xup, W, kp, bias, Y, relu, mask); \
    }
    CFM_CONV_LDS(8, 1)
    CFM_CONV_LDS(16, 1)
    CFM_CONV_LDS(16, 2)
    CFM_CONV_LDS(16, 3)
    CFM_CONV_LDS(32, 1)
    CFM_CONV_LDS(32, 2)
    CFM_CONV_LDS(32, 4)
    CFM_CONV_LDS(32, 6)
    CFM_CONV_LDS(48, 1)
    CFM_CONV_LDS(64, 2)
    CFM_CONV_LDS(64, 4)
    CFM_CONV_LDS(96, 2)
#undef CFM_CONV_LDS
    return false;
}

// Y = conv(X) for the (input channels, output channels) pairs of the network
// mask (may be null): the data gradient of a ReLU layer, zero where mask (the layer's forward
// output, [points][cout]) is not positive
static cfm_status conv_fwd(cfm_unet *u, const bf16 *X, const bf16 *Xup, int cin, const bf16 *W, int kp, const float *bias, bf16 *Y,
                           int cout, int level, int relu, int nb, const bf16 *mask = nullptr) {
    const int n = u->n >> level;
    if (cout % 16 != 0 || !(conv_xacc(cin, cout / 16, n, nb, u->stream, X, Xup, W, kp, bias, Y, relu, mask) ||
                            conv_lds(cin, cout / 16, n, nb, u->stream, X, Xup, W, kp, bias, Y, relu, mask)))
        return CFM_FAIL(CFM_EINVAL, "unet: no convolution kernel for %d -> %d channels", cin, cout);
    CFM_HIP(hipGetLastError());
    return CFM_OK;
}

// The forward pass of batch elements [b0, b0 + nb); d_in: the whole batch's input.
static cfm_status run_forward_dev(cfm_unet *u, const float *d_in, int b0, int nb) {
    const int n = u->n, n3 = n * n * n;
    const size_t o1 = u->P[0] / u->batch * b0, o2 = u->P[1] / u->batch * b0, o3 = u->P[2] / u->batch * b0;
    const size_t P1 = u->P[0] / u->batch * nb, P2 = u->P[1] / u->batch * nb, P3 = u->P[2] / u->batch * nb;
    bf16 *X0 = u->X0 + o1 * 8, *A0 = u->A0 + o1 * 16, *S1 = u->S1 + o1 * 16, *Q1 = u->Q1 + o2 * 16, *A2 = u->A2 + o2 * 32,
         *S2 = u->S2 + o2 * 32, *Q2 = u->Q2 + o3 * 32, *A4 = u->A4 + o3 * 64, *A5 = u->A5 + o3 * 64, *A6 = u->A6 + o2 * 32,
         *A7 = u->A7 + o2 * 32, *A8 = u->A8 + o1 * 16, *A9 = u->A9 + o1 * 16;
    hipLaunchKernelGGL(pack_input_kernel, blocks_for(P1), dim3(256), 0, u->stream, d_in + 2 * o1, X0, n3, nb);
    CFM_HIP(hipGetLastError());
    const float *b[kNConv];
    for (int i = 0; i < kNConv; ++i) b[i] = u->master + u->boff[i];
    cfm_status st;
#define CONV(I, X, Y) CONV2(I, X, nullptr, Y)
#define CONV2(I, X, XUP, Y) \
    if ((st = conv_fwd(u, X, XUP, kConv[I].cin, u->Wf[I], u->Kp[I], b[I], Y, kConv[I].cout, kConv[I].level, 1, nb)) != CFM_OK) return st
    CONV(0, X0, A0);
    CONV(1, A0, S1);
    hipLaunchKernelGGL(pool_fwd_kernel, blocks_for(P2 * 16 / 8), dim3(256), 0, u->stream, S1, Q1, 16, n, nb);
    CONV(2, Q1, A2);
    CONV(3, A2, S2);
    hipLaunchKernelGGL(pool_fwd_kernel, blocks_for(P3 * 32 / 8), dim3(256), 0, u->stream, S2, Q2, 32, n / 2, nb);
    CONV(4, Q2, A4);
    CONV(5, A4, A5);
    CONV2(6, S2, A5, A6);
    CONV(7, A6, A7);
    CONV2(8, S1, A7, A8);
    CONV(9, A8, A9);
#undef CONV
#undef CONV2
    hipLaunchKernelGGL(head_fwd_kernel, blocks_for(P1), dim3(256), 0, u->stream, A9, u->master + u->head_off,
                       u->pred + o1, P1);
    CFM_HIP(hipGetLastError());
    return CFM_OK;
}

// Parts of the batch that the forward pass is launched in.  In two, the first part's kernels run while
// the host copies the second part in (and, for an output, the second part's while the first is
// copied out): 8 x 64^3 1.61 ms against 1.96 in one.  Parts of fewer points than these would leave the
// deep levels' kernels few workgroups, for a copy that is over sooner than they are (2 x 64^3 648 us in
// two parts, 619 before; 12 x 36^3 799 and 781).
static int forward_parts(const cfm_unet *u) { return u->batch >= 2 && u->P[0] >= ((size_t)1 << 20) ? 2 : 1; }

// Copies the input in and enqueues the forward pass; with several parts, done[p] is recorded after part p.
static cfm_status run_forward(cfm_unet *u, const float *input_host) {
    const int parts = forward_parts(u);
    const size_t each = 2 * (u->P[0] / u->batch);
    if (parts == 1) {  // (nothing to run beside: a second stream would only add its waits, 17 us of a small pass's 233)
        CFM_HIP(hipMemcpyAsync(u->in_f, input_host, 4 * each * u->batch, hipMemcpyHostToDevice, u->stream));
        return run_forward_dev(u, u->in_f, 0, u->batch);
    }
    for (int p = 0; p < parts; ++p) {
        const int b0 = u->batch * p / parts, nb = u->batch * (p + 1) / parts - b0;
        CFM_HIP(hipMemcpyAsync(u->in_f + each * b0, input_host + each * b0, 4 * each * nb, hipMemcpyHostToDevice, u->copies));
        CFM_HIP(hipEventRecord(u->copied, u->copies));
        CFM_HIP(hipStreamWaitEvent(u->stream, u->copied, 0));
        const cfm_status st = run_forward_dev(u, u->in_f, b0, nb);
        if (st != CFM_OK) return st;
        CFM_HIP(hipEventRecord(u->done[p], u->stream));
    }
    return CFM_OK;
}

namespace cfm {
UnetView unet_view(cfm_unet *u) { return UnetView{u->n, u->batch, u->stream, u->in_f}; }
cfm_status unet_forward_device(cfm_unet *u, const float *d_in, const float **d_pred) {
    cfm_status st = run_forward_dev(u, d_in, 0, u->batch);
    if (st == CFM_OK && d_pred) *d_pred = u->pred;
    return st;
}
}  // namespace cfm

extern "C" cfm_status cfm_unet_forward(cfm_unet *u, const float *input, float *output) {
    if (!u || !input || !output) return CFM_EINVAL;
    cfm_status st = run_forward(u, input);
    if (st != CFM_OK) return st;
    const int parts = forward_parts(u);
    const size_t each = u->P[0] / u->batch;
    if (parts == 1) {
        CFM_HIP(hipMemcpyAsync(output, u->pred, 4 * u->P[0], hipMemcpyDeviceToHost, u->stream));
        CFM_HIP(hipStreamSynchronize(u->stream));
        return CFM_OK;
    }
    for (int p = 0; p < parts; ++p) {
        const int b0 = u->batch * p / parts, nb = u->batch * (p + 1) / parts - b0;
        CFM_HIP(hipStreamWaitEvent(u->copies, u->done[p], 0));
        CFM_HIP(hipMemcpyAsync(output + each * b0, u->pred + each * b0, 4 * each * nb, hipMemcpyDeviceToHost, u->copies));
    }
    CFM_HIP(hipStreamSynchronize(u->copies));
    CFM_HIP(hipStreamSynchronize(u->stream));
    return CFM_OK;
}

template <int CIN, int COUT>
static void launch_wgrad_rows(int nslab, hipStream_t st, const bf16 *X, const bf16 *Xup, const bf16 *dZ, int kp, float *partial,
                              const WgradShape &S) {
    const size_t lds = sizeof(bf16) * ((size_t)COUT * 72 + (size_t)3 * (S.rows + 2) * kWgradRows16) + sizeof(double) * COUT;
    // (short rows, eight to a block, take more than 64 KiB)
    static const bool big_lds_ok = hipFuncSetAttribute((const void *)conv3_wgrad_rows_kernel<CIN, COUT>,
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024) == hipSuccess;
    (void)big_lds_ok;
    hipLaunchKernelGGL((conv3_wgrad_rows_kernel<CIN, COUT>), dim3(nslab, (CIN + 15) / 16), dim3(192), lds, st, X, Xup,
                       dZ, kp, partial, S);
}

static bool wgrad_rows(int cin, int cout, int nslab, hipStream_t st, const bf16 *X, const bf16 *Xup, const bf16 *dZ, int kp,
                       float *partial, const WgradShape &S) {
#define CFM_WGRAD_ROWS(C, O)                                             \
    if (cin == C && cout == O) {                                         \
        launch_wgrad_rows<C, O>(nslab, st, X, Xup, dZ, kp, partial, S);  \
        return true;                                                     \
    }
    CFM_WGRAD_ROWS(8, 16)
    CFM_WGRAD_ROWS(16, 16)
    CFM_WGRAD_ROWS(16, 32)
    CFM_WGRAD_ROWS(32, 32)
    CFM_WGRAD_ROWS(48, 16)
    CFM_WGRAD_ROWS(32, 64)
    CFM_WGRAD_ROWS(64, 64)
    CFM_WGRAD_ROWS(96, 32)
#undef CFM_WGRAD_ROWS
    return false;
}

// gradients of conv I's weights and biases from its input X and output gradient dZ
static cfm_status conv_wgrad(cfm_unet *u, int I, const bf16 *X, const bf16 *dZ, const bf16 *Xup = nullptr) {
    const ConvSpec &s = kConv[I];
    const int Kp = u->Kp[I], count = s.cout * (Kp + 1);
    int nslab;
    const WgradShape S = wgrad_shape(u->n >> s.level, u->batch, s.cin, &nslab);
    if (!wgrad_rows(s.cin, s.cout, nslab, u->stream, X, Xup, dZ, Kp, u->partial, S))
        return CFM_FAIL(CFM_EINVAL, "unet: no weight-gradient kernel for %d -> %d channels", s.cin, s.cout);
    CFM_HIP(hipGetLastError());
    if (nslab >= 4 * kReduceParts) {
        const dim3 grid((unsigned)((count + 255) / 256), kReduceParts);
        hipLaunchKernelGGL(reduce_slab_parts_kernel, grid, dim3(256), 0, u->stream, u->partial, nslab, (size_t)count,
                           kReduceParts, u->rtmp);
        hipLaunchKernelGGL(reduce_slabs_kernel<double>, blocks_for(count), dim3(256), 0, u->stream, u->rtmp, kReduceParts,
                           s.cout, s.cin_real, s.cin, Kp, u->grad + u->woff[I], u->grad + u->boff[I]);
    } else {
        hipLaunchKernelGGL(reduce_slabs_kernel<float>, blocks_for(count), dim3(256), 0, u->stream, u->partial, nslab,
                           s.cout, s.cin_real, s.cin, Kp, u->grad + u->woff[I], u->grad + u->boff[I]);
    }
    CFM_HIP(hipGetLastError());
    return CFM_OK;
}

// dX = conv_transpose(dZ) for conv I (output channels = cin of the layer); with mask (the
// forward output of the ReLU layer feeding conv I), the gradient before that ReLU
static cfm_status conv_dgrad(cfm_unet *u, int I, const bf16 *dZ, bf16 *dX, const bf16 *mask = nullptr) {
    const ConvSpec &s = kConv[I];
    return conv_fwd(u, dZ, nullptr, s.cout, u->Wt[I], u->Kpt[I], nullptr, dX, s.cin, s.level, 0, u->batch, mask);
}

static cfm_status run_backward(cfm_unet *u, const float *target_host, double *loss) {
    const size_t P1 = u->P[0], P2 = u->P[1], P3 = u->P[2];
    const int n = u->n;
    if (forward_parts(u) > 1) {  // beside the forward pass, which still runs
        CFM_HIP(hipMemcpyAsync(u->target, target_host, 4 * P1, hipMemcpyHostToDevice, u->copies));
        CFM_HIP(hipEventRecord(u->copied, u->copies));
        CFM_HIP(hipStreamWaitEvent(u->stream, u->copied, 0));
    } else {
        CFM_HIP(hipMemcpyAsync(u->target, target_host, 4 * P1, hipMemcpyHostToDevice, u->stream));
    }
    const unsigned nb1 = (unsigned)((P1 + 255) / 256);
    hipLaunchKernelGGL(mse_kernel, dim3(nb1), dim3(256), 0, u->stream, u->pred, u->target, u->dpred, u->lpart, P1);
    const float *hw = u->master + u->head_off;
    // dZ9: the head's data gradient through the last ReLU
    hipLaunchKernelGGL(head_bwd_kernel, dim3(nb1), dim3(256), 0, u->stream, u->A9, hw, u->dpred, u->g1b, u->hpart, P1);
    CFM_HIP(hipGetLastError());
    // head gradient: reduce per-block partials (fixed order)
    hipLaunchKernelGGL(reduce_rows_kernel, dim3(17), dim3(1024), 0, u->stream, u->hpart, (int)nb1,
                       u->grad + u->head_off);
    cfm_status st;
#define CK(x) \
    if ((st = (x)) != CFM_OK) return st
    // Every ReLU backward is folded into the kernel producing the gradient it masks (the data-
    // gradient convs, the upsampling and pooling gradients, the head), and the skip gradients are
    // read in place from the concatenated buffers' gradients (g1c, g2c), which stay untouched
    // until the encoder levels use them.
    // decoder level 1
    CK(conv_wgrad(u, 9, u->A8, u->g1b));
    CK(conv_dgrad(u, 9, u->g1b, u->g1a, u->A8));       // dZ8
    CK(conv_wgrad(u, 8, u->S1, u->g1a, u->A7));
    CK(conv_dgrad(u, 8, u->g1a, u->g1c));               // dU1 [P1][48]
    hipLaunchKernelGGL(up_bwd_kernel, blocks_for(P2 * 32 / 8), dim3(256), 0, u->stream, u->g1c, u->g2b, 32, 48, 0,
                       n / 2, u->batch, u->A7);          // dZ7
    // decoder level 2
    CK(conv_wgrad(u, 7, u->A6, u->g2b));
    CK(conv_dgrad(u, 7, u->g2b, u->g2a, u->A6));       // dZ6
    CK(conv_wgrad(u, 6, u->S2, u->g2a, u->A5));
    CK(conv_dgrad(u, 6, u->g2a, u->g2c));               // dU2 [P2][96]
    hipLaunchKernelGGL(up_bwd_kernel, blocks_for(P3 * 64 / 8), dim3(256), 0, u->stream, u->g2c, u->g3b, 64, 96, 0,
                       n / 4, u->batch, u->A5);          // dZ5
    // bottleneck
    CK(conv_wgrad(u, 5, u->A4, u->g3b));
    CK(conv_dgrad(u, 5, u->g3b, u->g3a, u->A4));       // dZ4
    CK(conv_wgrad(u, 4, u->Q2, u->g3a));
    CK(conv_dgrad(u, 4, u->g3a, u->g3b));               // dQ2 [P3][32]
    hipLaunchKernelGGL(pool_bwd_kernel, blocks_for(P2 * 32 / 8), dim3(256), 0, u->stream, u->g3b, u->g2b, 32, n / 2,
                       u->batch, u->g2c, 96, 64, u->S2);  // dZ3 = relu'(S2) (pool' dQ2 + dS2 skip)
    // encoder level 2
    CK(conv_wgrad(u, 3, u->A2, u->g2b));
    CK(conv_dgrad(u, 3, u->g2b, u->g2a, u->A2));       // dZ2
    CK(conv_wgrad(u, 2, u->Q1, u->g2a));
    CK(conv_dgrad(u, 2, u->g2a, u->g2b));               // dQ1 [P2][16]
    hipLaunchKernelGGL(pool_bwd_kernel, blocks_for(P1 * 16 / 8), dim3(256), 0, u->stream, u->g2b, u->g1a, 16, n,
                       u->batch, u->g1c, 48, 32, u->S1);  // dZ1 = relu'(S1) (pool' dQ1 + dS1 skip)
    // encoder level 1
    CK(conv_wgrad(u, 1, u->A0, u->g1a));
    CK(conv_dgrad(u, 1, u->g1a, u->g1b, u->A0));       // dZ0
    CK(conv_wgrad(u, 0, u->X0, u->g1b));
#undef CK
    CFM_HIP(hipGetLastError());
    if (loss) {
        std::vector<double> lp(nb1);
        CFM_HIP(hipMemcpyAsync(lp.data(), u->lpart, 8 * nb1, hipMemcpyDeviceToHost, u->stream));
        CFM_HIP(hipStreamSynchronize(u->stream));
        double s = 0.0;
        for (double v : lp) s += v;
        *loss = s / (double)P1;
    }
    return CFM_OK;
}

extern "C" cfm_status cfm_unet_gradient(cfm_unet *u, const float *input, const float *target, float *grad,
                                        double *loss) {
    if (!u || !input || !target) return CFM_EINVAL;
    cfm_status st = run_forward(u, input);
    if (st == CFM_OK) st = run_backward(u, target, loss);
    if (st != CFM_OK) return st;
    if (grad) CFM_HIP(hipMemcpyAsync(grad, u->grad, 4 * u->nparam, hipMemcpyDeviceToHost, u->stream));
    CFM_HIP(hipStreamSynchronize(u->stream));
    return CFM_OK;
}

extern "C" cfm_status cfm_unet_train_step(cfm_unet *u, const float *input, const float *target, float lr,
                                          double *loss) {
    if (!u || !input || !target || !(lr > 0.f)) return CFM_EINVAL;
    cfm_status st = run_forward(u, input);
    if (st == CFM_OK) st = run_backward(u, target, loss);
    if (st != CFM_OK) return st;
    u->step += 1;
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.f - std::pow(b1, (float)u->step), c2 = 1.f - std::pow(b2, (float)u->step);
    hipLaunchKernelGGL(adam_kernel, blocks_for(u->nparam), dim3(256), 0, u->stream, u->master, u->grad, u->adam_m,
                       u->adam_v, u->nparam, lr, b1, b2, 1e-8f, c1, c2);
    CFM_HIP(hipGetLastError());
    st = pack_all_weights(u);
    if (st != CFM_OK) return st;
    CFM_HIP(hipStreamSynchronize(u->stream));
    return CFM_OK;
}

// He-uniform initialisation from a SplitMix64 stream: w ~ U(-a, a),
// a = sqrt(6 / fan_in); biases 0; head weights scaled by 0.1.
extern "C" cfm_status cfm_unet_init_params(uint64_t seed, float *params) {
    if (!params) return CFM_EINVAL;
    uint64_t s = seed ^ 0xA0761D6478BD642FULL;
    auto uni = [&]() {
        s += 0x9E3779B97F4A7C15ULL;
        uint64_t z = s;
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
        z ^= z >> 31;
        return (double)(z >> 11) * 0x1.0p-53;
    };
    size_t off = 0;
    for (const auto &c : kConv) {
        const double a = std::sqrt(6.0 / (27.0 * c.cin_real));
        const size_t nw = (size_t)c.cout * c.cin_real * 27;
        for (size_t i = 0; i < nw; ++i) params[off + i] = (float)((2.0 * uni() - 1.0) * a);
        off += nw;
        for (int i = 0; i < c.cout; ++i) params[off + i] = 0.f;
        off += c.cout;
    }
    const double a = 0.1 * std::sqrt(6.0 / kHeadIn);
    for (int i = 0; i < kHeadIn; ++i) params[off + i] = (float)((2.0 * uni() - 1.0) * a);
    params[off + kHeadIn] = 0.f;
    return CFM_OK;
}
