// Position derivatives from slopes kept by the forward.
//
// Inside its simplex every feature of a level is an affine function of the position, and the D numbers of its slope are all
// that the gradient w.r.t. the positions and the gradient of that gradient w.r.t. the upstream gradient need of the table:
//
//     positions_grad[n][k]   = sum over levels and features of  grad[level][f][n] * window[level] * slope[level][f][k][n]
//     grad_grad[level][f][n] = window[level] * sum over k of  double_positions_grad[n][k] * slope[level][f][k][n]
//
// The forward holds a point's vertices in registers and can leave the slopes behind (forward_kernel<..., true>): 4 D F bytes per point
// and level, written and read as a stream, where each of the two kernels above would locate the simplex and gather its D+1
// vertices again (8 to 32 bytes each, but of a line of 128 when the L2 misses).
//
// Measured (us; forward, position gradient of rows that leaves its level-major copy, grad-grad as rows, then the three together;
// gathering -> slopes).  The gathering kernels are bound by L2 requests or, with large slices, by the lines they miss; the two below run at
// 4.5 to 5.8 TB/s.  What the forward adds is less than its writes would take alone, because they pass while it waits for gathers.
//   D = 3, 24 levels of 2^18 slots, 2^20 points    285 -> 329   450 -> 191   386 -> 147   1120 -> 667
//   D = 4, the same                                411 -> 445   544 -> 230   478 -> 185   1432 -> 860
//   D = 8, 16 levels of 2^19 slots, 2^19 points    308 -> 348   465 -> 134   354 -> 120   1127 -> 602
//   D = 3, 16 live levels of 2^22 slots, 2^20      255 -> 295   353 -> 151   348 -> 112    955 -> 558
//   the same, 200001 points                         57 -> 67     81 -> 26     80 -> 21     218 -> 114
//   D = 3, 24 levels of 2^18 slots, 2^15 points   13.4 -> 15   24.5 -> 7.7  19.8 -> 7.7  57.7 -> 30.4
// Many features make the slopes as large as the vertices (D = 3, F = 8, 16 levels of 2^18 slots, 2^19 points: 96 bytes against four gathers
// of 32, 231 -> 353   366 -> 255   344 -> 202   941 -> 809); slopes_serve says where they are kept.  A position gradient that is not
// differentiated again gains less (kernels: D = 3, F = 2: 735 -> 520; F = 4: 672 -> 575; D = 4, F = 8: 415 -> 409; D = 3, F = 8: 597 -> 607, through
// the module 513 -> 505) or loses, where the gathers hit the first-level cache (D = 6, 24 levels of 2^11 slots, 2^19 points 287 -> 340, the pass of
// an SDF 1047 -> 978; 16 levels of 2^12 242 -> 250 and 889 -> 767).
// Error against 64 bits (2-norm, D = 2 to 8): position gradient 7.3e-8 - 9.9e-8 -> 5.9e-8 - 7.3e-8, grad-grad 6.5e-8 - 9.4e-8 -> 5.4e-8 - 7.1e-8.
//
// slopes[level][tile of 64 points][f * D + k][64]: what a wave of the forward writes for a level, and a wave here reads, is one contiguous
// piece.  A level whose window weight is 0 is neither written nor read.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "penc_lattice.hpp"

namespace penc {

constexpr int kSlopeTile = 64;

__host__ __device__ __forceinline__ size_t slope_tiles(int64_t n_points) { return static_cast<size_t>((n_points + kSlopeTile - 1) / kSlopeTile); }

// Where the slopes of point n at a level begin; those of the next (feature, coordinate) are kSlopeTile floats on.
template <int D, int F>
__device__ __forceinline__ size_t slope_offset(int n_points, int level, int n) {
    return ((static_cast<size_t>(level) * slope_tiles(n_points) + static_cast<uint32_t>(n) / kSlopeTile) * (D * F)) * kSlopeTile +
           static_cast<uint32_t>(n) % kSlopeTile;
}

// The slopes of a simplex from the values at its vertices.  A weight's derivative w.r.t. the elevated coordinate of rank m is
// 1/(D+1) at vertex D-m and -1/(D+1) at vertex D+1-m (vertex 0 for m = 0), so the derivative w.r.t. that coordinate is the
// difference of two vertices; `column` is the thread's LDS column (see sort_by_rank_lds), which brings the differences from rank order
// into the order of the coordinates, two features at a time.  The elevation then gives, for position k,
//     slope[k] = sf[k] * (sum over i <= k of dE[i] - (k+1) dE[k+1]).
template <int D, int F>
__device__ __forceinline__ void store_slopes(const fvec<D + 1> (&v)[F], ivec<D + 1> rank, uint2* column, uint32_t stride,
                                             const float* __restrict__ sf, float* __restrict__ out) {
    constexpr int D1 = D + 1;
    constexpr float kInv = 1.0f / D1, kInvRest = static_cast<float>(1.0 / D1 - static_cast<double>(kInv));
    static_for<F / 2>(PENC_BODY(p) {
        PENC_INDEX(p);
        static_for<D1>(PENC_BODY(m) {
            PENC_INDEX(m);
            constexpr int from = D - m, minus = m == 0 ? 0 : D1 - m;
            uint2 cell;
            cell.x = __builtin_bit_cast(uint32_t, v[2 * p][from] - v[2 * p][minus]);
            cell.y = __builtin_bit_cast(uint32_t, v[2 * p + 1][from] - v[2 * p + 1][minus]);
            column[m * stride] = cell;
        });
        fvec<D1> a, b;
        static_for<D1>(PENC_BODY(i) {
            PENC_INDEX(i);
            const int row = rank[i] < 0 ? 0 : (rank[i] > D ? D : rank[i]);  // (as in sort_by_rank_lds)
            const uint2 cell = column[static_cast<uint32_t>(row) * stride];
            a[i] = __builtin_bit_cast(float, cell.x);
            b[i] = __builtin_bit_cast(float, cell.y);
        });
        float sum_a = 0.0f, sum_b = 0.0f;
        static_for<D>(PENC_BODY(k) {
            PENC_INDEX(k);
            sum_a += a[k];
            sum_b += b[k];
            // sf / (D+1) in two parts: rounded to one, it would put the same relative error on every slope of the level
            const float scale = sf[k] * kInv, rest = __builtin_fmaf(sf[k], kInv, -scale) + sf[k] * kInvRest;
            const float da = __builtin_fmaf(-static_cast<float>(k + 1), a[k + 1], sum_a), db = __builtin_fmaf(-static_cast<float>(k + 1), b[k + 1], sum_b);
            // (non-temporal: the table slices the other waves gather from should stay in the L2)
            __builtin_nontemporal_store(__builtin_fmaf(da, scale, da * rest), out + (2 * p * D + k) * kSlopeTile);
            __builtin_nontemporal_store(__builtin_fmaf(db, scale, db * rest), out + ((2 * p + 1) * D + k) * kSlopeTile);
        });
    });
}

// A workgroup takes 64 points: lane = point, wave w takes levels w, w + kSlopeWaves, ...
constexpr int kSlopeWaves = 8, kSlopeBlock = kSlopeWaves * kSlopeTile;

// Gradient w.r.t. the positions.  The upstream gradient is [level][feature][n], or (kRows) rows of `grad_row_stride` floats, of
// which the [level][feature][n] copy is left in grad_level_major when the caller wants it: for what reads it a level at a time.
template <int D, int F, bool kRows>
__global__ void __launch_bounds__(kSlopeBlock)
positions_from_slopes_kernel(int n_points, int n_levels, const float* __restrict__ slopes, const float* __restrict__ window,
                             const float* __restrict__ grad, int64_t grad_row_stride, float* __restrict__ grad_level_major,
                             float* __restrict__ out) {
    extern __shared__ float tile[];  // rows: 64 x (columns | 1)
    __shared__ float partial[kSlopeWaves][kSlopeTile * D];
    const int base = blockIdx.x * kSlopeTile, count = n_points - base < kSlopeTile ? n_points - base : kSlopeTile;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int columns = n_levels * F, pitch = columns | 1;
    const int row = lane < count ? lane : count - 1, n = base + row;
    if constexpr (kRows) {
        // pairs of columns (rows are 8-byte aligned), the loads of four of them in flight together
        constexpr int kTogether = 4;
        const float* const rows = grad + static_cast<int64_t>(base) * grad_row_stride;
        const int pairs = columns / 2, n_pairs = count * pairs;
        int r = threadIdx.x / pairs, c = threadIdx.x % pairs;
        const int dr = kSlopeBlock / pairs, dc = kSlopeBlock % pairs;
        for (int i = threadIdx.x; i < n_pairs; i += kTogether * kSlopeBlock) {
            float2 v[kTogether];
            int at[kTogether];
#pragma unroll
            for (int u = 0; u < kTogether; ++u) {
                const bool in = i + u * kSlopeBlock < n_pairs;
                at[u] = in ? r * pitch + 2 * c : -1;
                v[u] = *reinterpret_cast<const float2*>(rows + (in ? r * grad_row_stride + 2 * c : 0));
                r += dr;
                c += dc;
                if (c >= pairs) {
                    c -= pairs;
                    ++r;
                }
            }
#pragma unroll
            for (int u = 0; u < kTogether; ++u)
                if (at[u] >= 0) {
                    tile[at[u]] = v[u].x;
                    tile[at[u] + 1] = v[u].y;
                }
        }
        __syncthreads();
        if (grad_level_major != nullptr && lane < count)
            for (int c = wave; c < columns; c += kSlopeWaves) grad_level_major[static_cast<size_t>(c) * n_points + n] = tile[lane * pitch + c];
    }
    fvec<D> total = 0.0f;
    for (int level = wave; level < n_levels; level += kSlopeWaves) {
        const float w_level = window[level];
        if (w_level == 0.0f) continue;
        const float* const s = slopes + slope_offset<D, F>(n_points, level, n);
        static_for<F>(PENC_BODY(f) {
            PENC_INDEX(f);
            float g;
            if constexpr (kRows) g = tile[row * pitch + level * F + f];
            else g = grad[(static_cast<size_t>(level) * F + f) * n_points + n];
            g *= w_level;
            static_for<D>(PENC_BODY(k) {
                PENC_INDEX(k);
                total[k] = __builtin_fmaf(g, s[(f * D + k) * kSlopeTile], total[k]);
            });
        });
    }
    static_for<D>(PENC_BODY(k) {
        PENC_INDEX(k);
        partial[wave][lane * D + k] = total[k];
    });
    __syncthreads();
    for (int i = threadIdx.x; i < count * D; i += kSlopeBlock) {
        // in double: the waves' sums are of one magnitude, and a value in eight roundings would lose what the slopes gain
        double acc = partial[0][i];
#pragma unroll
        for (int w = 1; w < kSlopeWaves; ++w) acc += partial[w][i];
        out[static_cast<size_t>(base) * D + i] = static_cast<float>(acc);
    }
}

// Gradient w.r.t. the upstream gradient: as [level][feature][n], or (kRows) as rows of `row_stride` floats.  Zeros in the extra levels.
template <int D, int F, bool kRows>
__global__ void __launch_bounds__(kSlopeBlock)
grad_grad_from_slopes_kernel(int n_points, int n_levels, int n_all_levels, const float* __restrict__ slopes, const float* __restrict__ window,
                             const float* __restrict__ double_pos_grad, float* __restrict__ out, int64_t row_stride) {
    extern __shared__ float tile[];  // rows: 64 x (columns | 1)
    // last points first: of what the position gradient has read before, the end is what the memory-side cache still holds (D = 4, 2^20
    // points: 189 -> 178 us; D = 3, 16 live levels: 111 -> 107)
    const int base = (gridDim.x - 1 - blockIdx.x) * kSlopeTile, count = n_points - base < kSlopeTile ? n_points - base : kSlopeTile;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int columns = n_all_levels * F, pitch = columns | 1;
    const int n = base + (lane < count ? lane : count - 1);
    fvec<D> q;
    static_for<D>(PENC_BODY(k) {
        PENC_INDEX(k); q[k] = double_pos_grad[static_cast<size_t>(n) * D + k]; });
    for (int level = wave; level < n_all_levels; level += kSlopeWaves) {
        const float w_level = level < n_levels ? window[level] : 0.0f;
        const bool live = w_level != 0.0f;
        const float* const s = slopes + slope_offset<D, F>(n_points, live ? level : 0, n);
        static_for<F>(PENC_BODY(f) {
            PENC_INDEX(f);
            float g = 0.0f;
            if (live) {
                static_for<D>(PENC_BODY(k) {
                    PENC_INDEX(k);
                    g = __builtin_fmaf(q[k], s[(f * D + k) * kSlopeTile], g);
                });
                g *= w_level;
            }
            if constexpr (kRows) tile[lane * pitch + level * F + f] = g;
            else if (lane < count) out[(static_cast<size_t>(level) * F + f) * n_points + n] = g;
        });
    }
    if constexpr (kRows) {
        __syncthreads();
        float* const to = out + static_cast<int64_t>(base) * row_stride;
        for (int r = wave; r < count; r += kSlopeWaves)
            for (int c = lane; c < columns; c += 64) to[r * row_stride + c] = tile[r * pitch + c];
    }
}

}  // namespace penc
