// HIP kernels (gfx950, wave64) and C-ABI entry points of the permutohedral-lattice hash encoding.
//
// Work decomposition
//   forward, grad-of-grad (the gathering half of the double backward) : a thread takes a point at one
//       level, or at two levels half the list apart.  Workgroups run row by row of levels, and where the
//       slices are small enough each die keeps its own share of the rows (LevelMap), so that the slices
//       being gathered from stay in its L2; the level's scale factors / shifts / window weight are
//       wave-uniform (scalar loads).
//   position backward : a thread sums a group of two of the levels the window leaves in registers; the
//       per-group partial sums are reduced in a fixed order, without atomics (the reference needs D
//       atomics per point-level because it gives each level its own block,
//       kernels/permutohedral_encoding/EncodingGPU.cuh:745-750).
//       Where the forward has kept the slopes of the features, both derivatives w.r.t. the positions read those instead of gathering
//       (penc_slopes.hpp).
//   small tables and small batches : a workgroup takes 64 points and all their levels, for the position
//       gradient and for results in rows (block_backward_pos_kernel, block_rows_kernel).
//   table backward (first order, the scattering half of the double backward, or both) : workgroups of
//       512 threads (1024 above 256 bins) walk groups of 2 to 16 tiles of points; neighbouring workgroups of a die take
//       the same points at different levels.  The scatter itself (LDS accumulate cache, slot-range
//       bins, direct atomics) is described in penc_scatter.hpp; small and ordinary batches are sorted
//       by slot range instead (penc_group_sort.hpp).
//   A level whose anneal-window weight is exactly 0 contributes exactly 0 everywhere (for finite
//   table values), so such levels skip the table traffic and only store their zeros.
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <mutex>
#include <type_traits>

#include "../../include/penc.h"
#include "penc_cells.hpp"
#include "penc_lattice.hpp"
#include "penc_group_sort.hpp"
#include "penc_reduce.hpp"
#include "penc_scatter.hpp"
#include "penc_slopes.hpp"
#include "penc_table_backward.hpp"

namespace penc {

constexpr int kPosLevelsPerGroup = 2;  // levels a position-gradient thread sums in registers (figures at backward_pos_kernel)

constexpr int kDefaultLevelsPerPass = 1 << 20;  // by default the suggested workspace bins all levels in one pass (measured fastest)

template <int D>
__device__ __forceinline__ fvec<D> load_point(const float* __restrict__ positions, int64_t n) {
    const float* p = positions + n * D;
    fvec<D> pos;
    static_for<D>(PENC_BODY(i) {
        PENC_INDEX(i); pos[i] = p[i]; });
    return pos;
}

// The D+1 table entries of a simplex (F features each: one load of F elements per vertex, two of 16
// bytes for eight floats), fetched back to back so that all loads are in flight together.
// f[k][r] is feature k of vertex r.  T is the table's element type: float, or __half / bfloat16_bits
// for a table kept in 16 bits (the values are widened exactly; all arithmetic stays fp32).
template <int D, int F>
struct Vertices {
    fvec<D + 1> f[F];
};
template <int D, int F, typename T>
__device__ __forceinline__ Vertices<D, F> load_vertices(const T* __restrict__ level_table, uvec<D + 1> h,
                                                        uint32_t capacity, uint32_t cap_mask) {
    static_assert(F == 2 || F == 4 || F == 8, "two, four or eight features per level");
    Vertices<D, F> v;
    static_for<D + 1>(PENC_BODY(r) {
        PENC_INDEX(r);
        const size_t slot = to_slot(h[r], capacity, cap_mask);
        if constexpr (sizeof(T) == 2) {
            // F halves in one load of 4, 8 or 16 bytes
            using Packed = typename std::conditional<F == 2, uint32_t, typename std::conditional<F == 4, uint2, uint4>::type>::type;
            const Packed raw = *reinterpret_cast<const Packed*>(level_table + F * slot);
            uint32_t words[F / 2];
            __builtin_memcpy(words, &raw, sizeof(raw));
            static_for<F / 2>(PENC_BODY(q) {
                PENC_INDEX(q);
                if constexpr (std::is_same<T, bfloat16_bits>::value) {
                    v.f[2 * q + 0][r] = __builtin_bit_cast(float, words[q] << 16);
                    v.f[2 * q + 1][r] = __builtin_bit_cast(float, words[q] & 0xFFFF0000u);
                } else {
                    const float2 x = __half22float2(__builtin_bit_cast(__half2, words[q]));
                    v.f[2 * q + 0][r] = x.x;
                    v.f[2 * q + 1][r] = x.y;
                }
            });
        } else if constexpr (F == 2) {
            const float2 x = *reinterpret_cast<const float2*>(level_table + 2 * slot);
            v.f[0][r] = x.x;
            v.f[1][r] = x.y;
        } else {
            static_for<F / 4>(PENC_BODY(q) {
                PENC_INDEX(q);
                const float4 x = *reinterpret_cast<const float4*>(level_table + F * slot + 4 * q);
                v.f[4 * q + 0][r] = x.x;
                v.f[4 * q + 1][r] = x.y;
                v.f[4 * q + 2][r] = x.z;
                v.f[4 * q + 3][r] = x.w;
            });
        }
    });
    return v;
}

// ------------------------------------------------------------------------------------------
// which (tile of points, row of levels) a workgroup of a gathering kernel takes
//
// A row is one level, or two levels `rows` apart: with the usual coarse-to-fine level list a level whose gathers hit the
// first-level cache with one that waits for the L2.  Each die has an L2 of its own, and workgroup i runs on die i % dies.
// With the grid as (tile, row) every die gathers from every level, so each of the eight L2s fetches the whole table: 400 MB
// for 24 slices of 2 MiB, 10 us whatever the number of points, a third of the forward of 2^16 points.  With `segment` != 0
// the (row, tile) pairs, row by row, are cut into rounds * dies segments and a die takes one segment of each round, in
// alternating directions (the dies' shares of coarse and fine rows then even out); a table slice is fetched by one or two dies.
// Measured, forward, D = 3, 24 levels of 2^18 slots (before -> after): 2^13 points 10.3 -> 5.3 us, 2^15 22.2 -> 12.6,
// 2^16 33.3 -> 23.4, 2^18 85.6 -> 76.4, 2^20 289 -> 283.
struct LevelMap {
    uint32_t tiles;    // workgroups per row
    uint32_t rows;
    uint32_t segment;  // (row, tile) pairs per segment; 0: the grid is (tile, row)
    uint32_t dies;
};
// The levels whose window weight is not 0, of up to 64; of more, all of them.  (For every lane of a wave at once.)
__device__ __forceinline__ unsigned long long live_levels(const float* __restrict__ window, int n_levels) {
    const int lane = static_cast<int>(threadIdx.x & 63);
    return __ballot(lane < n_levels && window[lane] != 0.0f);
}
constexpr int kMostLiveLevels = 64;
// Into how many groups of `per_group` the position gradient puts its levels.
__device__ __forceinline__ int live_groups(unsigned long long live, int n_levels, int per_group) {
    const int count = n_levels <= kMostLiveLevels ? __popcll(live) : n_levels;
    return (count + per_group - 1) / per_group;
}
__device__ __forceinline__ bool locate_work(const LevelMap& map, uint32_t& tile, uint32_t& row) {
    if (map.segment == 0u) {
        tile = blockIdx.x;
        row = blockIdx.y;
        return true;
    }
    const uint32_t die = blockIdx.x % map.dies, j = blockIdx.x / map.dies;
    const uint32_t round = j / map.segment;
    const uint32_t at = (round * map.dies + ((round & 1u) ? map.dies - 1u - die : die)) * map.segment + j % map.segment;
    row = at / map.tiles;
    tile = at % map.tiles;
    return row < map.rows;
}

// ------------------------------------------------------------------------------------------
// forward (EncodingGPU.cuh:68-256)
//
// One thread per point and one or two levels (the host says which).  Measured alternatives, all
// slower or equal: 2 or 4 points per
// thread (more loads in flight per lane: no gain, the kernel already runs at the rate this GPU
// sustains for random 8-byte loads from a 2 MiB slice); walking all the levels inside the thread with
// the positions kept in registers (20% slower at 2^20 points, 3x slower at 2^16: fewer, longer
// waves lose more than the re-read positions cost); interleaving workgroups of a coarse
// (compute-bound) and a fine (gather-bound) level, which takes the fine level's slice out of L2
// (30% slower).

// With kSlopes it also leaves the slopes of every feature behind (penc_slopes.hpp).  With kChosen the levels that `chosen` names are gathered from
// `cells` (chosen_cells_kernel).
template <int D, int F, typename T, bool kSlopes, bool kChosen>
__global__ void __launch_bounds__(kBlock)
forward_kernel(int n_points, int n_levels, int n_all_levels, LevelMap map, uint32_t capacity, uint32_t cap_mask, uint32_t in_cells,
               const float* __restrict__ positions, const T* __restrict__ table,
               const float* __restrict__ scale_factor, const float* __restrict__ random_shift,
               const float* __restrict__ window, float* __restrict__ sliced, float points_scaling, float* __restrict__ slopes,
               const T* __restrict__ cells, const uint32_t* __restrict__ chosen) {
    uint32_t tile, row;
    if (!locate_work(map, tile, row)) return;
    const int n = tile * kBlock + threadIdx.x;
    if (n >= n_points) return;
    __shared__ uint2 columns[(D + 1) * kBlock];
    const fvec<D> point = load_point<D>(positions, n);
    if (row == 0u) {  // extra levels carrying the raw positions (:106-121)
        for (int level = n_levels; level < n_all_levels; ++level) {
            float* out = sliced + (static_cast<size_t>(level) * F) * n_points + n;
            const int src = (level - n_levels) * F;
            const float* p = positions + static_cast<size_t>(n) * D;
            static_for<F>(PENC_BODY(k) {
                PENC_INDEX(k);
                out[static_cast<size_t>(k) * n_points] = src + k < D ? p[src + k] * points_scaling : 0.0f;
            });
        }
    }
#pragma unroll 1
    for (int level = static_cast<int>(row); level < n_levels; level += static_cast<int>(map.rows)) {
        float* out = sliced + (static_cast<size_t>(level) * F) * n_points + n;  // feature k at out[k * n_points]
        const float w_level = window[level];
        uint32_t here = 0u;
        if constexpr (kChosen) here = chosen[level];  // (before it is waited for)
        if (w_level == 0.0f) {
            static_for<F>(PENC_BODY(k) {
                PENC_INDEX(k); out[static_cast<size_t>(k) * n_points] = 0.0f; });
            continue;
        }
        const Located<D> s = locate<D>(point, random_shift + level * D, scale_factor + level * D);
        // residuals and hash steps into rank order through LDS: up to 6% faster than the select chains
        // of vertex_hashes() / barycentric() at D = 8, equal at D = 3
        uvec<D + 1> h;
        fvec<D + 1> sorted;
        sort_by_rank_lds<D>(columns + threadIdx.x, kBlock, s.rank, s.delta, s.hash0, sorted, h);
        const fvec<D + 1> w = barycentric_of_sorted<D>(sorted);
        const T* slice = table;
        if constexpr (kChosen) {
            if (here != 0u) {
                slice = cells;
                h = hashes_in_cells<D, line_slots<F, T>()>(h);
            }
        } else {
            h = hashes_in_copy<D, F, T>(in_cells, h);
        }
        const Vertices<D, F> v = load_vertices<D, F, T>(slice + static_cast<size_t>(level) * capacity * F, h, capacity, cap_mask);
        fvec<F> acc = 0.0f;
        static_for<D + 1>(PENC_BODY(r) {
            PENC_INDEX(r);
            const float wr = w[r] * w_level;
            static_for<F>(PENC_BODY(k) {
                PENC_INDEX(k); acc[k] = acc[k] + v.f[k][r] * wr; });
        });
        static_for<F>(PENC_BODY(k) {
            PENC_INDEX(k);
            // written once and not read here: the non-temporal hint keeps it from displacing the level's table slice
            __builtin_nontemporal_store(acc[k], out + static_cast<size_t>(k) * n_points);
        });
        if constexpr (kSlopes)
            store_slopes<D, F>(v.f, s.rank, columns + threadIdx.x, kBlock, scale_factor + level * D, slopes + slope_offset<D, F>(n_points, level, n));
    }
}

// ------------------------------------------------------------------------------------------
// backward w.r.t. positions (EncodingGPU.cuh:530-769)

// One thread per (point, group of levels): the levels of the group are summed in
// registers and stored once, at out[group][point][D].  With a single group (no workspace) `out` is
// the position gradient itself; otherwise it is a partial buffer that reduce_level_groups_kernel
// sums, in ascending group order, so the result is deterministic either way.  Small groups keep
// the whole chip on the same few levels at a time (their table slices stay in L2) and give the
// launch many more, shorter waves than one thread per point walking all levels.  (Doing this
// kernel's rank permutations through LDS, as the forward does, was measured: no gain.)
//
// Groups are made of the levels that the window leaves: with half of them masked there are half as many groups, whose sums are
// stored and read back, where a grouping of all levels left groups of one (2^20 points, 16 of 24 levels of 2^22 slots: 418 ->
// 385 us).  Two levels to a group: one, two, three, four at 2^20 points, D = 3, 24 levels of 2^18 slots 499 / 458 / 449 / 467 us,
// of 2^22 slots 1026 / 887 / 946 / 975; D = 4 632 / 547 / 557 / 588; D = 6, 16 levels, 2^19 points 305 / 270 / 269 / 277;
// D = 8, 2^19 slots 444 / 420 / 459 / 487.
template <int D, int F, typename T>
__global__ void __launch_bounds__(kBlock)
backward_pos_kernel(int n_points, int n_levels, int per_group, LevelMap map, uint32_t capacity, uint32_t cap_mask, uint32_t in_cells,
                    const float* __restrict__ positions, const T* __restrict__ table,
                    const float* __restrict__ scale_factor, const float* __restrict__ random_shift,
                    const float* __restrict__ window, const float* __restrict__ grad_sliced,
                    float* __restrict__ out) {
    uint32_t tile, row;
    if (!locate_work(map, tile, row)) return;
    const int n = tile * kBlock + threadIdx.x;
    const fvec<D> pos = load_point<D>(positions, n < n_points ? n : n_points - 1);  // (on its way while the window is looked at)
    unsigned long long live = live_levels(window, n_levels);
    const int groups = map.rows > 1u ? live_groups(live, n_levels, per_group) : 1;
    if (static_cast<int>(row) >= groups || n >= n_points) return;
    fvec<D> total = 0.0f;
    // The levels of a group are `groups` apart, not adjacent: with the usual coarse-to-fine level list a
    // group then pairs a coarse level, whose points share few slots, with a fine one, and the table slices
    // a die gathers from at any time fit its L2 (two adjacent fine levels are 4 MiB at 2^18 slots,
    // an L2's whole capacity).
    const int left = __popcll(live);
    const bool masked = n_levels <= kMostLiveLevels && left < n_levels;  // `live` names the levels, else their numbers do
    const int count = masked ? left : n_levels;
    int passed = 0;  // of `live`
    for (int k = static_cast<int>(row); k < count; k += groups) {
        int level = k;
        if (masked) {
            for (; passed < k; ++passed) live &= live - 1ull;
            level = __builtin_ctzll(live);
        }
        const float w_level = window[level];
        if (w_level == 0.0f) continue;
        const float* sf = scale_factor + level * D;
        const Located<D> s = locate<D>(pos, random_shift + level * D, sf);
        const uvec<D + 1> h = vertex_hashes<D>(s.rank, s.hash0);
        const Vertices<D, F> v = load_vertices<D, F, T>(table + static_cast<size_t>(level) * capacity * F,
                                                         hashes_in_copy<D, F, T>(in_cells, h), capacity, cap_mask);
        const float* gp = grad_sliced + (static_cast<size_t>(level) * F) * n_points + n;
        // the upstream gradient is read once (non-temporal: it should not displace the table slices)
        fvec<D + 1> dB = (v.f[0] * w_level) * __builtin_nontemporal_load(gp);  // :688-689, feature by feature
        static_for<F - 1>(PENC_BODY(kk) {
            PENC_INDEX(kk);
            constexpr int k = kk + 1;
            dB += (v.f[k] * w_level) * __builtin_nontemporal_load(gp + static_cast<size_t>(k) * n_points);
        });
        total += bary_grad_to_pos_grad<D>(s.rank, dB, sf);
    }
    float* o = out + (static_cast<size_t>(row) * n_points + n) * D;
    static_for<D>(PENC_BODY(i) {
        PENC_INDEX(i);
        o[i] = total[i];
    });
}

// Sums the partial position gradients of the groups in ascending order, one value to a thread.  What it waits for at small sizes
// is its chain of loads: those of kTogether groups are issued together (2^15 points, 12 groups: 11.5 -> 3.9 us; large sums are
// bound by the memory, 2^20 points 31 us).
// (16 bytes to a lane are slower, 50 us: the groups' sums lie a multiple of the memory's interleave apart, and loads of
// several groups from the same few waves meet on one channel.)
__global__ void __launch_bounds__(kBlock)
reduce_level_groups_kernel(const float* __restrict__ partial, const float* __restrict__ window, int per_group, int n_levels,
                           size_t n_values, float* __restrict__ out) {
    constexpr int kTogether = 8;
    const int groups = live_groups(live_levels(window, n_levels), n_levels, per_group);
    const size_t stride = static_cast<size_t>(gridDim.x) * kBlock;
    for (size_t i = static_cast<size_t>(blockIdx.x) * kBlock + threadIdx.x; i < n_values; i += stride) {
        float acc = groups > 0 ? partial[i] : 0.0f;
        for (int base = 1; base < groups; base += kTogether) {
            float v[kTogether];
#pragma unroll
            for (int u = 0; u < kTogether; ++u) v[u] = base + u < groups ? partial[static_cast<size_t>(base + u) * n_values + i] : 0.0f;
#pragma unroll
            for (int u = 0; u < kTogether; ++u)
                if (base + u < groups) acc += v[u];
        }
        out[i] = acc;
    }
}

// ------------------------------------------------------------------------------------------
// double backward from d(loss)/d(position gradient), the half that gathers: gradient w.r.t.
// grad_sliced_values (EncodingGPU.cuh:1260-1493).  One thread per point and one or two levels, like
// the forward.  (The other half, the scatter into the table gradient, is
// backward_table_kernel<D, false, true>.  One kernel doing both, with eight tiles per workgroup,
// was measured 7-13% slower than the two: the gathering half wants small workgroups, the scattering
// half large groups of points with the levels interleaved.)

template <int D, int F, typename T>
__global__ void __launch_bounds__(kBlock)
grad_grad_kernel(int n_points, int n_levels, int n_all_levels, LevelMap map, uint32_t capacity, uint32_t cap_mask, uint32_t in_cells,
                 const float* __restrict__ positions, const T* __restrict__ table,
                 const float* __restrict__ scale_factor, const float* __restrict__ random_shift,
                 const float* __restrict__ window, const float* __restrict__ double_pos_grad,
                 float* __restrict__ grad_grad_sliced) {
    uint32_t tile, row;
    if (!locate_work(map, tile, row)) return;
    const int n = tile * kBlock + threadIdx.x;
    if (n >= n_points) return;
    __shared__ uint2 columns[(D + 1) * kBlock];
    const fvec<D> point = load_point<D>(positions, n), q = load_point<D>(double_pos_grad, n);
    if (row == 0u) {  // concat levels: zeros (:1290-1295)
        for (size_t k = static_cast<size_t>(n_levels) * F; k < static_cast<size_t>(n_all_levels) * F; ++k) grad_grad_sliced[k * n_points + n] = 0.0f;
    }
#pragma unroll 1
    for (int level = static_cast<int>(row); level < n_levels; level += static_cast<int>(map.rows)) {
        float* o = grad_grad_sliced + (static_cast<size_t>(level) * F) * n_points + n;
        const float w_level = window[level];
        if (w_level == 0.0f) {
            static_for<F>(PENC_BODY(k) {
                PENC_INDEX(k); o[static_cast<size_t>(k) * n_points] = 0.0f; });
            continue;
        }
        const float* sf = scale_factor + level * D;
        const Located<D> s = locate<D>(point, random_shift + level * D, sf);
        // one trip through the thread's LDS column puts both the elevated gradient and the hash steps
        // into rank order (as in the forward)
        uvec<D + 1> h;
        fvec<D + 1> sorted;
        sort_by_rank_lds<D>(columns + threadIdx.x, kBlock, s.rank, pos_grad_grad_to_elevated<D>(q, sf), s.hash0, sorted, h);
        const Vertices<D, F> v = load_vertices<D, F, T>(table + static_cast<size_t>(level) * capacity * F,
                                                         hashes_in_copy<D, F, T>(in_cells, h), capacity, cap_mask);
        // dB[r] * w_level, then times the vertex value (:1484-1485)
        const fvec<D + 1> wr = sorted_elevated_grad_to_bary<D>(sorted) * w_level;
        fvec<F> gg = 0.0f;
        static_for<D + 1>(PENC_BODY(r) {
            PENC_INDEX(r);
            static_for<F>(PENC_BODY(k) {
                PENC_INDEX(k); gg[k] += wr[r] * v.f[k][r]; });
        });
        static_for<F>(PENC_BODY(k) {
            PENC_INDEX(k); o[static_cast<size_t>(k) * n_points] = gg[k]; });
    }
}

// ------------------------------------------------------------------------------------------
// all levels of a block of points in one workgroup
//
// A workgroup takes 64 points and all their levels: lane = point, wave w takes levels w, w + kBlockWaves, ...  What needs
// several launches at a level a time is one here: the sum of the position gradient over the levels happens in LDS, and rows
// (of a result, or of an upstream gradient) pass through an LDS tile, so no transpose precedes or follows.  Every die then gathers
// from every level, which is why this is for tables an L2 holds as a whole and for batches whose time is launches and latency
// (takes_point_blocks says where the lines lie).
constexpr int kBlockWaves = 8, kBlockPoints = 64, kPointBlock = kBlockWaves * kBlockPoints;

// Position gradient.  The upstream gradient is [level][feature][n], or (kRows) rows of `grad_row_stride` floats, of which the
// [level][feature][n] copy is left in grad_level_major when the caller wants it.
template <int D, int F, typename T, bool kRows>
__global__ void __launch_bounds__(kPointBlock)
block_backward_pos_kernel(int n_points, int n_levels, uint32_t capacity, uint32_t cap_mask, uint32_t in_cells, const float* __restrict__ positions,
                          const T* __restrict__ table, const float* __restrict__ scale_factor, const float* __restrict__ random_shift,
                          const float* __restrict__ window, const float* __restrict__ grad, int64_t grad_row_stride,
                          float* __restrict__ grad_level_major, float* __restrict__ out) {
    extern __shared__ float tile[];  // rows: kBlockPoints x (columns | 1)
    __shared__ float partial[kBlockWaves][kBlockPoints * D];
    const int base = blockIdx.x * kBlockPoints, count = n_points - base < kBlockPoints ? n_points - base : kBlockPoints;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int columns = n_levels * F, pitch = columns | 1;
    const int n = base + (lane < count ? lane : count - 1);
    const fvec<D> pos = load_point<D>(positions, n);
    if constexpr (kRows) {
        const float* const rows = grad + static_cast<int64_t>(base) * grad_row_stride;
        for (int r = wave; r < count; r += kBlockWaves)
            for (int c = lane; c < columns; c += 64) tile[r * pitch + c] = rows[r * grad_row_stride + c];
        __syncthreads();
        if (grad_level_major != nullptr && lane < count)
            for (int c = wave; c < columns; c += kBlockWaves) grad_level_major[static_cast<size_t>(c) * n_points + n] = tile[lane * pitch + c];
    }
    const int row = n - base;
    fvec<D> total = 0.0f;
    for (int level = wave; level < n_levels; level += kBlockWaves) {
        const float w_level = window[level];
        if (w_level == 0.0f) continue;
        const float* sf = scale_factor + level * D;
        const Located<D> s = locate<D>(pos, random_shift + level * D, sf);
        const uvec<D + 1> h = vertex_hashes<D>(s.rank, s.hash0);
        const Vertices<D, F> v = load_vertices<D, F, T>(table + static_cast<size_t>(level) * capacity * F,
                                                         hashes_in_copy<D, F, T>(in_cells, h), capacity, cap_mask);
        const auto upstream = [&](int k) {
            if constexpr (kRows) return tile[row * pitch + level * F + k];
            else return grad[(static_cast<size_t>(level) * F + k) * n_points + n];
        };
        fvec<D + 1> dB = (v.f[0] * w_level) * upstream(0);  // :688-689, feature by feature
        static_for<F - 1>(PENC_BODY(kk) {
            PENC_INDEX(kk);
            dB += (v.f[kk + 1] * w_level) * upstream(kk + 1);
        });
        total += bary_grad_to_pos_grad<D>(s.rank, dB, sf);
    }
    static_for<D>(PENC_BODY(i) {
        PENC_INDEX(i);
        partial[wave][lane * D + i] = total[i];
    });
    __syncthreads();
    for (int i = threadIdx.x; i < count * D; i += kPointBlock) {
        float acc = partial[0][i];
#pragma unroll
        for (int w = 1; w < kBlockWaves; ++w) acc += partial[w][i];
        out[static_cast<size_t>(base) * D + i] = acc;
    }
}

// The forward (kSecond = false) or the gradient w.r.t. the upstream gradient (kSecond = true) as rows of `row_stride` floats.  With
// kSlopes the forward also leaves the slopes of every feature behind (penc_slopes.hpp): a call that keeps them is the one launch that it is
// without them.
template <int D, int F, typename T, bool kSlopes, bool kSecond>
__global__ void __launch_bounds__(kPointBlock)
block_rows_kernel(int n_points, int n_levels, int n_all_levels, uint32_t capacity, uint32_t cap_mask, uint32_t in_cells, const float* __restrict__ positions,
                  const T* __restrict__ table, const float* __restrict__ scale_factor, const float* __restrict__ random_shift,
                  const float* __restrict__ window, const float* __restrict__ double_pos_grad, float points_scaling,
                  float* __restrict__ rows, int64_t row_stride, float* __restrict__ slopes) {
    extern __shared__ float tile[];  // kBlockPoints x (columns | 1)
    __shared__ uint2 rank_columns[kSlopes ? (D + 1) * kPointBlock : 1];
    const int base = blockIdx.x * kBlockPoints, count = n_points - base < kBlockPoints ? n_points - base : kBlockPoints;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int columns = n_all_levels * F, pitch = columns | 1;
    const int n = base + (lane < count ? lane : count - 1);
    const fvec<D> pos = load_point<D>(positions, n);
    fvec<D> q = 0.0f;
    if constexpr (kSecond) q = load_point<D>(double_pos_grad, n);
    float* const mine = tile + lane * pitch;
    for (int level = wave; level < n_all_levels; level += kBlockWaves) {
        if (level >= n_levels) {  // extra levels: the raw positions (:106-121), or zeros (:1290-1295)
            const int src = (level - n_levels) * F;
            const float* p = positions + static_cast<size_t>(n) * D;
            static_for<F>(PENC_BODY(k) {
                PENC_INDEX(k);
                mine[level * F + k] = !kSecond && src + k < D ? p[src + k] * points_scaling : 0.0f;
            });
            continue;
        }
        const float w_level = window[level];
        fvec<F> acc = 0.0f;
        if (w_level != 0.0f) {
            const float* sf = scale_factor + level * D;
            const Located<D> s = locate<D>(pos, random_shift + level * D, sf);
            const uvec<D + 1> h = vertex_hashes<D>(s.rank, s.hash0);
            const Vertices<D, F> v = load_vertices<D, F, T>(table + static_cast<size_t>(level) * capacity * F,
                                                         hashes_in_copy<D, F, T>(in_cells, h), capacity, cap_mask);
            const fvec<D + 1> w = kSecond ? pos_grad_grad_to_bary<D>(s.rank, q, sf) * w_level : barycentric<D>(s.rank, s.delta) * w_level;
            static_for<D + 1>(PENC_BODY(r) {
                PENC_INDEX(r);
                static_for<F>(PENC_BODY(k) {
                    PENC_INDEX(k); acc[k] = acc[k] + v.f[k][r] * w[r]; });
            });
            if constexpr (kSlopes)  // (lanes without a point repeat the last one)
                store_slopes<D, F>(v.f, s.rank, rank_columns + threadIdx.x, kPointBlock, sf, slopes + slope_offset<D, F>(n_points, level, n));
        }
        static_for<F>(PENC_BODY(k) {
            PENC_INDEX(k); mine[level * F + k] = acc[k]; });
    }
    __syncthreads();
    float* const to = rows + static_cast<int64_t>(base) * row_stride;
    for (int r = wave; r < count; r += kBlockWaves)
        for (int c = lane; c < columns; c += 64) to[r * row_stride + c] = tile[r * pitch + c];
}

// ------------------------------------------------------------------------------------------
// optimiser step on the table

// One fused AdamW update (decoupled weight decay, no amsgrad) in the order torch.optim.AdamW applies
// it: p *= 1 - lr*wd; m += (1-b1)(g - m); v = b2 v + (1-b2) g^2; p -= step_size * m / (sqrt(v)/c2 + eps).
// With skip_zero an entry whose gradient is exactly 0 is left alone altogether (moments, decay and
// value), which is how hash-grid tables are usually trained: most slots of a large table get no
// gradient in a step.  Four values per thread where the arrays allow 16-byte accesses.
struct AdamWStep {
    float decay;        // 1 - lr * weight_decay
    float one_minus_b1, b2, one_minus_b2;
    float step_size;    // lr / (1 - b1^step)
    float inv_c2;       // 1 / sqrt(1 - b2^step)
    float eps;
};
__device__ __forceinline__ void adamw_update(const AdamWStep& a, bool skip_zero, float g, float& p, float& m, float& v) {
    if (skip_zero && g == 0.0f) return;
    p = p * a.decay;
    m = m + a.one_minus_b1 * (g - m);
    v = v * a.b2 + a.one_minus_b2 * (g * g);
    p = p - a.step_size * (m / (__builtin_sqrtf(v) * a.inv_c2 + a.eps));
}
template <bool kVector>
__global__ void __launch_bounds__(kBlock)
adamw_step_kernel(float* __restrict__ params, const float* __restrict__ grads, float* __restrict__ exp_avg,
                  float* __restrict__ exp_avg_sq, size_t n, AdamWStep a, int skip_zero) {
    const size_t i = static_cast<size_t>(blockIdx.x) * kBlock + threadIdx.x;
    if constexpr (kVector) {
        if (i * 4 >= n) return;
        const float4 g = reinterpret_cast<const float4*>(grads)[i];
        if (skip_zero && g.x == 0.0f && g.y == 0.0f && g.z == 0.0f && g.w == 0.0f) return;
        float4 p = reinterpret_cast<float4*>(params)[i], m = reinterpret_cast<float4*>(exp_avg)[i],
               v = reinterpret_cast<float4*>(exp_avg_sq)[i];
        adamw_update(a, skip_zero, g.x, p.x, m.x, v.x);
        adamw_update(a, skip_zero, g.y, p.y, m.y, v.y);
        adamw_update(a, skip_zero, g.z, p.z, m.z, v.z);
        adamw_update(a, skip_zero, g.w, p.w, m.w, v.w);
        reinterpret_cast<float4*>(params)[i] = p;
        reinterpret_cast<float4*>(exp_avg)[i] = m;
        reinterpret_cast<float4*>(exp_avg_sq)[i] = v;
    } else {
        if (i >= n) return;
        float p = params[i], m = exp_avg[i], v = exp_avg_sq[i];
        const float g = grads[i];
        if (skip_zero && g == 0.0f) return;
        adamw_update(a, skip_zero, g, p, m, v);
        params[i] = p;
        exp_avg[i] = m;
        exp_avg_sq[i] = v;
    }
}

// The same update, or only the clearing of the gradient, restricted to the slot ranges a caller's map of
// touched ranges names (the sparse entry points): one workgroup per (slot range, level) looks at the
// range's flags (one per pair of features) and leaves at once when nothing was added there, so the
// cost follows what the batch touched and not the size of the table.  Within a touched range an entry
// with a gradient of exactly 0 is left alone, as with skip_zero.  `clear` zeroes the gradients the
// workgroup has used and the range's flags, which is what the next accumulation expects.
// The update takes 512 threads to a range: a workgroup's time is a chain of waits, and the launch ends with the last few of them (the sizes
// below, 128 / 256 / 512 / 1024 threads: 144 / 134 / 126 / 131 us).  Clearing alone keeps 256: it mostly finds nothing (an empty map of
// 12288 ranges 4.7 / 7.2 / 12.9 us with 256 / 512 / 1024).
template <bool kUpdate>
constexpr uint32_t kTouchedBlock = kUpdate ? 512u : 256u;

template <bool kUpdate, typename Vec>
__global__ void __launch_bounds__(kTouchedBlock<kUpdate>)
touched_ranges_kernel(float* __restrict__ params, float* __restrict__ grads, float* __restrict__ exp_avg,
                      float* __restrict__ exp_avg_sq, uint32_t capacity, uint32_t nr_feat, uint32_t n_ranges,
                      uint32_t range_shift, uint32_t* __restrict__ touched, AdamWStep a, int clear) {
    constexpr uint32_t kPer = sizeof(Vec) / sizeof(float);
    const uint32_t range = blockIdx.x, level = blockIdx.y, pairs = nr_feat / 2;
    uint32_t any = 0u;
    for (uint32_t p = 0; p < pairs; ++p) any |= touched[(static_cast<size_t>(level) * pairs + p) * n_ranges + range];
    if (any == 0u) return;
    const uint32_t slot0 = range << range_shift;
    const uint32_t slots = capacity - slot0 < (1u << range_shift) ? capacity - slot0 : (1u << range_shift);
    const size_t base = (static_cast<size_t>(level) * capacity + slot0) * nr_feat;  // a multiple of kPer floats (the host checks)
    const uint32_t n_vec = slots * nr_feat / kPer;
    Vec* const g_at = reinterpret_cast<Vec*>(grads + base);
    // What a workgroup waits for is memory, first for the gradients and then for the values of those that are not zero: both are
    // fetched for kTogether entries of a thread at a time (24 levels of 2^22 slots, a third of the ranges touched, 445 MiB read and 78
    // written: 145 us one by one, 134 with four; with the 512 threads above 126, eight 147).  The gradients are read once here
    // and need not displace anything: loaded with the non-temporal hint 119 us (the moments, loaded and stored that way, 145).
    constexpr uint32_t kTogether = 4;
    for (uint32_t first = threadIdx.x; first < n_vec; first += kTogether * kTouchedBlock<kUpdate>) {
        Vec gv[kTogether], pv[kTogether], mv[kTogether], vv[kTogether];
        bool nonzero[kTogether];
#pragma unroll
        for (uint32_t u = 0; u < kTogether; ++u) {
            const uint32_t i = first + u * kTouchedBlock<kUpdate>;
            if constexpr (kUpdate) {
                typedef float Words __attribute__((ext_vector_type(sizeof(Vec) / sizeof(float))));
                const Words w = __builtin_nontemporal_load(reinterpret_cast<const Words*>(g_at + (i < n_vec ? i : first)));
                __builtin_memcpy(&gv[u], &w, sizeof(Vec));
            } else {
                gv[u] = g_at[i < n_vec ? i : first];
            }
        }
#pragma unroll
        for (uint32_t u = 0; u < kTogether; ++u) {
            const uint32_t i = first + u * kTouchedBlock<kUpdate>;
            float g[kPer];
            __builtin_memcpy(g, &gv[u], sizeof(Vec));
            nonzero[u] = false;
#pragma unroll
            for (uint32_t k = 0; k < kPer; ++k) nonzero[u] = nonzero[u] || g[k] != 0.0f;
            nonzero[u] = nonzero[u] && i < n_vec;
            if constexpr (kUpdate) {
                if (nonzero[u]) {
                    pv[u] = reinterpret_cast<Vec*>(params + base)[i];
                    mv[u] = reinterpret_cast<Vec*>(exp_avg + base)[i];
                    vv[u] = reinterpret_cast<Vec*>(exp_avg_sq + base)[i];
                }
            }
        }
#pragma unroll
        for (uint32_t u = 0; u < kTogether; ++u) {
            const uint32_t i = first + u * kTouchedBlock<kUpdate>;
            if (!nonzero[u]) continue;
            if constexpr (kUpdate) {
                float g[kPer], p[kPer], m[kPer], v[kPer];
                __builtin_memcpy(g, &gv[u], sizeof(Vec));
                __builtin_memcpy(p, &pv[u], sizeof(Vec));
                __builtin_memcpy(m, &mv[u], sizeof(Vec));
                __builtin_memcpy(v, &vv[u], sizeof(Vec));
#pragma unroll
                for (uint32_t k = 0; k < kPer; ++k) adamw_update(a, true, g[k], p[k], m[k], v[k]);
                __builtin_memcpy(&pv[u], p, sizeof(Vec));
                __builtin_memcpy(&mv[u], m, sizeof(Vec));
                __builtin_memcpy(&vv[u], v, sizeof(Vec));
                reinterpret_cast<Vec*>(params + base)[i] = pv[u];
                reinterpret_cast<Vec*>(exp_avg + base)[i] = mv[u];
                reinterpret_cast<Vec*>(exp_avg_sq + base)[i] = vv[u];
            }
            if (clear) {
                Vec zero;
                __builtin_memset(&zero, 0, sizeof(zero));
                g_at[i] = zero;
            }
        }
    }
    if (clear) {
        __syncthreads();  // every thread has read the flags
        if (threadIdx.x < pairs) touched[(static_cast<size_t>(level) * pairs + threadIdx.x) * n_ranges + range] = 0u;
    }
}

// ------------------------------------------------------------------------------------------
// introspection

// kRoutine selects which of the equivalent device routines produces the slots and weights: the
// compare-and-select chains (vertex_hashes / barycentric: position backward, sorted groups), the thread-private LDS column
// (sort_by_rank_lds: forward, grad-of-grad), or what the scatter takes (scatter_simplex: a sorting network, of the first order or of both).
enum SimplexRoutine : int { kBySelects = 0, kByLds = 1, kByNetwork = 2, kByNetworkBothOrders = 3 };
template <int D, int kRoutine>
__global__ void __launch_bounds__(kBlock)
simplex_debug_kernel(int n_points, uint32_t capacity, uint32_t cap_mask, const float* __restrict__ positions,
                     const float* __restrict__ scale_factor, const float* __restrict__ random_shift,
                     int* __restrict__ rem0, int* __restrict__ rank, int* __restrict__ slot,
                     float* __restrict__ bary) {
    const int n = blockIdx.x * kBlock + threadIdx.x;
    if (n >= n_points) return;
    const int level = blockIdx.y;
    const Located<D> s = locate<D>(load_point<D>(positions, n), random_shift + level * D, scale_factor + level * D);
    uvec<D + 1> h;
    fvec<D + 1> w;
    if constexpr (kRoutine >= kByNetwork) {
        const fvec<D> point = load_point<D>(positions, n);
        const CyclicSimplex<D> c = scatter_simplex<D, true, kRoutine == kByNetworkBothOrders>(point, point, random_shift + level * D,
                                                                                             scale_factor + level * D, capacity, cap_mask);
        h = turn_back<D + 1>(c.slot, c.turned);
        w = turn_back<D + 1>(c.w, c.turned);
    } else if constexpr (kRoutine == kByLds) {
        __shared__ uint2 columns[(D + 1) * kBlock];
        fvec<D + 1> sorted;
        sort_by_rank_lds<D>(columns + threadIdx.x, kBlock, s.rank, s.delta, s.hash0, sorted, h);
        w = barycentric_of_sorted<D>(sorted);
    } else {
        h = vertex_hashes<D>(s.rank, s.hash0);
        w = barycentric<D>(s.rank, s.delta);
    }
    const size_t o = (static_cast<size_t>(level) * n_points + n) * (D + 1);
    static_for<D + 1>(PENC_BODY(i) {
        PENC_INDEX(i);
        if (rem0) rem0[o + i] = s.rem0[i];
        if (rank) rank[o + i] = s.rank[i];
        if (slot) slot[o + i] = static_cast<int>(kRoutine >= kByNetwork ? h[i] : to_slot(h[i], capacity, cap_mask));
        if (bary) bary[o + i] = w[i];
    });
}

// dst[c][r] = src[r][c] for a tall matrix (rows = points, cols = 2 * levels): what turns the
// row-major upstream gradient (N, 2L) an MLP delivers into the level-major (L, 2, N) layout the
// kernels read (the reference does this with a strided `.contiguous()` copy,
// src/pytorch_modules/funcs.py:47).  Each workgroup moves kTransposeRows rows through LDS: the
// read is one contiguous chunk, every write a run of 64 consecutive floats.
// A thread issues the loads of kTogether values together, as many as it has up to eight: with one load per trip a workgroup
// waited a dozen times (2^20 rows of 48 columns 98.1 -> 78.7 us, a copy of the array takes 74; 100000 of 96 22.2 -> 13.7;
// 200001 of 48 16.9 -> 15.4; fewer for few columns, of which a thread has one value to every four: 2^20 rows of 12 19.9 with one,
// 18.0 with four, 25.8 with eight).
constexpr int kTransposeRows = 64;  // rows per workgroup: one wavefront-wide run per written column
constexpr int kTransposeManyColumns = 32;

template <int kTogether>
__global__ void __launch_bounds__(kBlock)
transpose_kernel(const float* __restrict__ src, int64_t src_row_stride, float* __restrict__ dst, int64_t rows, int cols) {
    extern __shared__ float tile[];  // kTransposeRows x (cols | 1)
    const int64_t row0 = static_cast<int64_t>(blockIdx.x) * kTransposeRows;
    const int n_rows = rows - row0 < kTransposeRows ? static_cast<int>(rows - row0) : kTransposeRows;
    const int stride = cols | 1;  // odd: a column read walks all banks
    const float* chunk = src + row0 * src_row_stride;
    const int n_values = n_rows * cols;
    int r = threadIdx.x / cols, c = threadIdx.x % cols;
    const int dr = kBlock / cols, dc = kBlock % cols;
    for (int i = threadIdx.x; i < n_values; i += kTogether * kBlock) {
        float v[kTogether];
        int at[kTogether];
#pragma unroll
        for (int u = 0; u < kTogether; ++u) {
            const bool in = i + u * kBlock < n_values;
            at[u] = in ? r * stride + c : -1;
            v[u] = chunk[in ? r * src_row_stride + c : 0];
            r += dr;
            c += dc;
            if (c >= cols) {
                c -= cols;
                ++r;
            }
        }
#pragma unroll
        for (int u = 0; u < kTogether; ++u)
            if (at[u] >= 0) tile[at[u]] = v[u];
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane < n_rows)
        for (int col = wave; col < cols; col += kBlock / 64) dst[static_cast<int64_t>(col) * rows + row0 + lane] = tile[lane * stride + col];
}

// The other direction: dst[r][c] = src[c][r], from the [level][feature][n] layout the forward writes to rows
// dst[n][F * level + feature] of `dst_row_stride` floats (what a layer that wants contiguous rows reads; the
// reference's permute + reshape, src/pytorch_modules/modules.py:87, leaves that copy to the consumer).  Every
// read is a run of 64 consecutive floats, the write one contiguous chunk when the rows are dense.
template <int kTogether>
__global__ void __launch_bounds__(kBlock)
transpose_to_rows_kernel(const float* __restrict__ src, float* __restrict__ dst, int64_t dst_row_stride, int64_t rows, int cols) {
    extern __shared__ float tile[];  // kTransposeRows x (cols | 1)
    const int64_t row0 = static_cast<int64_t>(blockIdx.x) * kTransposeRows;
    const int n_rows = rows - row0 < kTransposeRows ? static_cast<int>(rows - row0) : kTransposeRows;
    const int stride = cols | 1;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane < n_rows)
        for (int first = wave; first < cols; first += kTogether * (kBlock / 64)) {
            float v[kTogether];
#pragma unroll
            for (int u = 0; u < kTogether; ++u) {
                const int col = first + u * (kBlock / 64) < cols ? first + u * (kBlock / 64) : first;
                v[u] = __builtin_nontemporal_load(src + static_cast<int64_t>(col) * rows + row0 + lane);
            }
#pragma unroll
            for (int u = 0; u < kTogether; ++u)
                if (first + u * (kBlock / 64) < cols) tile[lane * stride + first + u * (kBlock / 64)] = v[u];
        }
    __syncthreads();
    float* chunk = dst + row0 * dst_row_stride;
    const int n_values = n_rows * cols;
    int r = threadIdx.x / cols, c = threadIdx.x % cols;
    const int dr = kBlock / cols, dc = kBlock % cols;
    for (int i = threadIdx.x; i < n_values; i += kBlock) {
        chunk[r * dst_row_stride + c] = tile[r * stride + c];
        r += dr;
        c += dc;
        if (c >= cols) {
            c -= cols;
            ++r;
        }
    }
}

// A few host values into device memory, carried by the launch itself (penc_upload).
constexpr int kUploadValues = 128;
struct UploadValues {
    float v[kUploadValues];
};
__global__ void __launch_bounds__(kUploadValues) upload_kernel(UploadValues values, int n, float* __restrict__ dst) {
    const int i = threadIdx.x;
    if (i < n) dst[i] = values.v[i];
}

// Clears two arrays (the second may be empty): n2 and m2 count 8-byte units.
__global__ void __launch_bounds__(kBlock) fill_zero_kernel(float2* __restrict__ p, size_t n2, float2* __restrict__ q, size_t m2) {
    const size_t stride = static_cast<size_t>(gridDim.x) * kBlock, first = static_cast<size_t>(blockIdx.x) * kBlock + threadIdx.x;
    for (size_t i = first; i < n2; i += stride) p[i] = make_float2(0.0f, 0.0f);
    for (size_t i = first; i < m2; i += stride) q[i] = make_float2(0.0f, 0.0f);
}

// ------------------------------------------------------------------------------------------
// Scratch of penc_backward_static: device memory that is part of the loaded code object, so that
// callers who must not allocate (HIP graph capture, serving loops) still get the binned scatter.
// Every GPU the library runs on holds its own copy until the process ends.  In host code the
// array's name is only a handle for hipGetSymbolAddress: its device address is looked up once per
// device (static_scratch_of) and that pointer is what the launchers pass on.
static __device__ __align__(256) unsigned char scratch[PENC_STATIC_SCRATCH_BYTES];

// ------------------------------------------------------------------------------------------
// host side

inline int check_launch() { return hipGetLastError() == hipSuccess ? PENC_OK : PENC_ERR_LAUNCH; }

inline uint32_t mask_of(int capacity) {
    const uint32_t c = static_cast<uint32_t>(capacity);
    return (c & (c - 1)) == 0 ? c - 1 : 0u;
}

inline int check_geometry(int pos_dim, int nr_feat, int64_t n, int levels, int capacity, int extra) {
    if (pos_dim < 2 || pos_dim > 8) return PENC_ERR_UNSUPPORTED_POS_DIM;
    if (nr_feat != 2 && nr_feat != 4 && nr_feat != 8) return PENC_ERR_UNSUPPORTED_NR_FEAT;
    if (n <= 0 || levels <= 0 || capacity <= 0) return PENC_ERR_BAD_SIZE;
    const int64_t lim = (int64_t{1} << 31) - 1;
    if (n > lim / (nr_feat * (int64_t{levels} + extra)) || n > lim / pos_dim) return PENC_ERR_BAD_SIZE;
    if (int64_t{capacity} > lim / (nr_feat * int64_t{levels})) return PENC_ERR_BAD_SIZE;
    if (levels + extra > 65535) return PENC_ERR_BAD_SIZE;
    return PENC_OK;
}

inline bool aligned8(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 7u) == 0; }
// The table as the gathering kernels see it: fp32 (format 0), or 16 bits per value (the *_half entry
// points: PENC_TABLE_FP16 or PENC_TABLE_BF16).
struct TableRef {
    const void* values;
    int format;
    bool cells = false;  // PENC_TABLE_CELLS (penc_cells.hpp)
};
inline int slots_per_line(int nr_feat, int format) { return kLineBytes / (nr_feat * (format != 0 ? 2 : 4)); }
inline bool cells_possible(int nr_feat, int capacity, int format) {
    return capacity >= slots_per_line(nr_feat, format) && (capacity & (capacity - 1)) == 0;
}
inline int strip_cells(int table_format) { return table_format & ~PENC_TABLE_CELLS; }
inline bool known_format(int table_format) {
    const int format = strip_cells(table_format);
    return table_format == 0 || format == PENC_TABLE_FP16 || format == PENC_TABLE_BF16;
}
inline bool known_half_format(int table_format) { return known_format(table_format) && strip_cells(table_format) != 0; }
// (nr_feat is checked by the caller's check_geometry: whatever it refuses is none of this function's)
inline bool cells_fit(int table_format, int nr_feat, int capacity) {
    return (table_format & PENC_TABLE_CELLS) == 0 || nr_feat < 2 || nr_feat > 8 || cells_possible(nr_feat, capacity, strip_cells(table_format));
}
inline TableRef table_ref(const void* values, int table_format) {
    return TableRef{values, strip_cells(table_format), (table_format & PENC_TABLE_CELLS) != 0};
}
// a slot is gathered with one load (two of 16 bytes for eight floats): 4 to 16 bytes
inline bool table_aligned(const TableRef& t, int nr_feat) {
    const unsigned slot_bytes = static_cast<unsigned>(nr_feat) * (t.format != 0 ? 2u : 4u);
    return (reinterpret_cast<uintptr_t>(t.values) & ((slot_bytes < 16u ? slot_bytes : 16u) - 1u)) == 0;
}

// Clears the table gradient, and the bins' `direct` flags when there are bins (`flags` of
// `flag_bytes`, a multiple of 8), with a fill kernel (float2 granularity: the gradient is only
// guaranteed 8-byte alignment).  A kernel rather than hipMemsetAsync so that callers may capture
// the call in a HIP graph.
inline int clear_table_grad(float* g, int pair_levels, int capacity, void* flags, size_t flag_bytes, hipStream_t st) {
    const size_t n2 = static_cast<size_t>(pair_levels) * capacity;
    const size_t want = (n2 + kBlock * 8 - 1) / (kBlock * 8);
    const unsigned blocks = static_cast<unsigned>(want < 8192 ? want : 8192);
    hipLaunchKernelGGL(fill_zero_kernel, dim3(blocks), dim3(kBlock), 0, st, reinterpret_cast<float2*>(g), n2,
                       static_cast<float2*>(flags), flags != nullptr ? flag_bytes / sizeof(float2) : size_t{0});
    return check_launch();
}

// How a workspace is cut into slot-range bins (see penc_scatter.hpp).  The levels are processed in
// passes of `levels_per_pass`; every pass reuses the same bins, so a smaller workspace means more,
// shorter passes (whose records are more likely still in cache when they are read back), not less
// binning.
struct BinPlan {
    bool enabled = false;
    int levels_per_pass = 0;
    BinTarget target{};       // of the first pass; target.direct covers all levels, a pass starts at its first level's flags
    ClearTarget clear{};      // (plan_deferred, plan_late)
    size_t direct_bytes = 0;  // size of target.direct (to be cleared with the gradient)
    uintptr_t end = 0;        // of what is used of the workspace
};

// Bytes of the `direct` flags of all levels (one 4-byte flag per level and bin), padded to the workspace's alignment.
inline size_t direct_flag_bytes(int levels, uint32_t n_bins) {
    return (static_cast<size_t>(levels) * n_bins * sizeof(uint32_t) + 255u) & ~size_t{255};
}

// log2 of the slots per bin: kBinSlotsLog2 (what a reducer workgroup's LDS holds) up to kMaxBins bins, wider
// bins (summed one LDS-full after the other) for larger tables, up to kMaxBinSlotsLog2.
constexpr uint32_t bin_shift_for_capacity(int capacity) {
    uint32_t shift = kBinSlotsLog2;
    while (shift < static_cast<uint32_t>(kMaxBinSlotsLog2) &&
           ((static_cast<int64_t>(capacity) + (int64_t{1} << shift) - 1) >> shift) > kMaxBins)
        ++shift;
    return shift;
}

constexpr uint32_t bins_of_shift(int capacity, uint32_t shift) {
    return static_cast<uint32_t>((static_cast<int64_t>(capacity) + (int64_t{1} << shift) - 1) >> shift);
}
// Bins per level; more than kMaxBins means the table is too large for binning.
constexpr uint32_t bins_for_capacity(int capacity) { return bins_of_shift(capacity, bin_shift_for_capacity(capacity)); }

// The width of the bins of a dense gradient whose workspace has room for the slack of more segments (penc_scatter_useful_bytes): where there are fewer
// (bin, level) pairs than reducers wanted, so that several would share a bin and add into the gradient with atomics (60 ns each), bins of half the width
// and less, down to 2^10 slots, until there are kFineBinsWanted pairs, each reduced by one workgroup of a part of a compute unit's LDS (a few where
// there are fewer pairs all the same, kFineBinsShared).  Scatter and
// reduction, us:
//   D = 3, 24 levels   2^16 slots, 2^20 points 517 -> 481   2^14 598 -> 488   2^12, 2^19 points 408 -> 270;  6 levels of 2^16, 2^20 points 145 -> 128
//          16 levels   2^18 points, 2^16 slots 105 -> 98   2^14 131 -> 101   100003 slots 108 -> 98;  12 levels of 2^18, 2^19 points 134 -> 125
//   D = 2, 16 levels   2^16 slots, 2^18 points 83 -> 73, four features 125 -> 117;  2^17, 2^19 points 124 -> 123
//   D = 5, 16 levels   2^16 slots, 2^18 points 177 -> 160;  D = 6 of 2^14 217 -> 204;  D = 8 of 2^16 255 -> 250, 8 levels of 2^18, 2^17 points 97 -> 91
// With four dimensions the accumulate cache leaves some slots of the coarse levels out, whose records several reducers of a bin share
// better than one (16 levels, 2^18 points: 2^16 slots 130 -> 137, 2^17 126 -> 132; 2^15 131 -> 122).
// A table that is one bin has room there for everything a group leaves; of narrower ones one can run over, where points that hardly share slots
// crowd a range of them, and what finds no room is added to the gradient in fp32 one by one, as it is for any table of several bins that is not written whole, instead of in
// the reducer's sums in fp64.
constexpr uint32_t kReduceWorkgroupsWanted = 512;  // two per compute unit
constexpr uint32_t kFineBinsWanted = 768, kFineBinsMostPairs4d = 128;
constexpr uint32_t fine_bin_shift(int pos_dim, int capacity, int pair_levels) {
    uint32_t shift = bin_shift_for_capacity(capacity);
    const uint32_t levels = static_cast<uint32_t>(pair_levels), pairs = bins_of_shift(capacity, shift) * levels;
    if (shift != static_cast<uint32_t>(kBinSlotsLog2) || pairs >= (pos_dim == 4 ? kFineBinsMostPairs4d : kReduceWorkgroupsWanted)) return shift;
    while (shift > static_cast<uint32_t>(kFinestBinSlotsLog2) && bins_of_shift(capacity, shift) * levels < kFineBinsWanted &&
           bins_of_shift(capacity, shift - 1) <= static_cast<uint32_t>(kStageBins))
        --shift;
    return shift;
}
// A width is doubled only where it leaves more than kMaxBins bins, so wide bins are always more than half as many: their scatter is
// that of many bins.
static_assert(kMaxBins / 2 >= static_cast<int>(kFewerOpenLinesMinBins) && kFewerOpenLinesMinBins >= static_cast<uint32_t>(kStageBins),
              "wide bins are many bins, and many bins are sorted by stream_tile_many");
static_assert(bin_shift_for_capacity((kMaxBins << kBinSlotsLog2) + 1) > static_cast<uint32_t>(kBinSlotsLog2) &&
                  bins_for_capacity((kMaxBins << kBinSlotsLog2) + 1) > kFewerOpenLinesMinBins,
              "the smallest table with wide bins");

constexpr int64_t kMinSlotsPerContribution = 8;
constexpr int64_t kLargeGroupsMinWorkgroups = 3000;  // about four per workgroup slot of the chip (256 CUs x 3)

inline unsigned scatter_groups(int64_t n, int tiles_per_group) {
    const int64_t group_points = static_cast<int64_t>(tiles_per_group) * kScatterBlock;
    return static_cast<unsigned>((n + group_points - 1) / group_points);
}

// Tiles per scattering workgroup of the table backward.  Larger groups mean longer record segments
// (less slack, longer bursts for the reducer) and fewer cache flushes; they are taken when the
// launch still has several workgroups for every slot of the chip (measured: 3-13% faster then,
// slower otherwise).  The same rule serves the scattering half of the double backward.
// Small batches take smaller groups, down to two tiles, until the launch has a workgroup for every slot of
// the chip (measured at 24 levels, D = 3: 2^16 points 0.074 -> 0.064 ms with four tiles, 2^15 points
// 0.065 -> 0.055 ms and 2^14 points 0.062 -> 0.048 ms with two; 2^17 points are best with eight).  That is for the
// small batches that the sorted groups below do not take: few levels, sparse or mostly empty gradients, a workspace too small.
constexpr int64_t kMinWorkgroups = 768;  // three per compute unit
// Rows of an upstream gradient are read by every level of a group, and what a die holds of them at a time should fit its L2: 96
// workgroups (three to a compute unit, up to four dimensions) of 16 tiles read 6 MB of rows, however many levels those rows have.  With
// eight tiles the longer segments are missed less than the rows.  Forward and backward of the module from rows, us, 16 -> 8 tiles, all at sizes
// that take 16 otherwise (about 25 M points times levels):
//   D = 3, 24 levels       2^17 slots 789 -> 764   2^18 790 -> 778   2^19 926 -> 913;  2^16 slots (8 bins, shared by reducers) 742 -> 739
//          16 levels       2^17 826 -> 813   2^18 1072 -> 1069   2^19 915 -> 908;  2^16 slots 892 -> 907, 20 levels 1166 -> 1176
//          few levels, which keep in step anyway   12 of 2^18 772 -> 768   10 780 -> 779;  8 1033 -> 1038   6 780 -> 788
//   D = 4, 24 levels       2^18 1036 -> 1025   2^19 1292 -> 1288;  2^17 926 -> 929, 16 levels 1072 -> 1088, of 2^16 1238 -> 1248
//          10 levels       2^18 1018 -> 1007;  8 1292 -> 1309
// Not from five dimensions on, where two workgroups to a compute unit read 4 MB (D = 5, 24 levels 1294 -> 1318, 32 levels 1690 -> 1736; D = 7, 16
// levels 2384 -> 2412; D = 8 1985 -> 1981), with two dimensions (scatter and reduction 230 -> 236), four features (317 -> 320), whose rows
// more than one pair of features reads, or more than kStageBins bins, whose runs are short as it is (2^22 slots 1212 -> 1290).  A spectrum of
// scales without fine levels, which the launch does not know of, has few records to gain or lose by (24 levels down to 1e-2: 552 -> 563).
constexpr int kShortGroupsMinLevels = 10;
inline bool short_groups(int pos_dim, uint32_t feat_pairs, int levels, int capacity, bool rows) {
    const uint32_t bins = bins_for_capacity(capacity);
    return rows && (pos_dim == 3 || pos_dim == 4) && feat_pairs == 1u && levels >= kShortGroupsMinLevels &&
           bins >= (pos_dim == 3 ? 16u : 32u) && bins <= static_cast<uint32_t>(kStageBins);
}
inline int table_backward_tiles(int64_t n, int levels) {
    if (static_cast<int64_t>(scatter_groups(n, kScatterTilesLarge)) * levels >= kLargeGroupsMinWorkgroups) return kScatterTilesLarge;
    int tiles = kScatterTiles;
    while (tiles > 2 && static_cast<int64_t>(scatter_groups(n, tiles)) * levels < kMinWorkgroups) tiles /= 2;
    return tiles;
}

// Split records (10 bytes in two arrays) where a tile's records leave in long runs (the
// workgroup-wide sort), whole ones (12 bytes) elsewhere (see BinRecord).
inline size_t record_bytes(int pos_dim, uint32_t n_bins) {
    return pos_dim <= kWorkgroupSortMaxDim && n_bins <= static_cast<uint32_t>(kStageBins) ? kSplitRecordBytes : sizeof(BinRecord);
}

// Records one scattering workgroup may leave in one bin: its share of the
// group's contributions (D+1 per point) plus the flushed cache lines, with three standard deviations
// of a uniform hash on top.  A segment that still overflows spills to direct atomics.
inline uint32_t wanted_segment_capacity(int pos_dim, uint32_t n_bins, int tiles_per_group) {
    const double mean = (static_cast<double>(tiles_per_group) * kScatterBlock * (pos_dim + 1) + kCacheLines) / n_bins;
    const uint32_t cap = static_cast<uint32_t>(mean + 3.0 * __builtin_sqrt(mean) + 8.0);
    // split records: a multiple of four per segment keeps every segment's values 16-byte aligned
    return record_bytes(pos_dim, n_bins) == kSplitRecordBytes ? (cap + 3u) & ~3u : cap;
}

inline size_t bin_bytes_per_level(int pos_dim, uint32_t n_bins, uint32_t n_groups, uint32_t segment_capacity) {
    const size_t segments = static_cast<size_t>(n_bins) * n_groups;
    return segments * (sizeof(uint32_t) + static_cast<size_t>(segment_capacity) * record_bytes(pos_dim, n_bins));
}

inline BinPlan plan_bins(int pos_dim, int64_t n, int levels, int capacity, uint32_t bin_shift, int tiles_per_group, void* workspace,
                         size_t bytes) {
    BinPlan p;
    const uint32_t n_bins = bins_of_shift(capacity, bin_shift);
    const uint32_t n_groups = scatter_groups(n, tiles_per_group);
    if (workspace == nullptr || n_bins > static_cast<uint32_t>(kMaxBins)) return p;
    // few contributions per slot: the reducer's fixed cost per bin (clearing and flushing 128 KiB of
    // LDS) exceeds what direct atomics cost (measured crossover: one contribution per eight slots)
    if (n * (pos_dim + 1) * kMinSlotsPerContribution <= capacity) return p;
    const uintptr_t base = (reinterpret_cast<uintptr_t>(workspace) + 255u) & ~uintptr_t{255};
    const size_t lost = base - reinterpret_cast<uintptr_t>(workspace);
    const size_t flag_bytes = direct_flag_bytes(levels, n_bins);
    if (bytes < lost + flag_bytes + 4096) return p;
    bytes -= lost + flag_bytes + 256;
    const size_t segments = static_cast<size_t>(n_bins) * n_groups;
    const bool split = record_bytes(pos_dim, n_bins) == kSplitRecordBytes;
    uint32_t cap = wanted_segment_capacity(pos_dim, n_bins, tiles_per_group);
    if (bytes < bin_bytes_per_level(pos_dim, n_bins, n_groups, cap)) {  // not even one level at the wanted size: shrink the segments
        if (bytes < segments * (sizeof(uint32_t) + 16 * record_bytes(pos_dim, n_bins))) return p;
        cap = static_cast<uint32_t>((bytes / segments - sizeof(uint32_t)) / record_bytes(pos_dim, n_bins));
        if (split) cap &= ~3u;
    }
    // the scattering kernel addresses a level's records with 32-bit byte offsets
    const uint64_t max_records_per_level = 0xFFFFFFFFull / (split ? sizeof(RecordValues) : sizeof(BinRecord));
    if (segments * cap > max_records_per_level) {
        cap = static_cast<uint32_t>(max_records_per_level / segments);
        if (split) cap &= ~3u;
        if (cap < 16) return p;
    }
    const size_t fit = bytes / bin_bytes_per_level(pos_dim, n_bins, n_groups, cap);
    p.levels_per_pass = static_cast<int>(fit < static_cast<size_t>(levels) ? fit : static_cast<size_t>(levels));
    // wide bins are served by bin_reduce_levels_kernel only
    if (bin_shift > static_cast<uint32_t>(kBinSlotsLog2) &&
        (cap > kLevelsMaxSegment || n_groups > static_cast<uint32_t>(kReduceBlock)))
        return p;
    p.target.n_bins = n_bins;
    p.target.n_groups = n_groups;
    p.target.segment_capacity = cap;
    p.target.bin_shift = bin_shift;
    p.target.direct = reinterpret_cast<uint32_t*>(base);
    p.direct_bytes = flag_bytes;
    const uintptr_t counts_at = base + flag_bytes;
    p.target.counts = reinterpret_cast<uint32_t*>(counts_at);
    const size_t counts_bytes = (static_cast<size_t>(p.levels_per_pass) * segments * sizeof(uint32_t) + 255u) & ~size_t{255};
    const size_t records_per_pass = static_cast<size_t>(p.levels_per_pass) * segments * cap;
    p.target.records = reinterpret_cast<void*>(counts_at + counts_bytes);
    p.target.slots = split ? reinterpret_cast<uint16_t*>(counts_at + counts_bytes + records_per_pass * sizeof(RecordValues)) : nullptr;
    p.end = counts_at + counts_bytes + records_per_pass * record_bytes(pos_dim, n_bins);
    p.enabled = true;
    return p;
}

// Fill, scatter, reduction and late adds, us, fill apart -> in the scatter (24 levels unless given; more beside ClearTarget):
//   D = 3, 2^22 slots  2^20 points 1081 -> 1012, near a surface with 16 levels live 600 -> 530;  2^23 slots, 2^19 points 1039 -> 984
//          2^20        2^20 points from rows 652 -> 650;  16 levels 424 -> 425
//   D = 2, 16 levels of 2^20, 2^18 points 133 -> 121;  D = 4, 16 levels of 2^20, 2^18 points 186 -> 173;  D = 8, of 2^22, 2^17 points 465 -> 360
// A smaller gradient takes no longer to fill than the lists take to be added (few bins: written_whole).  With workgroups of 512
// threads, not for less than one round of them, which the clearing ones put off (D = 8, 2^20 slots: 480 workgroups 80 -> 85, 89 -> 93, 111 -> 121;  588
// of them 95 -> 89, 600 120 -> 107).
constexpr size_t kClearInScatterBytes = size_t{64} << 20;
constexpr int64_t kClearMinWorkgroups = 512;  // two to a compute unit
inline bool clears_in_scatter(uint32_t n_bins, int pair_levels, int capacity, int64_t workgroups) {
    return n_bins > static_cast<uint32_t>(kStageBins) && static_cast<size_t>(pair_levels) * capacity * sizeof(float2) >= kClearInScatterBytes &&
           (n_bins > kFewerOpenLinesMinBins || workgroups >= kClearMinWorkgroups);
}
// Threads to a die that clear and do nothing else, and up to how many points times levels.  Beyond, a share each -> rows apart, 2^20 points, us: 2^22 slots 1014 ->
// 987, along rays 900 -> 890, 1e-3 774 -> 763, 1e-2 597 -> 623, near a surface with 16 levels live 530 -> 543;  2^21 830 -> 804, along rays, 1e-2, 463 ->
// 478;  2^20 650 -> 639, 388 -> 400, 16 levels 426 -> 430.
constexpr uint32_t kClearingThreads = 4096;
constexpr int64_t kClearApartMaxWork = 16000000;
// What the lists of deferred adds (ClearTarget) take behind the bins, for all levels at once.
inline size_t deferred_bytes(int pos_dim, int pair_levels, uint32_t n_groups, int tiles_per_group) {
    return static_cast<size_t>(pair_levels) * n_groups * (deferred_room(pos_dim, tiles_per_group) * sizeof(BinRecord) + sizeof(uint32_t)) + 512;
}
inline bool place_lists(BinPlan& p, int pos_dim, int pair_levels, int tiles_per_group, const void* workspace, size_t bytes) {
    const uintptr_t base = (p.end + 255u) & ~uintptr_t{255};
    if (base + deferred_bytes(pos_dim, pair_levels, p.target.n_groups, tiles_per_group) > reinterpret_cast<uintptr_t>(workspace) + bytes) return false;
    p.clear.room = deferred_room(pos_dim, tiles_per_group);
    p.clear.kept = reinterpret_cast<BinRecord*>(base);
    p.clear.counts = reinterpret_cast<uint32_t*>(base + static_cast<size_t>(pair_levels) * p.target.n_groups * p.clear.room * sizeof(BinRecord));
    return true;
}
// Gives the plan of a dense gradient such lists where its scatter has the instance that clears, takes all levels in one launch, and the workspace has room
// for them.
inline bool plan_deferred(BinPlan& p, int pos_dim, int64_t nr_positions, int pair_levels, int capacity, int tiles_per_group, const float* table_grad, const void* workspace,
                          size_t bytes) {
    if (!p.enabled || !clears_in_scatter(p.target.n_bins, pair_levels, capacity, static_cast<int64_t>(p.target.n_groups) * pair_levels) || p.levels_per_pass < pair_levels) return false;
    if ((reinterpret_cast<uintptr_t>(table_grad) & 15u) != 0 || !place_lists(p, pos_dim, pair_levels, tiles_per_group, workspace, bytes)) return false;
    p.clear.pairs = static_cast<uint64_t>(pair_levels) * capacity;
    p.clear.flags = static_cast<uint32_t>(p.direct_bytes / sizeof(uint32_t));
    const uint32_t threads = p.target.n_bins > kFewerOpenLinesMinBins ? kScatterBlockManyBins : kScatterBlock;
    p.clear.rows = nr_positions * pair_levels < kClearApartMaxWork ? kClearingThreads / threads : 0u;
    return true;
}

// When a table gradient takes the sorted groups of penc_group_sort.hpp, and how they cut its workspace.
//
// Up to 2^22 looked-up slots (points x vertices x levels), 6 x 2^20 at three and four dimensions: there the scatter, its fill and its
// reduction are latency, beyond it the records of the coarse levels, which the scatter absorbs, cost more (us, scatter ->
// sorted groups; L = 16 unless given):
//   D = 3, L = 24, 2^18 slots  500 points 23.2 -> 19.9, 2^14 points 51.0 -> 36.8, 2^15 56.9 -> 44.8 (3.1 M slots), 2^16 67.0 -> 61.4 (6.3 M),
//                              along rays 69.8 -> 56.9, 125000 points 98 -> 95, 250000 points 141 -> 185
//   D = 3, 2^16 slots          2^12 points 29.6 -> 16.9, 2^16 points 70.5 -> 49.9 (4.2 M)
//   D = 4, L = 24, 2^18 slots  34000 points 69.1 -> 53.9, 50000 points 77.8 -> 64.0 (6 M), 92000 points 102 -> 107
//   D = 5, 2^18 slots          31250 points 58.7 -> 43.8 (3 M), 42700 points 63.8 -> 62.0, 52000 points 74.3 -> 79.8 (5 M)
//   D = 8, 2^18 slots          2000 points 40.1 -> 22.6, 2^15 points 71.1 -> 66.6 (4.7 M), 2^16 points 101 -> 137
//   D = 2, F = 4, 2^16 slots   2^12 points 34.5 -> 19.5;  D = 4, F = 8, 2^18 slots  2^16 points 171 -> 142 (5.2 M), 2^17 points 259 -> 272
// And up to 4096 points to a level and pair of features: a level's records are summed by as many workgroups as it has ranges,
// and with many points on few levels those with a coarse level's slots end last (six levels of 2^12 slots, D = 2, 83000
// points 26.7 -> 32.9, 228000 points 44.8 -> 71.6; of 2^18 slots, D = 3, 62500 points 36.4 -> 42.3; eight of 2^14, D = 5, 31000 points
// 52.5 -> 36.9, 85000 points 65.5 -> 93.4).
// Writing every slot once is what a dense gradient costs either way; a batch that leaves most of a large table empty is better served
// by a fill and a few direct adds (24 levels: 2^20 slots, 500 points 43 -> 47, 2^12 points 55 -> 57; 2^22 slots, 2^12 points 211 -> 232,
// 2^14 points 290 -> 261).  Sparse gradients have no fill to save and pay for every range that got one record: 2^20
// slots, 2^12 points 55 -> 88, 2^14 points 126 -> 101; 2^18 slots, 2000 points 29 -> 36, 2^15 points 56 -> 54.5.
constexpr int64_t group_sort_max_lookups(int pos_dim) { return pos_dim == 3 || pos_dim == 4 ? int64_t{6} << 20 : int64_t{4} << 20; }
constexpr int64_t kGroupSortPointsPerLevel = 4096, kGroupSortSlotsPerLookup = 64, kGroupSortSparseSlotsPerLookup = 16;
constexpr uint32_t kRangeSlotsLog2 = 12, kRangeMinSlotsLog2 = 9, kRangeWorkgroupsWanted = 512, kRangeManyGroups = 32;
constexpr size_t kGroupSortAnyFillBytes = size_t{64} << 20;
inline bool group_sort_serves(int pos_dim, int64_t n, int levels, int feat_pairs, int capacity, bool sparse) {
    const int64_t lookups = n * (pos_dim + 1);
    if (lookups * levels > group_sort_max_lookups(pos_dim) || n > kGroupSortPointsPerLevel * levels * feat_pairs || capacity > (kGroupMaxRanges << kBinSlotsLog2)) return false;
    if (sparse) return capacity <= kGroupSortSparseSlotsPerLookup * lookups;
    return static_cast<size_t>(capacity) * levels * feat_pairs * sizeof(float2) <= kGroupSortAnyFillBytes || capacity <= kGroupSortSlotsPerLookup * lookups;
}
struct GroupSortPlan {
    bool enabled = false;
    GroupSort sort{};
};
// Bytes of the arrays for `pair_levels` pairs of features (for levels of several pairs a little more than they need).
inline size_t group_sort_bytes(int pos_dim, int64_t n, int pair_levels) {
    const size_t groups = static_cast<size_t>((n + kGroupPoints - 1) / kGroupPoints), records = static_cast<size_t>(pos_dim + 1) * kGroupPoints;
    return static_cast<size_t>(pair_levels) * groups * (records * (sizeof(RecordValues) + sizeof(uint16_t)) + (kGroupMaxRanges + 2) * sizeof(uint16_t)) + 1024;
}
inline GroupSortPlan plan_group_sort(int pos_dim, int64_t n, int levels, int feat_pairs, int capacity, bool sparse, void* workspace,
                                     size_t bytes) {
    GroupSortPlan p;
    const int pair_levels = levels * feat_pairs;
    if (workspace == nullptr || !group_sort_serves(pos_dim, n, levels, feat_pairs, capacity, sparse)) return p;
    const uintptr_t base = (reinterpret_cast<uintptr_t>(workspace) + 255u) & ~uintptr_t{255};
    if (bytes < group_sort_bytes(pos_dim, n, pair_levels) + (base - reinterpret_cast<uintptr_t>(workspace))) return p;
    GroupSort& g = p.sort;
    g.n_groups = static_cast<uint32_t>((n + kGroupPoints - 1) / kGroupPoints);
    g.records = static_cast<uint32_t>((pos_dim + 1) * kGroupPoints);
    // ranges of 4096 slots (two workgroups per compute unit, and all of a wave's stores to one stretch), narrower ones where they
    // leave compute units idle: two workgroups per unit, four where every workgroup sums many groups (D = 4, 16 levels of
    // 2^16 slots, 2^15 points: 64.7 -> 53.4 us; D = 3, 2^12 points: 19.2 with four, 16.8 with two)
    const uint32_t wanted = g.n_groups >= kRangeManyGroups ? 2 * kRangeWorkgroupsWanted : kRangeWorkgroupsWanted;
    const auto ranges = [&](uint32_t shift) { return static_cast<uint32_t>((static_cast<int64_t>(capacity) + (int64_t{1} << shift) - 1) >> shift); };
    g.range_shift = kRangeSlotsLog2;
    while (ranges(g.range_shift) > static_cast<uint32_t>(kGroupMaxRanges)) ++g.range_shift;  // at most kBinSlotsLog2: see group_sort_serves
    while (g.range_shift > kRangeMinSlotsLog2 && ranges(g.range_shift) * static_cast<uint32_t>(pair_levels) < wanted &&
           ranges(g.range_shift - 1) <= static_cast<uint32_t>(kGroupMaxRanges))
        --g.range_shift;
    g.n_ranges = ranges(g.range_shift);
    const size_t all = static_cast<size_t>(g.n_groups) * g.records;
    g.values = reinterpret_cast<RecordValues*>(base);
    g.slots = reinterpret_cast<uint16_t*>(base + static_cast<size_t>(pair_levels) * all * sizeof(RecordValues));
    g.starts = g.slots + static_cast<size_t>(levels) * all;
    p.enabled = true;
    return p;
}

// Running consecutive passes on two streams (scatter pass p+1 while pass p is reduced) was tried and
// measured 10-15% slower than one pass over all levels on one stream; hence a single stream.
// Narrow bins, which end sooner, are shared up to one pair of bin and level to a compute unit, and up to kFineBinsSharedCrowded pairs where a slot of at most 2^11
// has eight contributions and more.  Scatter and reduction, alone -> shared (as wide bins), 2^19 points, us:
//   128 pairs  D = 3, 16 levels of 2^13 slots 235 -> 182 (246), along rays 246 -> 195 (237)   D = 8, 8 levels of 2^14 295 -> 245 (253), 364 -> 290 (292)
//   192        D = 2, 24 of 2^13 198 -> 160 (208), 217 -> 172 (200);  D = 4, 6 of 2^15 96 -> 88 (109), 111 -> 93 (103);  D = 3, 24 of 2^13 282 -> 247 (402)
//   384        D = 3, 12 of 2^15 125 -> 126 (159), 140 -> 130 (144);  6 of 2^17, four contributions to a slot 35.1 -> 36.8 (48)
//              bins of 2^12: D = 5, 6 of 2^18 141 -> 147 (151), along rays 148 -> 146 (145)
constexpr unsigned kFineBinsShared = 256, kFineBinsSharedCrowded = 448;
constexpr unsigned kMaxReduceSplits = 16;

// How many workgroups share a bin: enough for every compute unit.
inline unsigned reduce_splits(uint32_t n_bins, uint32_t bin_shift, uint32_t n_groups, int64_t lookups, int n_levels_in_pass) {
    const unsigned pairs = n_bins * static_cast<unsigned>(n_levels_in_pass);
    unsigned enough = kReduceWorkgroupsWanted;
    if (bin_shift < static_cast<uint32_t>(kBinSlotsLog2)) {
        const bool crowded = bin_shift <= 11u && lookups >= static_cast<int64_t>(n_bins) << (bin_shift + 3);
        enough = (crowded ? kFineBinsSharedCrowded : kFineBinsShared) + 1;
    }
    unsigned splits = pairs >= enough ? 1u : (kReduceWorkgroupsWanted + pairs - 1) / pairs;
    if (splits > n_groups) splits = n_groups;
    return splits > kMaxReduceSplits ? kMaxReduceSplits : splits;
}

inline bool few_bins_alone(uint32_t n_bins, uint32_t bin_shift, uint32_t n_groups, int64_t lookups, int pair_levels) {
    return n_bins <= static_cast<uint32_t>(kStageBins) && reduce_splits(n_bins, bin_shift, n_groups, lookups, pair_levels) == 1u;
}
// The gradient of a table of few bins is written whole by its reducers (LateTarget) where each has a bin to itself, all levels are one pass and the bins have kBinSlots slots.
// Fill, scatter and reduction, us: 24 levels of 2^18 slots, D = 3, 2^20 points 8 + 320 + 125 -> 317 + 124, 2^18 points 8 + 89 + 40 -> 89 + 40, 131007 points along rays
// 9 + 50 + 14.8 -> 51.5 + 20.3;  D = 8, 16 levels of 2^19, 2^19 points 11 + 289 + 131 -> 290 + 132.
// Narrow bins have little to fill, and short segments, which run over where few slots are hot; what does goes into the gradient one by one while the scatter does other things, but as late
// adds it waits in the one reducer of the hot bin: D = 8, 16 levels of 2^16 slots down to 1e-2, 2^18 points near a surface 5 + 193 + 39 -> 179 + 115, 12 levels
// 5 + 146 + 42 -> 147 + 118;  D = 2, 16 levels of 2^16 5 + 57 + 9 -> 64 + 14;  otherwise a pass is up to 4% shorter written whole, 0.6% on average over 330 geometries.
// More than two pairs of features write every slot in parts, 8 bytes of 64 at a time (forward and table gradient, 16 levels of 2^18 slots, 131072 points along rays, the window on 0.4
// of them: D = 3, eight features 103 -> 125, four 77 -> 77; all levels 239 -> 246, four 133 -> 128).
// With two dimensions a level's hashes fill the bins unevenly, and a full one's reducer is what the launch waits for (24 levels of 2^18 slots: 2^20 points 9 + 279 + 80 -> 271 + 144,
// 2^18 points 8 + 69 + 29 -> 68 + 35;  18 levels, 2^19 points 7 + 100 + 35 -> 98 + 53, 2^17 points 8 + 36 + 16 -> 37 + 19).
constexpr int64_t kWholeMaxPoints2d = 1 << 18;
inline bool written_whole(int pos_dim, uint32_t feat_pairs, int64_t nr_positions, uint32_t n_bins, uint32_t bin_shift, uint32_t n_groups, int pair_levels) {
    return bin_shift == static_cast<uint32_t>(kBinSlotsLog2) && feat_pairs <= 2u && (pos_dim > 2 || nr_positions <= kWholeMaxPoints2d) &&
           few_bins_alone(n_bins, bin_shift, n_groups, nr_positions * (pos_dim + 1), pair_levels);
}
inline bool plan_late(BinPlan& p, int pos_dim, uint32_t feat_pairs, int64_t nr_positions, int pair_levels, int tiles_per_group, const void* workspace, size_t bytes) {
    if (!p.enabled || p.levels_per_pass < pair_levels ||
        !written_whole(pos_dim, feat_pairs, nr_positions, p.target.n_bins, p.target.bin_shift, p.target.n_groups, pair_levels))
        return false;
    return place_lists(p, pos_dim, pair_levels, tiles_per_group, workspace, bytes);
}

inline int reduce_bins(const BinPlan& p, int64_t lookups, const float* window, int first_level, int n_levels_in_pass, int capacity,
                       uint32_t feat_pairs, float* table_grad, hipStream_t st) {
    const unsigned splits = reduce_splits(p.target.n_bins, p.target.bin_shift, p.target.n_groups, lookups, n_levels_in_pass);
    // many bins with a few thousand records each: workgroups that keep their bin and walk several levels
    // (bins wider than kBinSlots are planned only where this kernel can serve them)
    const bool wide = p.target.bin_shift > static_cast<uint32_t>(kBinSlotsLog2);
    if (wide || (p.target.slots == nullptr && p.target.n_bins > static_cast<uint32_t>(kStageBins) && splits == 1 &&
                 p.target.segment_capacity <= kLevelsMaxSegment && p.target.n_groups <= static_cast<uint32_t>(kReduceBlock))) {
        const unsigned levels = static_cast<unsigned>(n_levels_in_pass);
        unsigned per_bin = (levels + kLevelsMaxPerWorkgroup - 1) / kLevelsMaxPerWorkgroup;
        const unsigned to_fill = (kReduceWorkgroupsWanted + p.target.n_bins - 1) / p.target.n_bins;  // two workgroups per compute unit, one after the other
        if (per_bin < to_fill) per_bin = to_fill;
        if (per_bin > levels) per_bin = levels;
#define PENC_LAUNCH_LEVELS(UNROLL)                                                                                                          \
    hipLaunchKernelGGL(bin_reduce_levels_kernel<UNROLL>, dim3(p.target.n_bins, per_bin), dim3(kReduceBlock), 0, st, p.target, window,       \
                       static_cast<uint32_t>(capacity), feat_pairs, table_grad, first_level, static_cast<uint32_t>(levels))
        if (p.target.segment_capacity <= kLevelsShortSegment) PENC_LAUNCH_LEVELS(kLevelsShortUnroll);
        else PENC_LAUNCH_LEVELS(kLevelsUnroll);
#undef PENC_LAUNCH_LEVELS
        return check_launch();
    }
    const dim3 grid(p.target.n_bins, n_levels_in_pass, splits);
    const LateTarget late = p.target.n_bins <= static_cast<uint32_t>(kStageBins) ? LateTarget(p.clear) : LateTarget{};
#define PENC_LAUNCH_REDUCE(SPLIT, SLOTS_LOG2)                                                                                                       \
    case SLOTS_LOG2:                                                                                                                                \
        hipLaunchKernelGGL((bin_reduce_kernel<SPLIT, SLOTS_LOG2>), grid, dim3(reduce_threads(SLOTS_LOG2)), 0, st, p.target, window,                 \
                           static_cast<uint32_t>(capacity), feat_pairs, table_grad, first_level, late);                                            \
        break;
#define PENC_LAUNCH_REDUCE_ALL(SPLIT)                                                                                                               \
    switch (p.target.bin_shift) {                                                                                                                   \
        PENC_LAUNCH_REDUCE(SPLIT, 10) PENC_LAUNCH_REDUCE(SPLIT, 11) PENC_LAUNCH_REDUCE(SPLIT, 12) PENC_LAUNCH_REDUCE(SPLIT, 13)                     \
    }
    static_assert(kFinestBinSlotsLog2 == 10 && kBinSlotsLog2 == 13, "an instance for every width");
    if (p.target.slots != nullptr) {
        PENC_LAUNCH_REDUCE_ALL(true)
    } else {
        PENC_LAUNCH_REDUCE_ALL(false)
    }
#undef PENC_LAUNCH_REDUCE_ALL
#undef PENC_LAUNCH_REDUCE
    return check_launch();
}

#define PENC_DISPATCH_D(D_, ...)                                  \
    switch (D_) {                                                  \
        case 2: { constexpr int DD = 2; __VA_ARGS__; } break;      \
        case 3: { constexpr int DD = 3; __VA_ARGS__; } break;      \
        case 4: { constexpr int DD = 4; __VA_ARGS__; } break;      \
        case 5: { constexpr int DD = 5; __VA_ARGS__; } break;      \
        case 6: { constexpr int DD = 6; __VA_ARGS__; } break;      \
        case 7: { constexpr int DD = 7; __VA_ARGS__; } break;      \
        case 8: { constexpr int DD = 8; __VA_ARGS__; } break;      \
        default: return PENC_ERR_UNSUPPORTED_POS_DIM;              \
    }

// The same with the number of features per level (2, 4 or 8) as the constant FF.
#define PENC_DISPATCH_DF(D_, F_, ...)                                   \
    if ((F_) == 8) {                                                    \
        constexpr int FF = 8;                                           \
        PENC_DISPATCH_D(D_, __VA_ARGS__)                                \
    } else if ((F_) == 4) {                                             \
        constexpr int FF = 4;                                           \
        PENC_DISPATCH_D(D_, __VA_ARGS__)                                \
    } else {                                                            \
        constexpr int FF = 2;                                           \
        PENC_DISPATCH_D(D_, __VA_ARGS__)                                \
    }

// The same with the table's element type (float, __half or bfloat16_bits) as TT.
#define PENC_DISPATCH_DFT(D_, F_, FORMAT_, ...)                         \
    if ((FORMAT_) == PENC_TABLE_BF16) {                                 \
        using TT = bfloat16_bits;                                       \
        PENC_DISPATCH_DF(D_, F_, __VA_ARGS__)                           \
    } else if ((FORMAT_) == PENC_TABLE_FP16) {                          \
        using TT = __half;                                              \
        PENC_DISPATCH_DF(D_, F_, __VA_ARGS__)                           \
    } else {                                                            \
        using TT = float;                                               \
        PENC_DISPATCH_DF(D_, F_, __VA_ARGS__)                           \
    }

inline unsigned tiles(int64_t n) { return static_cast<unsigned>((n + kBlock - 1) / kBlock); }

// Device address of this GPU's copy of `scratch`, looked up on the first call with that GPU
// current and kept for the life of the process.  Returns nullptr when the lookup fails.
constexpr int kMaxDevices = 64;
inline void* static_scratch_of_current_device() {
    static std::mutex lock;
    static void* address[kMaxDevices] = {};
    int device = -1;
    if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= kMaxDevices) return nullptr;
    std::lock_guard<std::mutex> guard(lock);
    if (address[device] == nullptr) {
        void* p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess) {
            (void)hipGetLastError();  // the failure is reported by the caller's status code, not by a later launch check
            return nullptr;
        }
        address[device] = p;
    }
    return address[device];
}

// Accelerator dies of the current GPU (each with an L2 of its own; workgroup i of a launch runs on
// die i % dies), asked of the runtime once per device.  kDefaultDies when the runtime does not say.
inline uint32_t dies_of_current_device() {
    static std::mutex lock;
    static uint32_t dies[kMaxDevices] = {};
    int device = -1;
    if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= kMaxDevices) return kDefaultDies;
    std::lock_guard<std::mutex> guard(lock);
    if (dies[device] == 0u) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeNumberOfXccs, device) != hipSuccess) {
            (void)hipGetLastError();
            n = 0;
        }
        dies[device] = n >= 1 && n <= 64 ? static_cast<uint32_t>(n) : kDefaultDies;
    }
    return dies[device];
}

// Levels a thread of the forward and of the gathering half of the double backward takes: two up to
// pos_dim 4 (measured on the forward at 2^20 points, 24 levels: 0.310 -> 0.302 ms at pos_dim 3, 0.275 -> 0.259 ms with a
// 2^22-slot table, 0.396 -> 0.392 ms at pos_dim 4; at pos_dim 8 0.283 -> 0.298 ms) and once the launch fills the chip twice
// over with pairs (eight workgroups of four wavefronts per compute unit; 2^15 points: 12.6 us with single levels, 15.9 with
// pairs, 2^16 23.4 and 24.8, 131 k 31.4 and 30.5).
constexpr int64_t kPairsMinWorkgroups = 4096;
inline int gather_levels_per_thread(int pos_dim, int64_t n, int levels) {
    return pos_dim <= 4 && static_cast<int64_t>(tiles(n)) * ((levels + 1) / 2) >= kPairsMinWorkgroups ? 2 : 1;
}

// The largest table slice (bytes of one level) a die keeps to itself.  Up to here several slices at once fit the memory-side
// cache; with 32 MiB slices on every die that cache thrashes (2^22 slots: the forward 251 us with all dies on the same
// rows, 325 with segments; 2^20 slots: 138.5 and 135.5).
constexpr size_t kMaxSegmentSliceBytes = size_t{8} << 20;

// The map of a launch over `levels` levels, `levels_per_row` to a thread, and its grid.  Rounds: few rounds mean few fetches of
// each slice, more of them a more even share of the coarse and the fine rows for every die (a fine row costs up to five
// coarse ones).  Rows of two levels are even in themselves: three rounds, four where there are fewer rows than dies.  Rows of
// one level: three rounds while the launch is small and the fetches are a good part of it, then eight (forward, D = 6, 16 levels,
// 2^18 points: 92.5 us without segments, 94.1 / 91.2 / 91.2 with 3 / 5 / 8 rounds; D = 8, 24 levels, 20000 points: 31.4, then
// 18.1 / 21.0 / 22.4), and none for launches so large that the fetches no longer matter but the dies' unequal ends do
// (D = 5, 2^20 points: 289 and 295 us; position backward, D = 3, samples along rays, 2^20 points: 287 and 295 us).
struct GatherLaunch {
    LevelMap map;
    dim3 grid;
};
constexpr uint64_t kSmallGather = 8192, kLargeGather = 65536;  // (row, tile) pairs
inline GatherLaunch plan_gather(int64_t n, int levels, int levels_per_row, size_t slice_bytes, uint64_t most_pairs = uint64_t{1} << 30) {
    GatherLaunch g;
    g.map.tiles = tiles(n);
    g.map.rows = static_cast<uint32_t>((levels + levels_per_row - 1) / levels_per_row);
    g.map.segment = 0;
    g.map.dies = dies_of_current_device();
    g.grid = dim3(g.map.tiles, g.map.rows);
    const uint64_t work = static_cast<uint64_t>(g.map.tiles) * g.map.rows;
    // (with fewer single levels than dies the shares cannot be evened out: 6 levels of 300 k points 30.4 -> 33.1 us)
    if (g.map.dies < 2 || g.map.rows < (levels_per_row > 1 ? 2u : g.map.dies) || slice_bytes > kMaxSegmentSliceBytes ||
        work >= (levels_per_row > 1 ? most_pairs : kLargeGather))
        return g;
    const uint32_t rounds = levels_per_row > 1 ? (g.map.rows >= g.map.dies ? 3 : 4) : (work < kSmallGather ? 3 : 8);
    const uint64_t segments = static_cast<uint64_t>(rounds) * g.map.dies;
    g.map.segment = static_cast<uint32_t>((work + segments - 1) / segments);
    g.grid = dim3(static_cast<uint32_t>(segments * g.map.segment));
    return g;
}
inline size_t slice_bytes(int capacity, int nr_feat, const int format) {
    return static_cast<size_t>(capacity) * nr_feat * (format != 0 ? 2 : 4);
}

}  // namespace penc

using namespace penc;

// The part of a table gradient that comes through the position gradient: nothing, the whole of it (double_pos_grad alone;
// `grad` is then the upstream gradient of the first backward), or one of two summands (with `upstream`, [L][F][N]: the upstream
// gradient of the first backward; `grad` is that of the encoded values).
struct SecondGradient {
    const float* double_pos_grad = nullptr;
    const float* upstream = nullptr;
};

// The table gradient of penc_backward / penc_backward_table_rowmajor: clear, scatter, reduce the
// bins, in as many passes over the levels as the workspace asks for.  grad_row_stride == 0 means
// the [level][feature][n] layout, otherwise the gradient is rows of that many floats.  With
// double_pos_grad the same for the table-gradient half of the double backward.  grad_level_major (rows
// only, may be NULL) receives the upstream gradient in [level][feature][n] order as a by-product.
// With `touched` (the sparse entry points) nothing is cleared: the sums are added to a gradient the caller
// keeps across calls, and `touched` [pair level][slot range] is that caller's record of the slot ranges
// that hold anything; it takes the place of the workspace's flags of direct adds.
static int table_backward(int pos_dim, int nr_feat, int64_t nr_positions, int nr_levels, int capacity, const float* positions,
                          const float* scale_factor, const float* random_shift, const float* anneal_window,
                          const float* grad, int64_t grad_row_stride, const SecondGradient& second,
                          float* lattice_values_grad, float* grad_level_major, void* workspace, size_t workspace_bytes,
                          hipStream_t st, uint32_t* touched = nullptr) {
    const int n = static_cast<int>(nr_positions);
    const uint32_t cap = static_cast<uint32_t>(capacity), mask = mask_of(capacity);
    // every pair of features is scattered like a level of its own (see backward_table_kernel)
    const uint32_t feat_pairs = static_cast<uint32_t>(nr_feat / 2);
    const int pair_levels = nr_levels * static_cast<int>(feat_pairs);
    TableLaunch t{};
    t.stream = st;
    t.rows = grad_row_stride != 0;
    t.second_order = second.double_pos_grad != nullptr;
    t.n_points = n;
    t.feat_pairs = feat_pairs;
    t.capacity = cap;
    t.cap_mask = mask;
    t.positions = positions;
    t.scale_factor = scale_factor;
    t.random_shift = random_shift;
    t.window = anneal_window;
    t.grad = grad;
    t.grad_row_stride = grad_row_stride;
    t.double_pos_grad = second.double_pos_grad;
    t.second_grad = second.upstream;
    t.table_grad = lattice_values_grad;
    t.grad_level_major = grad_level_major;
    const uint32_t dies = dies_of_current_device();
    const GroupSortPlan sorted = plan_group_sort(pos_dim, nr_positions, nr_levels, static_cast<int>(feat_pairs), capacity, touched != nullptr,
                                                 workspace, workspace_bytes);
    if (sorted.enabled) {
        const GroupSort& g = sorted.sort;
        // (few groups: spread over the dies rather than kept together on one)
        t.dies = g.n_groups >= 2 * dies ? dies : 0u;
        const uint32_t padded = t.dies != 0u ? (g.n_groups + dies - 1) / dies * dies : g.n_groups;
        t.grid = dim3(padded * static_cast<uint32_t>(nr_levels));
        PENC_DISPATCH_D(pos_dim, launch_group_sort<DD>(t, g, static_cast<uint32_t>(nr_levels)));
        if (int rc = check_launch()) return rc;
        // a reader per group, of 16 to 256 threads
        uint32_t lanes_log2 = 4;
        while (lanes_log2 < 8 && (static_cast<uint32_t>(kRangeBlock) >> (lanes_log2 + 1)) >= g.n_groups) ++lanes_log2;
        const uint32_t items = (static_cast<uint32_t>(nr_levels) * g.n_ranges + dies - 1) / dies * dies * feat_pairs;
        hipLaunchKernelGGL(range_sum_kernel, dim3(items), dim3(kRangeBlock),
                           (size_t{2} << g.range_shift) * sizeof(double), st, g, anneal_window, cap, feat_pairs, static_cast<uint32_t>(nr_levels),
                           lanes_log2, dies, touched, bins_for_capacity(capacity), bin_shift_for_capacity(capacity), lattice_values_grad);
        return check_launch();
    }
    int tiles_per_group = table_backward_tiles(nr_positions, pair_levels);
    if (tiles_per_group > kScatterTiles && short_groups(pos_dim, feat_pairs, pair_levels, capacity, t.rows)) tiles_per_group = kScatterTiles;
    const uint32_t bin_shift = bin_shift_for_capacity(capacity), fine_shift = touched == nullptr ? fine_bin_shift(pos_dim, capacity, pair_levels) : bin_shift;
    BinPlan plan;
    if (fine_shift != bin_shift) plan = plan_bins(pos_dim, nr_positions, pair_levels, capacity, fine_shift, tiles_per_group, workspace, workspace_bytes);
    if (!plan.enabled || plan.levels_per_pass < pair_levels)
        plan = plan_bins(pos_dim, nr_positions, pair_levels, capacity, bin_shift, tiles_per_group, workspace, workspace_bytes);
    if (!plan.enabled && tiles_per_group > kScatterTiles) {  // wide bins need short segments: smaller groups of points
        tiles_per_group = kScatterTiles;
        plan = plan_bins(pos_dim, nr_positions, pair_levels, capacity, bin_shift, tiles_per_group, workspace, workspace_bytes);
    }
    if (touched != nullptr) {
        plan.target.direct = touched;
        plan.target.n_bins = bins_for_capacity(capacity);
        plan.target.bin_shift = bin_shift_for_capacity(capacity);
    } else if (plan_deferred(plan, pos_dim, nr_positions, pair_levels, capacity, tiles_per_group, lattice_values_grad, workspace, workspace_bytes)) {
        // the scattering kernel clears
    } else if (plan_late(plan, pos_dim, feat_pairs, nr_positions, pair_levels, tiles_per_group, workspace, workspace_bytes)) {
        // the reducers write all of it
    } else if (int rc = clear_table_grad(lattice_values_grad, pair_levels, capacity, plan.enabled ? plan.target.direct : nullptr,
                                         plan.direct_bytes, st)) {
        return rc;
    }
    uint32_t* const direct_flags = plan.target.direct;
    const int per_pass = plan.enabled ? plan.levels_per_pass : pair_levels;
    for (int first = 0; first < pair_levels; first += per_pass) {
        const int count = pair_levels - first < per_pass ? pair_levels - first : per_pass;
        const unsigned padded_groups = (scatter_groups(nr_positions, tiles_per_group) + dies - 1) / dies * dies;
        if (direct_flags != nullptr) plan.target.direct = direct_flags + static_cast<size_t>(first) * plan.target.n_bins;
        t.grid = dim3(padded_groups * static_cast<unsigned>(count) + plan.clear.rows * dies);
        t.many_bins = plan.target.records != nullptr && plan.target.n_bins > static_cast<uint32_t>(kStageBins);
        t.most_bins = direct_flags != nullptr && plan.target.n_bins > kFewerOpenLinesMinBins;
        t.wide_bins = direct_flags != nullptr && plan.target.bin_shift > static_cast<uint32_t>(kBinSlotsLog2);
        t.first_level = first;
        t.n_pass_levels = static_cast<uint32_t>(count);
        t.dies = dies;
        t.tiles_per_group = tiles_per_group;
        t.bins = plan.target;
        t.clear = plan.clear;
        PENC_DISPATCH_D(pos_dim, launch_table_backward<DD>(t));
        if (int rc = check_launch()) return rc;
        if (plan.enabled)
            if (int rc = reduce_bins(plan, nr_positions * (pos_dim + 1), anneal_window, first, count, capacity, feat_pairs, lattice_values_grad, st)) return rc;
    }
    if (plan.clear.pairs != 0u) {
        hipLaunchKernelGGL(add_deferred_kernel, dim3(plan.target.n_groups, static_cast<unsigned>(pair_levels)), dim3(kBlock), 0, st, plan.clear, anneal_window,
                           cap, feat_pairs, lattice_values_grad);
        return check_launch();
    }
    return PENC_OK;
}

// Whether a call takes the kernels that keep all levels of 64 points in a workgroup, where the LDS holds their rows.  Always
// when an L2 of 4 MiB holds most of the table (position gradient, D = 3, 17 levels of 2^14 slots, 2^20 points: 246 -> 174 us,
// 2^16 points 21.5 -> 13.1; forward in rows 223 -> 171 and 21.2 -> 14.3); up to 12 M gathers where it holds a third (D = 4, 16
// levels of 2^16 slots: position gradient from rows 2^17 points 50.5 -> 44.8 us, 2^20 points 316 -> 352); else as long as every
// die fetching the slices it needs of the whole table costs less than the launches saved (D = 3, 24 levels of 2^18 slots:
// 4097 points 13.2 -> 9.6 us, 2^14 points 18.4 -> 16.0, 2^15 points 25.5 -> 26.1).
constexpr size_t kBlocksTableBytes = size_t{6} << 20, kBlocksMidTableBytes = size_t{12} << 20;
constexpr int64_t kBlocksMaxGathers = 1500000, kBlocksMidMaxGathers = 12000000;
constexpr int kBlocksMaxColumns = 255;
static bool takes_point_blocks(int pos_dim, int64_t n, int levels, int capacity, int nr_feat, int columns, int table_format) {
    if (columns > kBlocksMaxColumns) return false;
    const size_t table = static_cast<size_t>(levels) * slice_bytes(capacity, nr_feat, table_format);
    if (table <= kBlocksTableBytes) return true;
    return n * levels * (pos_dim + 1) <= (table <= kBlocksMidTableBytes ? kBlocksMidMaxGathers : kBlocksMaxGathers);
}
static size_t block_tile_bytes(int columns) { return static_cast<size_t>(kBlockPoints) * (columns | 1) * sizeof(float); }
static unsigned point_blocks(int64_t n) { return static_cast<unsigned>((n + kBlockPoints - 1) / kBlockPoints); }

static int block_positions_backward(int pos_dim, int nr_feat, int64_t nr_positions, int nr_levels, int capacity, const float* positions,
                                    const TableRef& table, const float* scale_factor, const float* random_shift,
                                    const float* anneal_window, const float* grad, int64_t grad_row_stride, float* grad_level_major,
                                    float* positions_grad, hipStream_t st) {
    const uint32_t in_cells = table.cells ? 1u : 0u;
#define PENC_LAUNCH_BLOCKS(ROWS, LDS)                                                                                                       \
    PENC_DISPATCH_DFT(pos_dim, nr_feat, table.format,                                                                                      \
                      hipLaunchKernelGGL((block_backward_pos_kernel<DD, FF, TT, ROWS>), dim3(point_blocks(nr_positions)),                  \
                                         dim3(kPointBlock), LDS, st, static_cast<int>(nr_positions), nr_levels,                            \
                                         static_cast<uint32_t>(capacity), mask_of(capacity), in_cells, positions, static_cast<const TT*>(table.values), \
                                         scale_factor, random_shift, anneal_window, grad, grad_row_stride, grad_level_major, positions_grad))
    if (grad_row_stride != 0) {
        PENC_LAUNCH_BLOCKS(true, block_tile_bytes(nr_levels * nr_feat));
    } else {
        PENC_LAUNCH_BLOCKS(false, 0);
    }
#undef PENC_LAUNCH_BLOCKS
    return check_launch();
}

template <bool kSlopes, bool kSecond>
static int block_rows(int pos_dim, int nr_feat, int64_t nr_positions, int nr_levels, int extra, int capacity, const float* positions,
                      const TableRef& table, const float* scale_factor, const float* random_shift, const float* anneal_window,
                      const float* double_positions_grad, float points_scaling, float* rows, int64_t row_stride, float* slopes, hipStream_t st) {
    const uint32_t in_cells = table.cells ? 1u : 0u;
    PENC_DISPATCH_DFT(pos_dim, nr_feat, table.format,
                      hipLaunchKernelGGL((block_rows_kernel<DD, FF, TT, kSlopes, kSecond>), dim3(point_blocks(nr_positions)), dim3(kPointBlock),
                                         block_tile_bytes((nr_levels + extra) * nr_feat), st, static_cast<int>(nr_positions), nr_levels,
                                         nr_levels + extra, static_cast<uint32_t>(capacity), mask_of(capacity), in_cells, positions,
                                         static_cast<const TT*>(table.values), scale_factor, random_shift, anneal_window,
                                         double_positions_grad, points_scaling, rows, row_stride, slopes));
    return check_launch();
}

// The position gradient of penc_backward / penc_backward_rowmajor from a level-major upstream gradient:
// levels in groups of kPosLevelsPerGroup when the workspace can hold the partial sums, else one
// thread per point walks all levels.
static int positions_backward(int pos_dim, int nr_feat, int64_t nr_positions, int nr_levels, int capacity, const float* positions,
                              const TableRef& table, const float* scale_factor, const float* random_shift,
                              const float* anneal_window, const float* grad_level_major, float* positions_grad,
                              void* workspace, size_t workspace_bytes, hipStream_t st) {
    if (takes_point_blocks(pos_dim, nr_positions, nr_levels, capacity, nr_feat, nr_levels * nr_feat, table.format))
        return block_positions_backward(pos_dim, nr_feat, nr_positions, nr_levels, capacity, positions, table, scale_factor, random_shift,
                                        anneal_window, grad_level_major, 0, nullptr, positions_grad, st);
    const int n = static_cast<int>(nr_positions);
    const uint32_t cap = static_cast<uint32_t>(capacity), mask = mask_of(capacity);
    const size_t n_values = static_cast<size_t>(nr_positions) * pos_dim;
    int per_group = nr_levels, groups = 1;
    float* partial = positions_grad;
    const uintptr_t ws = (reinterpret_cast<uintptr_t>(workspace) + 255u) & ~uintptr_t{255};
    const int want_groups = (nr_levels + kPosLevelsPerGroup - 1) / kPosLevelsPerGroup;
    if (workspace != nullptr && want_groups > 1 &&
        workspace_bytes >= (ws - reinterpret_cast<uintptr_t>(workspace)) + want_groups * n_values * sizeof(float)) {
        per_group = kPosLevelsPerGroup;
        groups = want_groups;
        partial = reinterpret_cast<float*>(ws);
    }
    const GatherLaunch g = plan_gather(nr_positions, nr_levels, per_group, slice_bytes(capacity, nr_feat, table.format), kLargeGather / 2);
    const uint32_t in_cells = table.cells ? 1u : 0u;
    PENC_DISPATCH_DFT(pos_dim, nr_feat, table.format,
                      hipLaunchKernelGGL((backward_pos_kernel<DD, FF, TT>), g.grid, dim3(kBlock), 0, st, n, nr_levels, per_group, g.map, cap, mask, in_cells, positions,
                                         static_cast<const TT*>(table.values), scale_factor, random_shift, anneal_window,
                                         grad_level_major, partial));
    if (int rc = check_launch()) return rc;
    if (groups > 1) {
        // four values to a thread where that still fills the chip
        const size_t per_block = kBlock * (n_values >= size_t{1} << 19 ? 4 : 1);
        const size_t want = (n_values + per_block - 1) / per_block;
        hipLaunchKernelGGL(reduce_level_groups_kernel, dim3(static_cast<unsigned>(want < 8192 ? want : 8192)), dim3(kBlock), 0, st, partial,
                           anneal_window, per_group, nr_levels, n_values, positions_grad);
        if (int rc = check_launch()) return rc;
    }
    return PENC_OK;
}

static int transpose_rows(const float* src, int64_t src_row_stride, float* dst, int64_t rows, int cols, hipStream_t st) {
    const size_t lds = static_cast<size_t>(kTransposeRows) * (cols | 1) * sizeof(float);
    if (cols <= 0 || cols > 255 || lds > 64 * 1024) return PENC_ERR_BAD_SIZE;
    const unsigned blocks = static_cast<unsigned>((rows + kTransposeRows - 1) / kTransposeRows);
    hipLaunchKernelGGL(cols <= 8 ? transpose_kernel<2> : cols < kTransposeManyColumns ? transpose_kernel<4> : transpose_kernel<8>, dim3(blocks), dim3(kBlock), lds, st, src, src_row_stride, dst, rows, cols);
    return check_launch();
}

static int transpose_to_rows(const float* src, float* dst, int64_t dst_row_stride, int64_t rows, int cols, hipStream_t st) {
    const size_t lds = static_cast<size_t>(kTransposeRows) * (cols | 1) * sizeof(float);
    if (cols <= 0 || cols > 255 || lds > 64 * 1024) return PENC_ERR_BAD_SIZE;
    const unsigned blocks = static_cast<unsigned>((rows + kTransposeRows - 1) / kTransposeRows);
    hipLaunchKernelGGL(cols <= 8 ? transpose_to_rows_kernel<2> : cols < kTransposeManyColumns ? transpose_to_rows_kernel<4> : transpose_to_rows_kernel<8>, dim3(blocks), dim3(kBlock), lds, st, src, dst, dst_row_stride, rows, cols);
    return check_launch();
}

// penc_backward and penc_backward_static: argument checks, then the table gradient (clear, scatter,
// reduce) and the position gradient on the same stream.
static int backward_impl(int pos_dim, int nr_feat, int64_t nr_positions, int nr_levels, int capacity,
                         const float* positions, const TableRef& table, const float* scale_factor,
                         const float* random_shift, const float* anneal_window,
                         const float* grad_sliced_values, float* lattice_values_grad, float* positions_grad,
                         void* workspace, size_t workspace_bytes, void* stream, uint32_t* touched = nullptr,
                         const SecondGradient& second = {}) {
    if (int rc = check_geometry(pos_dim, nr_feat, nr_positions, nr_levels, capacity, 0)) return rc;
    if (!positions || !scale_factor || !random_shift || !anneal_window || !grad_sliced_values)
        return PENC_ERR_NULL_POINTER;
    if (!lattice_values_grad && !positions_grad) return PENC_ERR_NULL_POINTER;
    if (positions_grad && !table.values) return PENC_ERR_NULL_POINTER;
    if ((table.values && !table_aligned(table, nr_feat)) || !aligned8(lattice_values_grad)) return PENC_ERR_MISALIGNED;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (lattice_values_grad)
        if (int rc = table_backward(pos_dim, nr_feat, nr_positions, nr_levels, capacity, positions, scale_factor, random_shift,
                                    anneal_window, grad_sliced_values, 0, second, lattice_values_grad, nullptr, workspace,
                                    workspace_bytes, st, touched))
            return rc;
    if (positions_grad)
        return positions_backward(pos_dim, nr_feat, nr_positions, nr_levels, capacity, positions, table, scale_factor,
                                  random_shift, anneal_window, grad_sliced_values, positions_grad, workspace, workspace_bytes, st);
    return PENC_OK;
}

// The levels of an fp32 table that a forward gathers from cells made for it (chosen_cells_kernel).
struct ChosenCells {
    const void* cells = nullptr;
    const uint32_t* levels = nullptr;
};

static int forward_impl(int pos_dim, int nr_feat, int64_t nr_positions, int nr_levels, int capacity,
                        const float* positions, const TableRef& table, const float* scale_factor,
                        const float* random_shift, const float* anneal_window, float* sliced_values,
                        int concat_points, float points_scaling, void* stream, float* slopes = nullptr, const ChosenCells& chosen = {}) {
    const int extra = penc_extra_levels(pos_dim, nr_feat, concat_points);
    if (int rc = check_geometry(pos_dim, nr_feat, nr_positions, nr_levels, capacity, extra)) return rc;
    if (!positions || !table.values || !scale_factor || !random_shift || !anneal_window || !sliced_values)
        return PENC_ERR_NULL_POINTER;
    if (!table_aligned(table, nr_feat)) return PENC_ERR_MISALIGNED;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const GatherLaunch g = plan_gather(nr_positions, nr_levels, gather_levels_per_thread(pos_dim, nr_positions, nr_levels),
                                       slice_bytes(capacity, nr_feat, table.format));
    const uint32_t in_cells = table.cells ? 1u : 0u;
#define PENC_LAUNCH_FORWARD(FEAT, TYPE, SLOPES, CHOSEN)                                                                                  \
    hipLaunchKernelGGL((forward_kernel<DD, FEAT, TYPE, SLOPES, CHOSEN>), g.grid, dim3(kBlock), 0, st, static_cast<int>(nr_positions),     \
                       nr_levels, nr_levels + extra, g.map, static_cast<uint32_t>(capacity), mask_of(capacity), in_cells, positions,     \
                       static_cast<const TYPE*>(table.values), scale_factor, random_shift, anneal_window, sliced_values, points_scaling, \
                       slopes, static_cast<const TYPE*>(chosen.cells), chosen.levels)
    if (chosen.levels != nullptr) {  // (two or four features)
        if (nr_feat == 4 && slopes != nullptr) {
            PENC_DISPATCH_D(pos_dim, PENC_LAUNCH_FORWARD(4, float, true, true))
        } else if (nr_feat == 4) {
            PENC_DISPATCH_D(pos_dim, PENC_LAUNCH_FORWARD(4, float, false, true))
        } else if (slopes != nullptr) {
            PENC_DISPATCH_D(pos_dim, PENC_LAUNCH_FORWARD(2, float, true, true))
        } else {
            PENC_DISPATCH_D(pos_dim, PENC_LAUNCH_FORWARD(2, float, false, true))
        }
    } else if (slopes != nullptr) {
        PENC_DISPATCH_DFT(pos_dim, nr_feat, table.format, PENC_LAUNCH_FORWARD(FF, TT, true, false));
    } else {
        PENC_DISPATCH_DFT(pos_dim, nr_feat, table.format, PENC_LAUNCH_FORWARD(FF, TT, false, false));
    }
#undef PENC_LAUNCH_FORWARD
    return check_launch();
}

extern "C" {

const char* penc_status_string(int status) {
    switch (status) {
        case PENC_OK: return "ok";
        case PENC_ERR_NULL_POINTER: return "a required pointer is NULL";
        case PENC_ERR_BAD_SIZE: return "nr_positions, nr_levels and capacity must be positive and every array must stay below 2^31 elements";
        case PENC_ERR_UNSUPPORTED_POS_DIM: return "pos_dim must be 2,3,4,5,6,7 or 8";
        case PENC_ERR_UNSUPPORTED_NR_FEAT: return "nr_feat_per_level must be 2, 4 or 8";
        case PENC_ERR_MISALIGNED: return "lattice_values must be aligned to one slot (at most 16 bytes), lattice_values_grad and gradient rows to 8 bytes";
        case PENC_ERR_LAUNCH: return "the HIP runtime rejected a kernel launch";
        case PENC_ERR_WORKSPACE_TOO_SMALL: return "the workspace cannot hold the level-major array the call needs (penc_backward_rowmajor_workspace_bytes, penc_forward_rowmajor_workspace_bytes)";
        case PENC_ERR_UNSUPPORTED_TABLE_FORMAT: return "table_format must be PENC_TABLE_FP16 or PENC_TABLE_BF16, with PENC_TABLE_CELLS for capacities that are powers of two and fill a line";
        case PENC_ERR_SCRATCH_TOO_SMALL: return "the problem is too large for the library's static scratch (penc_static_scratch_bytes): use penc_backward with a workspace";
        default: return "unknown status";
    }
}

int penc_extra_levels(int pos_dim, int nr_feat, int concat_points) {
    if (!concat_points || nr_feat <= 0) return 0;
    return (pos_dim + nr_feat - 1) / nr_feat;
}

size_t penc_scatter_workspace_bytes(int pos_dim, int64_t nr_positions, int nr_levels, int capacity, int levels_per_pass) {
    if (pos_dim < 2 || pos_dim > 8 || nr_positions <= 0 || nr_levels <= 0 || capacity <= 0) return 0;
    const uint32_t n_bins = bins_for_capacity(capacity);
    if (n_bins > static_cast<uint32_t>(kMaxBins)) return 0;
    if (levels_per_pass <= 0) levels_per_pass = kDefaultLevelsPerPass;
    if (levels_per_pass > nr_levels) levels_per_pass = nr_levels;
    // the larger of what the two gradient calls plan for (they may group the points differently)
    size_t per_level = 0;
    for (const int tiles : {kScatterTiles, table_backward_tiles(nr_positions, nr_levels)}) {
        const size_t need = bin_bytes_per_level(pos_dim, n_bins, scatter_groups(nr_positions, tiles),
                                                wanted_segment_capacity(pos_dim, n_bins, tiles));
        per_level = need > per_level ? need : per_level;
    }
    const size_t binned = per_level * static_cast<size_t>(levels_per_pass) + direct_flag_bytes(nr_levels, n_bins) + 1024;
    // (how many pairs of features share a level is not known here: up to four)
    const bool may_sort = levels_per_pass == nr_levels && nr_positions * (pos_dim + 1) * ((nr_levels + 3) / 4) <= group_sort_max_lookups(pos_dim) &&
                          nr_positions <= kGroupSortPointsPerLevel * nr_levels;
    const size_t sorted = may_sort ? group_sort_bytes(pos_dim, nr_positions, nr_levels) + 256 : 0;
    return sorted > binned ? sorted : binned;
}

// feat_pairs: of the levels that `pair_levels` counts, for what a call of so many pairs has a use for; 0: for whatever number, at most.
static size_t scatter_extra_bytes(int pos_dim, uint32_t feat_pairs, int64_t nr_positions, int pair_levels, int capacity) {
    const uint32_t n_bins = bins_for_capacity(capacity), shift = bin_shift_for_capacity(capacity), fine_shift = fine_bin_shift(pos_dim, capacity, pair_levels);
    const int64_t lookups = nr_positions * (pos_dim + 1);
    const int most_tiles = table_backward_tiles(nr_positions, pair_levels);
    if (n_bins > static_cast<uint32_t>(kMaxBins) || lookups * kMinSlotsPerContribution <= capacity) return 0;
    size_t lists = 0, narrow = 0;
    for (const int tiles : {kScatterTiles, most_tiles}) {
        const uint32_t groups = scatter_groups(nr_positions, tiles), fine = bins_of_shift(capacity, fine_shift);
        const size_t need = deferred_bytes(pos_dim, pair_levels, groups, tiles), bins = bin_bytes_per_level(pos_dim, fine, groups, wanted_segment_capacity(pos_dim, fine, tiles)) * pair_levels;
        if (clears_in_scatter(n_bins, pair_levels, capacity, static_cast<int64_t>(scatter_groups(nr_positions, most_tiles)) * pair_levels) ||
            (feat_pairs != 0u ? written_whole(pos_dim, feat_pairs, nr_positions, fine, fine_shift, groups, pair_levels)
                              : few_bins_alone(fine, fine_shift, groups, lookups, pair_levels)))
            lists = need > lists ? need : lists;
        if (fine_shift != shift) narrow = bins > narrow ? bins : narrow;
    }
    if (lists != 0) lists += 256;
    if (narrow == 0) return lists;
    const size_t want = narrow + direct_flag_bytes(pair_levels, bins_of_shift(capacity, fine_shift)) + 8192 + lists;
    const size_t have = penc_scatter_workspace_bytes(pos_dim, nr_positions, pair_levels, capacity, pair_levels);
    return want > have ? want - have : 0;
}

size_t penc_scatter_extra_bytes(int pos_dim, int64_t nr_positions, int nr_levels, int capacity) {
    if (pos_dim < 2 || pos_dim > 8 || nr_positions <= 0 || nr_levels <= 0 || capacity <= 0) return 0;
    return scatter_extra_bytes(pos_dim, 0u, nr_positions, nr_levels, capacity);
}

size_t penc_scatter_useful_bytes(int pos_dim, int nr_feat_per_level, int64_t nr_positions, int nr_levels, int capacity) {
    if (pos_dim < 2 || pos_dim > 8 || nr_positions <= 0 || nr_levels <= 0 || capacity <= 0) return 0;
    if (nr_feat_per_level != 2 && nr_feat_per_level != 4 && nr_feat_per_level != 8) return 0;
    const int feat_pairs = nr_feat_per_level / 2;
    if (group_sort_serves(pos_dim, nr_positions, nr_levels, feat_pairs, capacity, false)) return 0;
    return scatter_extra_bytes(pos_dim, static_cast<uint32_t>(feat_pairs), nr_positions, nr_levels * feat_pairs, capacity);
}

size_t penc_positions_workspace_bytes(int pos_dim, int64_t nr_positions, int nr_levels) {
    if (pos_dim < 2 || pos_dim > 8 || nr_positions <= 0 || nr_levels <= kPosLevelsPerGroup) return 0;
    const size_t groups = static_cast<size_t>((nr_levels + kPosLevelsPerGroup - 1) / kPosLevelsPerGroup);
    return groups * static_cast<size_t>(nr_positions) * pos_dim * sizeof(float) + 256;
}

int penc_scale_factors(int pos_dim, int nr_levels, const float* sigmas, float* scale_factor_out) {
    if (!sigmas || !scale_factor_out) return PENC_ERR_NULL_POINTER;
    if (pos_dim < 1 || nr_levels < 1) return PENC_ERR_BAD_SIZE;
    for (int l = 0; l < nr_levels; ++l)
        for (int i = 0; i < pos_dim; ++i) {
            // the reference divides a float32 tensor element by a host scalar (Encoding.cuh:62-63), which ATen
            // evaluates as element * (1.0f / scalar): two roundings, up to one unit in the last place away
            // from a true division
            const float numerator = static_cast<float>(1.0 / __builtin_sqrt(static_cast<double>((i + 1) * (i + 2))));
            const float reciprocal = 1.0f / sigmas[l];
            scale_factor_out[l * pos_dim + i] = numerator * reciprocal;
        }
    return PENC_OK;
}

int penc_forward(int pos_dim, int nr_feat, int64_t nr_positions, int nr_levels, int capacity,
                 const float* positions, const float* lattice_values, const float* scale_factor,
                 const float* random_shift, const float* anneal_window, float* sliced_values,
                 int concat_points, float points_scaling, void* stream) {
    return forward_impl(pos_dim, nr_feat, nr_positions, nr_levels, capacity, positions, TableRef{lattice_values, 0},
                        scale_factor, random_shift, anneal_window, sliced_values, concat_points, points_scaling, stream);
}

size_t penc_forward_rowmajor_workspace_bytes(int pos_dim, int nr_feat, int64_t nr_positions, int nr_levels, int concat_points) {
    if (pos_dim < 2 || pos_dim > 8 || (nr_feat != 2 && nr_feat != 4 && nr_feat != 8) || nr_positions <= 0 || nr_levels <= 0) return 0;
    const size_t cols = static_cast<size_t>(nr_feat) * (nr_levels + penc_extra_levels(pos_dim, nr_feat, concat_points));
    return cols * static_cast<size_t>(nr_positions) * sizeof(float) + 256;
}

int penc_forward_rowmajor(int pos_dim, int nr_feat, int64_t nr_positions, int nr_levels, int capacity,
                          const float* positions, const float* lattice_values, const float* scale_factor,
                          const float* random_shift, const float* anneal_window, float* sliced_rows, int64_t row_stride,
                          int concat_points, float points_scaling, void* workspace, size_t workspace_bytes, void* stream) {
    const int extra = penc_extra_levels(pos_dim, nr_feat, concat_points);
    if (int rc = check_geometry(pos_dim, nr_feat, nr_positions, nr_levels, capacity, extra)) return rc;
    if (!sliced_rows) return PENC_ERR_NULL_POINTER;
    const int cols = nr_feat * (nr_levels + extra);
    if (cols > 255 || row_stride < cols || row_stride * nr_positions >= (int64_t{1} << 31)) return PENC_ERR_BAD_SIZE;
    const uintptr_t base = (reinterpret_cast<uintptr_t>(workspace) + 255u) & ~uintptr_t{255};
    const size_t need = static_cast<size_t>(cols) * static_cast<size_t>(nr_positions) * sizeof(float);
    if (workspace == nullptr || workspace_bytes < (base - reinterpret_cast<uintptr_t>(workspace)) + need) return PENC_ERR_WORKSPACE_TOO_SMALL;
    if (takes_point_blocks(pos_dim, nr_positions, nr_levels, capacity, nr_feat, cols, 0)) {
        if (!positions || !lattice_values || !scale_factor || !random_shift || !anneal_window) return PENC_ERR_NULL_POINTER;
        const TableRef table{lattice_values, 0};
        if (!table_aligned(table, nr_feat)) return PENC_ERR_MISALIGNED;
        return block_rows<false, false>(pos_dim, nr_feat, nr_positions, nr_levels, extra, capacity, positions, table, scale_factor, random_shift,
                                        anneal_window, nullptr, points_scaling, sliced_rows, row_stride, nullptr, static_cast<hipStream_t>(stream));
    }
    float* level_major = reinterpret_cast<float*>(base);
    if (int rc = forward_impl(pos_dim, nr_feat, nr_positions, nr_levels, capacity, positions, TableRef{lattice_values, 0}, scale_factor,
                              random_shift, anneal_window, level_major, concat_points, points_scaling, stream))
        return rc;
    return transpose_to_rows(level_major, sliced_rows, row_stride, nr_positions, cols, static_cast<hipStream_t>(stream));
}

int penc_forward_half(int pos_dim, int nr_feat, int64_t nr_positions, int nr_levels, int capacity,
                      const float* positions, const void* lattice_values_half, int table_format,
                      const float* scale_factor, const float* random_shift, const float* anneal_window,
                      float* sliced_values, int concat_points, float points_scaling, void* stream) {
    if (!known_half_format(table_format) || !cells_fit(table_format, nr_feat, capacity)) return PENC_ERR_UNSUPPORTED_TABLE_FORMAT;
    return forward_impl(pos_dim, nr_feat, nr_positions, nr_levels, capacity, positions, table_ref(lattice_values_half, table_format),
                        scale_factor, random_shift, anneal_window, sliced_values, concat_points, points_scaling, stream);
}

int penc_backward(int pos_dim, int nr_feat, int64_t nr_positions, int nr_levels, int capacity,
                  const float* positions, const float* lattice_values, const float* scale_factor,
                  const float* random_shift, const float* anneal_window,
                  const float* grad_sliced_values, float* lattice_values_grad, float* positions_grad,
                  void* workspace, size_t workspace_bytes, void* stream) {
    return backward_impl(pos_dim, nr_feat, nr_positions, nr_levels, capacity, positions, TableRef{lattice_values, 0},
                         scale_factor, random_shift, anneal_window, grad_sliced_values, lattice_values_grad, positions_grad,
                         workspace, workspace_bytes, stream);
}

size_t penc_static_scratch_bytes(void) { return PENC_STATIC_SCRATCH_BYTES; }

int penc_backward_static(int pos_dim, int nr_feat, int64_t nr_positions, int nr_levels, int capacity,
                         const float* positions, const float* lattice_values, const float* scale_factor,
                         const float* random_shift, const float* anneal_window,
                         const float* grad_sliced_values, float* lattice_values_grad, float* positions_grad,
                         void* stream) {
    if (int rc = check_geometry(pos_dim, nr_feat, nr_positions, nr_levels, capacity, 0)) return rc;
    // the scratch must hold the slot-range records of at least one level (more levels per pass as
    // they fit), a pair of features counting as a level; a problem the scatter does not bin (a capacity
    // beyond the bins' reach, too few contributions per slot) needs no scratch at all
    const int pair_levels = nr_levels * (nr_feat / 2);
    const bool binned = bins_for_capacity(capacity) <= static_cast<uint32_t>(kMaxBins) &&
                        nr_positions * (pos_dim + 1) * kMinSlotsPerContribution > capacity;
    if (lattice_values_grad != nullptr && binned &&
        penc_scatter_workspace_bytes(pos_dim, nr_positions, pair_levels, capacity, 1) > PENC_STATIC_SCRATCH_BYTES)
        return PENC_ERR_SCRATCH_TOO_SMALL;
    void* ws = static_scratch_of_current_device();
    if (ws == nullptr) return PENC_ERR_LAUNCH;
    return backward_impl(pos_dim, nr_feat, nr_positions, nr_levels, capacity, positions, TableRef{lattice_values, 0},
                         scale_factor, random_shift, anneal_window, grad_sliced_values, lattice_values_grad, positions_grad, ws,
                         PENC_STATIC_SCRATCH_BYTES, stream);
}

static int check_rows(const float* grad_rows, int64_t grad_row_stride, int64_t nr_positions, int nr_levels, int nr_feat) {
    if (!grad_rows) return PENC_ERR_NULL_POINTER;
    if (grad_row_stride < nr_feat * static_cast<int64_t>(nr_levels) || (grad_row_stride & 1) != 0 ||
        grad_row_stride * nr_positions >= (int64_t{1} << 31))
        return PENC_ERR_BAD_SIZE;
    if (!aligned8(grad_rows)) return PENC_ERR_MISALIGNED;
    return PENC_OK;
}

size_t penc_backward_rowmajor_workspace_bytes(int pos_dim, int nr_feat, int64_t nr_positions, int nr_levels, int capacity,
                                              int want_lattice_values_grad, int want_positions_grad) {
    if (pos_dim < 2 || pos_dim > 8 || (nr_feat != 2 && nr_feat != 4 && nr_feat != 8) || nr_positions <= 0 || nr_levels <= 0 || capacity <= 0)
        return 0;
    size_t scratch = 0;
    if (want_lattice_values_grad)
        scratch = penc_scatter_workspace_bytes(pos_dim, nr_positions, nr_levels * (nr_feat / 2), capacity, 0);
    if (!want_positions_grad) return scratch;
    const size_t partial = penc_positions_workspace_bytes(pos_dim, nr_positions, nr_levels);
    const size_t copy = static_cast<size_t>(nr_levels) * nr_feat * static_cast<size_t>(nr_positions) * sizeof(float);
    return 512 + copy + (scratch > partial ? scratch : partial);
}

static int backward_rowmajor_impl(int pos_dim, int nr_feat, int64_t nr_positions, int nr_levels, int capacity,
                                  const float* positions, const TableRef& table, const float* scale_factor,
                                  const float* random_shift, const float* anneal_window, const float* grad_rows,
                                  int64_t grad_row_stride, float* lattice_values_grad, float* positions_grad,
                                  void* workspace, size_t workspace_bytes, void* stream, uint32_t* touched = nullptr,
                                  const SecondGradient& second = {}) {
    if (int rc = check_geometry(pos_dim, nr_feat, nr_positions, nr_levels, capacity, 0)) return rc;
    if (!positions || !scale_factor || !random_shift || !anneal_window) return PENC_ERR_NULL_POINTER;
    if (!lattice_values_grad && !positions_grad) return PENC_ERR_NULL_POINTER;
    if (positions_grad && !table.values) return PENC_ERR_NULL_POINTER;
    if (int rc = check_rows(grad_rows, grad_row_stride, nr_positions, nr_levels, nr_feat)) return rc;
    if ((table.values && !table_aligned(table, nr_feat)) || !aligned8(lattice_values_grad)) return PENC_ERR_MISALIGNED;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (!positions_grad)
        return table_backward(pos_dim, nr_feat, nr_positions, nr_levels, capacity, positions, scale_factor, random_shift,
                              anneal_window, grad_rows, grad_row_stride, second, lattice_values_grad, nullptr, workspace,
                              workspace_bytes, st, touched);
    // The position gradient gathers level by level and reads its upstream gradient as [level][feature][n]:
    // that copy lives at the front of the workspace; the rest serves the scatter and then the partial sums.
    const size_t copy_bytes = static_cast<size_t>(nr_levels) * nr_feat * static_cast<size_t>(nr_positions) * sizeof(float);
    const uintptr_t base = (reinterpret_cast<uintptr_t>(workspace) + 255u) & ~uintptr_t{255};
    const size_t lost = base - reinterpret_cast<uintptr_t>(workspace);
    if (workspace == nullptr || workspace_bytes < lost + copy_bytes) return PENC_ERR_WORKSPACE_TOO_SMALL;
    float* level_major = reinterpret_cast<float*>(base);
    const size_t copy_span = (copy_bytes + 255u) & ~size_t{255};
    void* rest = workspace_bytes >= lost + copy_span + 256 ? reinterpret_cast<void*>(base + copy_span) : nullptr;
    const size_t rest_bytes = rest ? workspace_bytes - lost - copy_span : 0;
    if (lattice_values_grad) {
        // the scattering kernel reads every (point, level) pair of the rows anyway and leaves the copy behind
        if (int rc = table_backward(pos_dim, nr_feat, nr_positions, nr_levels, capacity, positions, scale_factor, random_shift,
                                    anneal_window, grad_rows, grad_row_stride, second, lattice_values_grad, level_major,
                                    rest, rest_bytes, st, touched))
            return rc;
    } else {
        const int cols = nr_feat * nr_levels;
        if (takes_point_blocks(pos_dim, nr_positions, nr_levels, capacity, nr_feat, cols, table.format))  // straight from the rows
            return block_positions_backward(pos_dim, nr_feat, nr_positions, nr_levels, capacity, positions, table, scale_factor,
                                            random_shift, anneal_window, grad_rows, grad_row_stride, nullptr, positions_grad, st);
        if (cols > 255) return PENC_ERR_BAD_SIZE;
        if (int rc = transpose_rows(grad_rows, grad_row_stride, level_major, nr_positions, cols, st)) return rc;
    }
    return positions_backward(pos_dim, nr_feat, nr_positions, nr_levels, capacity, positions, table, scale_factor,
                              random_shift, anneal_window, level_major, positions_grad, rest, rest_bytes, st);
}

int penc_backward_rowmajor(int pos_dim, int nr_feat, int64_t nr_positions, int nr_levels, int capacity,
                           const float* positions, const float* lattice_values, const float* scale_factor,
                           const float* random_shift, const float* anneal_window, const float* grad_rows,
                           int64_t grad_row_stride, float* lattice_values_grad, float* positions_grad,
                           void* workspace, size_t workspace_bytes, void* stream) {
    return backward_rowmajor_impl(pos_dim, nr_feat, nr_positions, nr_levels, capacity, positions, TableRef{lattice_values, 0},
                                  scale_factor, random_shift, anneal_window, grad_rows, grad_row_stride, lattice_values_grad,
                                  positions_grad, workspace, workspace_bytes, stream);
}

int penc_backward_half(int pos_dim, int nr_feat, int64_t nr_positions, int nr_levels, int capacity,
                       const float* positions, const void* lattice_values_half, int table_format,
                       const float* scale_factor, const float* random_shift, const float* anneal_window,
                       const float* grad, int64_t grad_row_stride, float* lattice_values_grad, float* positions_grad,
                       void* workspace, size_t workspace_bytes, void* stream) {
    if (!known_half_format(table_format) || !cells_fit(table_format, nr_feat, capacity)) return PENC_ERR_UNSUPPORTED_TABLE_FORMAT;
    const TableRef table = table_ref(lattice_values_half, table_format);
    if (grad_row_stride != 0)
        return backward_rowmajor_impl(pos_dim, nr_feat, nr_positions, nr_levels, capacity, positions, table, scale_factor,
                                      random_shift, anneal_window, grad, grad_row_stride, lattice_values_grad, positions_grad,
                                      workspace, workspace_bytes, stream);
    return backward_impl(pos_dim, nr_feat, nr_positions, nr_levels, capacity, positions, table, scale_factor, random_shift,
                         anneal_window, grad, lattice_values_grad, positions_grad, workspace, workspace_bytes, stream);
}

int penc_backward_table_rowmajor(int pos_dim, int nr_feat, int64_t nr_positions, int nr_levels, int capacity,
                                 const float* positions, const float* scale_factor, const float* random_shift,
                                 const float* anneal_window, const float* grad_rows, int64_t grad_row_stride,
                                 float* lattice_values_grad, void* workspace, size_t workspace_bytes, void* stream) {
    if (!lattice_values_grad) return PENC_ERR_NULL_POINTER;
    return penc_backward_rowmajor(pos_dim, nr_feat, nr_positions, nr_levels, capacity, positions, nullptr, scale_factor,
                                  random_shift, anneal_window, grad_rows, grad_row_stride, lattice_values_grad, nullptr,
                                  workspace, workspace_bytes, stream);
}

static int double_backward_impl(int pos_dim, int nr_feat, int64_t nr_positions, int nr_levels, int capacity,
                                const float* positions, const TableRef& table, const float* scale_factor,
                                const float* random_shift, const float* anneal_window,
                                const float* double_positions_grad, const float* grad, int64_t grad_row_stride,
                                float* lattice_values_grad, float* grad_grad_sliced_values, int concat_points,
                                void* workspace, size_t workspace_bytes, void* stream, uint32_t* touched = nullptr) {
    const int extra = penc_extra_levels(pos_dim, nr_feat, concat_points);
    if (int rc = check_geometry(pos_dim, nr_feat, nr_positions, nr_levels, capacity, extra)) return rc;
    if (!positions || !table.values || !scale_factor || !random_shift || !anneal_window ||
        !double_positions_grad || !grad)
        return PENC_ERR_NULL_POINTER;
    if (!lattice_values_grad && !grad_grad_sliced_values) return PENC_ERR_NULL_POINTER;
    if (!table_aligned(table, nr_feat) || !aligned8(lattice_values_grad)) return PENC_ERR_MISALIGNED;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (grad_grad_sliced_values) {
        const GatherLaunch g = plan_gather(nr_positions, nr_levels, gather_levels_per_thread(pos_dim, nr_positions, nr_levels),
                                           slice_bytes(capacity, nr_feat, table.format));
        const uint32_t in_cells = table.cells ? 1u : 0u;
        PENC_DISPATCH_DFT(pos_dim, nr_feat, table.format,
                          hipLaunchKernelGGL((grad_grad_kernel<DD, FF, TT>), g.grid, dim3(kBlock), 0, st,
                                             static_cast<int>(nr_positions), nr_levels, nr_levels + extra, g.map, static_cast<uint32_t>(capacity),
                                             mask_of(capacity), in_cells, positions, static_cast<const TT*>(table.values), scale_factor,
                                             random_shift, anneal_window, double_positions_grad, grad_grad_sliced_values));
        if (int rc = check_launch()) return rc;
    }
    if (!lattice_values_grad) return PENC_OK;
    return table_backward(pos_dim, nr_feat, nr_positions, nr_levels, capacity, positions, scale_factor, random_shift, anneal_window,
                          grad, grad_row_stride, SecondGradient{double_positions_grad, nullptr}, lattice_values_grad, nullptr, workspace,
                          workspace_bytes, st, touched);
}

int penc_double_backward_from_positions(int pos_dim, int nr_feat, int64_t nr_positions, int nr_levels,
                                        int capacity, const float* positions,
                                        const float* lattice_values, const float* scale_factor,
                                        const float* random_shift, const float* anneal_window,
                                        const float* double_positions_grad,
                                        const float* grad_sliced_values, float* lattice_values_grad,
                                        float* grad_grad_sliced_values, int concat_points, void* workspace,
                                        size_t workspace_bytes, void* stream) {
    return double_backward_impl(pos_dim, nr_feat, nr_positions, nr_levels, capacity, positions, TableRef{lattice_values, 0},
                                scale_factor, random_shift, anneal_window, double_positions_grad, grad_sliced_values, 0,
                                lattice_values_grad, grad_grad_sliced_values, concat_points, workspace, workspace_bytes,
                                stream);
}

int penc_double_backward_from_positions_rowmajor(int pos_dim, int nr_feat, int64_t nr_positions, int nr_levels,
                                                 int capacity, const float* positions, const float* lattice_values,
                                                 const float* scale_factor, const float* random_shift,
                                                 const float* anneal_window, const float* double_positions_grad,
                                                 const float* grad_rows, int64_t grad_row_stride,
                                                 float* lattice_values_grad, float* grad_grad_sliced_values,
                                                 int concat_points, void* workspace, size_t workspace_bytes,
                                                 void* stream) {
    if (nr_levels > 0 && nr_positions > 0)
        if (int rc = check_rows(grad_rows, grad_row_stride, nr_positions, nr_levels, nr_feat)) return rc;
    return double_backward_impl(pos_dim, nr_feat, nr_positions, nr_levels, capacity, positions, TableRef{lattice_values, 0},
                                scale_factor, random_shift, anneal_window, double_positions_grad, grad_rows,
                                grad_row_stride, lattice_values_grad, grad_grad_sliced_values, concat_points, workspace,
                                workspace_bytes, stream);
}

int penc_double_backward_from_positions_half(int pos_dim, int nr_feat, int64_t nr_positions, int nr_levels, int capacity,
                                             const float* positions, const void* lattice_values_half, int table_format,
                                             const float* scale_factor, const float* random_shift,
                                             const float* anneal_window, const float* double_positions_grad,
                                             const float* grad, int64_t grad_row_stride, float* lattice_values_grad,
                                             float* grad_grad_sliced_values, int concat_points, void* workspace,
                                             size_t workspace_bytes, void* stream) {
    if (!known_half_format(table_format) || !cells_fit(table_format, nr_feat, capacity)) return PENC_ERR_UNSUPPORTED_TABLE_FORMAT;
    if (grad_row_stride != 0 && nr_levels > 0 && nr_positions > 0)
        if (int rc = check_rows(grad, grad_row_stride, nr_positions, nr_levels, nr_feat)) return rc;
    return double_backward_impl(pos_dim, nr_feat, nr_positions, nr_levels, capacity, positions,
                                table_ref(lattice_values_half, table_format), scale_factor, random_shift, anneal_window,
                                double_positions_grad, grad, grad_row_stride, lattice_values_grad, grad_grad_sliced_values,
                                concat_points, workspace, workspace_bytes, stream);
}

int penc_backward_both_orders(int pos_dim, int nr_feat, int64_t nr_positions, int nr_levels, int capacity,
                              const float* positions, const void* lattice_values, int table_format, const float* scale_factor,
                              const float* random_shift, const float* anneal_window, const float* grad, int64_t grad_row_stride,
                              const float* double_positions_grad, const float* first_grad, float* lattice_values_grad,
                              uint32_t* touched, float* positions_grad, void* workspace, size_t workspace_bytes, void* stream) {
    if (!known_format(table_format) || !cells_fit(table_format, nr_feat, capacity)) return PENC_ERR_UNSUPPORTED_TABLE_FORMAT;
    if (!lattice_values_grad || !double_positions_grad || !first_grad) return PENC_ERR_NULL_POINTER;
    const TableRef table = table_ref(lattice_values, table_format);
    const SecondGradient second{double_positions_grad, first_grad};
    if (grad_row_stride != 0)
        return backward_rowmajor_impl(pos_dim, nr_feat, nr_positions, nr_levels, capacity, positions, table, scale_factor,
                                      random_shift, anneal_window, grad, grad_row_stride, lattice_values_grad, positions_grad,
                                      workspace, workspace_bytes, stream, touched, second);
    return backward_impl(pos_dim, nr_feat, nr_positions, nr_levels, capacity, positions, table, scale_factor, random_shift,
                         anneal_window, grad, lattice_values_grad, positions_grad, workspace, workspace_bytes, stream, touched,
                         second);
}

int penc_backward_positions_rowmajor(int pos_dim, int nr_feat, int64_t nr_positions, int nr_levels, int capacity,
                                     const float* positions, const void* lattice_values, int table_format, const float* scale_factor,
                                     const float* random_shift, const float* anneal_window, const float* grad_rows,
                                     int64_t grad_row_stride, float* grad_level_major, float* positions_grad, void* workspace,
                                     size_t workspace_bytes, void* stream) {
    if (!known_format(table_format) || !cells_fit(table_format, nr_feat, capacity)) return PENC_ERR_UNSUPPORTED_TABLE_FORMAT;
    if (int rc = check_geometry(pos_dim, nr_feat, nr_positions, nr_levels, capacity, 0)) return rc;
    const TableRef table = table_ref(lattice_values, table_format);
    if (!positions || !table.values || !scale_factor || !random_shift || !anneal_window || !grad_level_major || !positions_grad)
        return PENC_ERR_NULL_POINTER;
    if (int rc = check_rows(grad_rows, grad_row_stride, nr_positions, nr_levels, nr_feat)) return rc;
    if (!table_aligned(table, nr_feat)) return PENC_ERR_MISALIGNED;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int cols = nr_feat * nr_levels;
    if (takes_point_blocks(pos_dim, nr_positions, nr_levels, capacity, nr_feat, cols, table.format))
        return block_positions_backward(pos_dim, nr_feat, nr_positions, nr_levels, capacity, positions, table, scale_factor, random_shift,
                                        anneal_window, grad_rows, grad_row_stride, grad_level_major, positions_grad, st);
    if (int rc = transpose_rows(grad_rows, grad_row_stride, grad_level_major, nr_positions, cols, st)) return rc;
    return positions_backward(pos_dim, nr_feat, nr_positions, nr_levels, capacity, positions, table, scale_factor, random_shift,
                              anneal_window, grad_level_major, positions_grad, workspace, workspace_bytes, st);
}

int penc_grad_grad_rowmajor(int pos_dim, int nr_feat, int64_t nr_positions, int nr_levels, int capacity,
                            const float* positions, const void* lattice_values, int table_format, const float* scale_factor,
                            const float* random_shift, const float* anneal_window, const float* double_positions_grad,
                            float* grad_grad_rows, int64_t row_stride, int concat_points, void* workspace, size_t workspace_bytes,
                            void* stream) {
    if (!known_format(table_format) || !cells_fit(table_format, nr_feat, capacity)) return PENC_ERR_UNSUPPORTED_TABLE_FORMAT;
    const int extra = penc_extra_levels(pos_dim, nr_feat, concat_points);
    if (int rc = check_geometry(pos_dim, nr_feat, nr_positions, nr_levels, capacity, extra)) return rc;
    const TableRef table = table_ref(lattice_values, table_format);
    if (!positions || !table.values || !scale_factor || !random_shift || !anneal_window || !double_positions_grad || !grad_grad_rows)
        return PENC_ERR_NULL_POINTER;
    const int cols = nr_feat * (nr_levels + extra);
    if (cols > 255 || row_stride < cols || row_stride * nr_positions >= (int64_t{1} << 31)) return PENC_ERR_BAD_SIZE;
    if (!table_aligned(table, nr_feat)) return PENC_ERR_MISALIGNED;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (takes_point_blocks(pos_dim, nr_positions, nr_levels, capacity, nr_feat, cols, table.format))
        return block_rows<false, true>(pos_dim, nr_feat, nr_positions, nr_levels, extra, capacity, positions, table, scale_factor, random_shift,
                                       anneal_window, double_positions_grad, 1.0f, grad_grad_rows, row_stride, nullptr, st);
    const uintptr_t base = (reinterpret_cast<uintptr_t>(workspace) + 255u) & ~uintptr_t{255};
    const size_t need = static_cast<size_t>(cols) * static_cast<size_t>(nr_positions) * sizeof(float);
    if (workspace == nullptr || workspace_bytes < (base - reinterpret_cast<uintptr_t>(workspace)) + need) return PENC_ERR_WORKSPACE_TOO_SMALL;
    float* const level_major = reinterpret_cast<float*>(base);
    if (int rc = double_backward_impl(pos_dim, nr_feat, nr_positions, nr_levels, capacity, positions, table, scale_factor, random_shift,
                                      anneal_window, double_positions_grad, /* read by the table half only */ level_major, 0, nullptr,
                                      level_major, concat_points, nullptr, 0, stream))
        return rc;
    return transpose_to_rows(level_major, grad_grad_rows, row_stride, nr_positions, cols, st);
}

// Where a forward's slopes are worth keeping for the position gradient and the grad-grad (all three together, us, gathering -> slopes; more
// in penc_slopes.hpp).  With two features per level where no workgroup takes all levels of its points (takes_point_blocks), and there too once
// the batch is large enough: D = 3, 16 levels of 2^13 slots, 2^16 points 44.3 -> 28.3, 2^20 575 -> 396; D = 8, 16 levels of 2^12, 5001
// points 23.9 -> 13.1.  But a pass on fewer points waits for the host, which keeping slopes costs some 3 us (an allocation more, and what is looked
// at before they are used), so the line lies where the kernels take as long as the host does: at 3.2 M points times levels times dimensions.
// Passes of an SDF, and forward and position gradient alone, through the module:
//   D = 3, 16 levels of 2^14 slots   2^14 points 122.6 -> 126.4, 54.5 -> 57.6   2^16 (3.1 M) 130 -> 130, 56 -> 58   2^17 194 -> 161, 55 -> 57
//   D = 5, 10 levels of 2^14         2^15 points 124.7 -> 127.6, 55.0 -> 57.6   2^16 (3.3 M) 138 -> 136, 54 -> 55   2^17 212 -> 168, 58 -> 56
//   D = 8, 16 levels of 2^12         2^14 points 128 -> 128                     2^15 (4.2 M) 131 -> 131             2^16 196 -> 168
//   D = 3, 24 levels of 2^18 slots   2048 points 122.8 -> 125.5, 54.1 -> 57.1   2^14, the first without blocks, 132.9 -> 124.5, 60.6 -> 56.8
// (A captured graph, which waits for no host, would gain below the line too.)
// With four features where no such workgroups serve (D = 3, 16 levels, 2^18 points: 2^12 slots 159 -> 170, 2^14 176 -> 173, 2^15 218 -> 174, 2^16
// 224 -> 179; D = 5, 2^14 269 -> 283).  With eight where besides no L2 holds a level (D = 3, 16 levels: 2^16 slots, 2^18 points 358 -> 347
// but 224 -> 241 without the grad-grad, 2^18 slots 941 -> 809; 2^15 points 90 -> 56; D = 4, 2^16 slots 225 -> 233; D = 8, 2^18 slots 178 -> 117).
constexpr size_t kSlopesMinSliceBytes = size_t{4} << 20;
constexpr int64_t kSlopesMinWork = 3200000;
static bool slopes_serve(int pos_dim, int nr_feat, int64_t n, int levels, int capacity, int table_format) {
    const bool blocks = takes_point_blocks(pos_dim, n, levels, capacity, nr_feat, levels * nr_feat, table_format);
    if (nr_feat == 2) return !blocks || n * levels * pos_dim >= kSlopesMinWork;
    return !blocks && (nr_feat == 4 || slice_bytes(capacity, nr_feat, table_format) > kSlopesMinSliceBytes);
}

size_t penc_slopes_bytes(int pos_dim, int nr_feat, int64_t nr_positions, int nr_levels, int capacity, int table_format) {
    if (check_geometry(pos_dim, nr_feat, nr_positions, nr_levels, capacity, 0) != PENC_OK || nr_levels * nr_feat > 255) return 0;
    if (!slopes_serve(pos_dim, nr_feat, nr_positions, nr_levels, capacity, strip_cells(table_format))) return 0;
    return static_cast<size_t>(nr_levels) * slope_tiles(nr_positions) * kSlopeTile * pos_dim * nr_feat * sizeof(float);
}

// Whether a forward in rows that keeps slopes takes the kernel that keeps all levels of 64 points in a workgroup, as the one without slopes does
// there; else it is forward_kernel and a transpose, whose launch alone costs a pass that waits for the host 4 to 5 us (D = 3, 16 levels of 2^14
// slots, forward and position gradient through the module, 16384 points 62.3 -> 58.1 us, 56 without slopes).  Where the device is what is waited
// for (two launches -> one; forward and position gradient, then the pass of an SDF): D = 3, 16 levels of 2^14 slots, 2^17 points 58.7 -> 57.1,
// 169 -> 164, 2^19 points 164 -> 147, 516 -> 489; D = 5, 10 levels 165 -> 152, 519 -> 503; D = 6, 24 levels of 2^11 slots 338 -> 340, 995 -> 973.
// From seven dimensions on the columns that bring the slopes into the order of the coordinates leave room for too few workgroups (D = 7, the same
// 375 -> 392, 1272 -> 1264; D = 8 425 -> 466, 1330 -> 1353, 16 levels of 2^12 slots, 2^17 points 82.7 -> 88.4 and 2^16 60.1 -> 54.9 and 58.9 -> 61.1).
static bool slopes_in_point_blocks(int pos_dim, int64_t n, int levels, int capacity, int nr_feat, int columns, int table_format) {
    return takes_point_blocks(pos_dim, n, levels, capacity, nr_feat, columns, table_format) &&
           (pos_dim <= 6 || n * levels * (pos_dim + 1) <= kBlocksMidMaxGathers);
}

int penc_forward_slopes(int pos_dim, int nr_feat, int64_t nr_positions, int nr_levels, int capacity, const float* positions,
                        const void* lattice_values, int table_format, const float* scale_factor, const float* random_shift,
                        const float* anneal_window, float* sliced_values, float* sliced_rows, int64_t row_stride, float* slopes,
                        int concat_points, float points_scaling, void* stream) {
    if (!known_format(table_format) || !cells_fit(table_format, nr_feat, capacity)) return PENC_ERR_UNSUPPORTED_TABLE_FORMAT;
    if (!slopes) return PENC_ERR_NULL_POINTER;
    const int extra = penc_extra_levels(pos_dim, nr_feat, concat_points), cols = nr_feat * (nr_levels + extra);
    if (sliced_rows != nullptr && (cols > 255 || row_stride < cols || row_stride * nr_positions >= (int64_t{1} << 31))) return PENC_ERR_BAD_SIZE;
    const TableRef table = table_ref(lattice_values, table_format);
    if (sliced_rows != nullptr && slopes_in_point_blocks(pos_dim, nr_positions, nr_levels, capacity, nr_feat, cols, table.format)) {
        if (int rc = check_geometry(pos_dim, nr_feat, nr_positions, nr_levels, capacity, extra)) return rc;
        if (!positions || !table.values || !scale_factor || !random_shift || !anneal_window || !sliced_values) return PENC_ERR_NULL_POINTER;
        if (!table_aligned(table, nr_feat)) return PENC_ERR_MISALIGNED;
        return block_rows<true, false>(pos_dim, nr_feat, nr_positions, nr_levels, extra, capacity, positions, table, scale_factor, random_shift,
                                       anneal_window, nullptr, points_scaling, sliced_rows, row_stride, slopes, static_cast<hipStream_t>(stream));
    }
    if (int rc = forward_impl(pos_dim, nr_feat, nr_positions, nr_levels, capacity, positions, table, scale_factor,
                              random_shift, anneal_window, sliced_values, concat_points, points_scaling, stream, slopes))
        return rc;
    return sliced_rows == nullptr ? PENC_OK : transpose_to_rows(sliced_values, sliced_rows, row_stride, nr_positions, cols, static_cast<hipStream_t>(stream));
}

static size_t slope_tile_bytes(int columns) { return static_cast<size_t>(kSlopeTile) * (columns | 1) * sizeof(float); }

int penc_backward_positions_slopes(int pos_dim, int nr_feat, int64_t nr_positions, int nr_levels, const float* slopes,
                                   const float* anneal_window, const float* grad, int64_t grad_row_stride, float* grad_level_major,
                                   float* positions_grad, void* stream) {
    if (int rc = check_geometry(pos_dim, nr_feat, nr_positions, nr_levels, 1, 0)) return rc;
    if (!slopes || !anneal_window || !grad || !positions_grad) return PENC_ERR_NULL_POINTER;
    const int cols = nr_feat * nr_levels;
    const bool rows = grad_row_stride != 0;
    if (rows)
        if (int rc = check_rows(grad, grad_row_stride, nr_positions, nr_levels, nr_feat)) return rc;
    if (rows && cols > 255) return PENC_ERR_BAD_SIZE;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const dim3 grid(static_cast<unsigned>(slope_tiles(nr_positions)));
#define PENC_LAUNCH_SLOPES(ROWS)                                                                                                       \
    PENC_DISPATCH_DF(pos_dim, nr_feat,                                                                                                 \
                     hipLaunchKernelGGL((positions_from_slopes_kernel<DD, FF, ROWS>), grid, dim3(kSlopeBlock),                         \
                                        ROWS ? slope_tile_bytes(cols) : 0, st, static_cast<int>(nr_positions), nr_levels, slopes,      \
                                        anneal_window, grad, grad_row_stride, grad_level_major, positions_grad))
    if (rows) {
        PENC_LAUNCH_SLOPES(true);
    } else {
        PENC_LAUNCH_SLOPES(false);
    }
#undef PENC_LAUNCH_SLOPES
    return check_launch();
}

int penc_grad_grad_slopes(int pos_dim, int nr_feat, int64_t nr_positions, int nr_levels, const float* slopes, const float* anneal_window,
                          const float* double_positions_grad, float* grad_grad, int64_t row_stride, int concat_points, void* stream) {
    const int extra = penc_extra_levels(pos_dim, nr_feat, concat_points);
    if (int rc = check_geometry(pos_dim, nr_feat, nr_positions, nr_levels, 1, extra)) return rc;
    if (!slopes || !anneal_window || !double_positions_grad || !grad_grad) return PENC_ERR_NULL_POINTER;
    const int cols = nr_feat * (nr_levels + extra);
    const bool rows = row_stride != 0;
    if (rows && (cols > 255 || row_stride < cols || row_stride * nr_positions >= (int64_t{1} << 31))) return PENC_ERR_BAD_SIZE;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const dim3 grid(static_cast<unsigned>(slope_tiles(nr_positions)));
#define PENC_LAUNCH_SLOPES(ROWS)                                                                                                       \
    PENC_DISPATCH_DF(pos_dim, nr_feat,                                                                                                 \
                     hipLaunchKernelGGL((grad_grad_from_slopes_kernel<DD, FF, ROWS>), grid, dim3(kSlopeBlock),                         \
                                        ROWS ? slope_tile_bytes(cols) : 0, st, static_cast<int>(nr_positions), nr_levels,              \
                                        nr_levels + extra, slopes, anneal_window, double_positions_grad, grad_grad, row_stride))
    if (rows) {
        PENC_LAUNCH_SLOPES(true);
    } else {
        PENC_LAUNCH_SLOPES(false);
    }
#undef PENC_LAUNCH_SLOPES
    return check_launch();
}

// The scalars of one AdamW step as torch.optim.AdamW forms them (in double), rounded once for the kernel.
static AdamWStep adamw_scalars(double lr, double beta1, double beta2, double eps, double weight_decay, int64_t step) {
    AdamWStep a;
    a.decay = static_cast<float>(1.0 - lr * weight_decay);
    a.one_minus_b1 = static_cast<float>(1.0 - beta1);
    a.b2 = static_cast<float>(beta2);
    a.one_minus_b2 = static_cast<float>(1.0 - beta2);
    a.step_size = static_cast<float>(lr / (1.0 - __builtin_pow(beta1, static_cast<double>(step))));
    a.inv_c2 = static_cast<float>(1.0 / __builtin_sqrt(1.0 - __builtin_pow(beta2, static_cast<double>(step))));
    a.eps = static_cast<float>(eps);
    return a;
}

int penc_adamw_step(float* params, const float* grads, float* exp_avg, float* exp_avg_sq, int64_t n, double lr,
                    double beta1, double beta2, double eps, double weight_decay, int64_t step, int skip_zero_gradients,
                    void* stream) {
    if (!params || !grads || !exp_avg || !exp_avg_sq) return PENC_ERR_NULL_POINTER;
    if (n <= 0 || step <= 0) return PENC_ERR_BAD_SIZE;
    const AdamWStep a = adamw_scalars(lr, beta1, beta2, eps, weight_decay, step);
    hipStream_t st = static_cast<hipStream_t>(stream);
    const uintptr_t all = reinterpret_cast<uintptr_t>(params) | reinterpret_cast<uintptr_t>(grads) |
                          reinterpret_cast<uintptr_t>(exp_avg) | reinterpret_cast<uintptr_t>(exp_avg_sq);
    const size_t count = static_cast<size_t>(n);
    const size_t vector_part = (all & 15u) == 0 ? count / 4 * 4 : 0;
    if (vector_part != 0) {
        const size_t blocks = (vector_part / 4 + kBlock - 1) / kBlock;
        if (blocks > 0x7FFFFFFFull) return PENC_ERR_BAD_SIZE;
        hipLaunchKernelGGL(adamw_step_kernel<true>, dim3(static_cast<unsigned>(blocks)), dim3(kBlock), 0, st, params, grads,
                           exp_avg, exp_avg_sq, vector_part, a, skip_zero_gradients);
        if (int rc = check_launch()) return rc;
    }
    if (vector_part != count) {
        const size_t rest = count - vector_part;
        const size_t blocks = (rest + kBlock - 1) / kBlock;
        if (blocks > 0x7FFFFFFFull) return PENC_ERR_BAD_SIZE;
        hipLaunchKernelGGL(adamw_step_kernel<false>, dim3(static_cast<unsigned>(blocks)), dim3(kBlock), 0, st,
                           params + vector_part, grads + vector_part, exp_avg + vector_part, exp_avg_sq + vector_part, rest, a,
                           skip_zero_gradients);
        if (int rc = check_launch()) return rc;
    }
    return PENC_OK;
}

size_t penc_touched_map_entries(int nr_feat, int nr_levels, int capacity) {
    if ((nr_feat != 2 && nr_feat != 4 && nr_feat != 8) || nr_levels <= 0 || capacity <= 0) return 0;
    return static_cast<size_t>(nr_levels) * (nr_feat / 2) * bins_for_capacity(capacity);
}

int penc_touched_range_slots(int capacity) { return capacity > 0 ? 1 << bin_shift_for_capacity(capacity) : 0; }

int penc_backward_sparse(int pos_dim, int nr_feat, int64_t nr_positions, int nr_levels, int capacity,
                         const float* positions, const float* lattice_values, const float* scale_factor,
                         const float* random_shift, const float* anneal_window, const float* grad, int64_t grad_row_stride,
                         float* lattice_values_grad, uint32_t* touched, float* positions_grad, void* workspace,
                         size_t workspace_bytes, void* stream) {
    if (!lattice_values_grad || !touched) return PENC_ERR_NULL_POINTER;
    const TableRef table{lattice_values, 0};
    if (grad_row_stride != 0)
        return backward_rowmajor_impl(pos_dim, nr_feat, nr_positions, nr_levels, capacity, positions, table, scale_factor,
                                      random_shift, anneal_window, grad, grad_row_stride, lattice_values_grad, positions_grad,
                                      workspace, workspace_bytes, stream, touched);
    return backward_impl(pos_dim, nr_feat, nr_positions, nr_levels, capacity, positions, table, scale_factor, random_shift,
                         anneal_window, grad, lattice_values_grad, positions_grad, workspace, workspace_bytes, stream, touched);
}

int penc_double_backward_from_positions_sparse(int pos_dim, int nr_feat, int64_t nr_positions, int nr_levels, int capacity,
                                               const float* positions, const float* lattice_values,
                                               const float* scale_factor, const float* random_shift,
                                               const float* anneal_window, const float* double_positions_grad,
                                               const float* grad, int64_t grad_row_stride, float* lattice_values_grad,
                                               uint32_t* touched, float* grad_grad_sliced_values, int concat_points,
                                               void* workspace, size_t workspace_bytes, void* stream) {
    if (!lattice_values_grad || !touched) return PENC_ERR_NULL_POINTER;
    if (grad_row_stride != 0 && nr_levels > 0 && nr_positions > 0)
        if (int rc = check_rows(grad, grad_row_stride, nr_positions, nr_levels, nr_feat)) return rc;
    return double_backward_impl(pos_dim, nr_feat, nr_positions, nr_levels, capacity, positions, TableRef{lattice_values, 0},
                                scale_factor, random_shift, anneal_window, double_positions_grad, grad, grad_row_stride,
                                lattice_values_grad, grad_grad_sliced_values, concat_points, workspace, workspace_bytes, stream,
                                touched);
}

// The launch shared by penc_adamw_step_sparse and penc_clear_touched: one workgroup per (slot range, level).
static int launch_touched_ranges(bool update, float* params, float* grads, float* exp_avg, float* exp_avg_sq, int nr_feat,
                                 int nr_levels, int capacity, uint32_t* touched, const AdamWStep& a, int clear, void* stream) {
    if (!grads || !touched || (update && (!params || !exp_avg || !exp_avg_sq))) return PENC_ERR_NULL_POINTER;
    if ((nr_feat != 2 && nr_feat != 4 && nr_feat != 8)) return PENC_ERR_UNSUPPORTED_NR_FEAT;
    if (nr_levels <= 0 || nr_levels > 65535 || capacity <= 0) return PENC_ERR_BAD_SIZE;
    const uintptr_t all = reinterpret_cast<uintptr_t>(grads) |
                          (update ? reinterpret_cast<uintptr_t>(params) | reinterpret_cast<uintptr_t>(exp_avg) |
                                        reinterpret_cast<uintptr_t>(exp_avg_sq)
                                  : uintptr_t{0});
    if ((all & 7u) != 0) return PENC_ERR_MISALIGNED;
    const uint32_t n_ranges = bins_for_capacity(capacity), shift = bin_shift_for_capacity(capacity);
    // 16 bytes at a time where every level's first value is 16-byte aligned, else 8 (a slot of two features)
    const bool wide = (all & 15u) == 0 && (static_cast<int64_t>(capacity) * nr_feat) % 4 == 0;
    const dim3 grid(n_ranges, static_cast<unsigned>(nr_levels));
    hipStream_t st = static_cast<hipStream_t>(stream);
#define PENC_LAUNCH_TOUCHED(UPDATE, VEC)                                                                                   \
    hipLaunchKernelGGL((touched_ranges_kernel<UPDATE, VEC>), grid, dim3(kTouchedBlock<UPDATE>), 0, st, params, grads, exp_avg, exp_avg_sq, \
                       static_cast<uint32_t>(capacity), static_cast<uint32_t>(nr_feat), n_ranges, shift, touched, a, clear)
    if (update && wide) PENC_LAUNCH_TOUCHED(true, float4);
    else if (update) PENC_LAUNCH_TOUCHED(true, float2);
    else if (wide) PENC_LAUNCH_TOUCHED(false, float4);
    else PENC_LAUNCH_TOUCHED(false, float2);
#undef PENC_LAUNCH_TOUCHED
    return check_launch();
}

int penc_adamw_step_sparse(float* params, float* grads, float* exp_avg, float* exp_avg_sq, int nr_feat, int nr_levels,
                           int capacity, uint32_t* touched, double lr, double beta1, double beta2, double eps,
                           double weight_decay, int64_t step, int clear, void* stream) {
    if (step <= 0) return PENC_ERR_BAD_SIZE;
    return launch_touched_ranges(true, params, grads, exp_avg, exp_avg_sq, nr_feat, nr_levels, capacity, touched,
                                 adamw_scalars(lr, beta1, beta2, eps, weight_decay, step), clear, stream);
}

int penc_clear_touched(float* grads, int nr_feat, int nr_levels, int capacity, uint32_t* touched, void* stream) {
    return launch_touched_ranges(false, nullptr, grads, nullptr, nullptr, nr_feat, nr_levels, capacity, touched, AdamWStep{}, 1,
                                 stream);
}

// Levels of the column-major copy that are made at a time: what stays in the memory-side cache until it is read (24 levels of 2^22 slots in
// bfloat16, 32 / 64 / 128 / 384 MiB at a time 386 / 361 / 337 / 365 us, fp32 64 / 128 / 256 568 / 513 / 590).
constexpr size_t kCellChunkBytes = size_t{128} << 20;

size_t penc_table_cells_workspace_bytes(int nr_feat, int nr_levels, int capacity, int table_format) {
    if ((nr_feat != 2 && nr_feat != 4 && nr_feat != 8) || nr_levels <= 0 || capacity <= 0) return 0;
    if (strip_cells(table_format) != table_format || !known_half_format(table_format) || !cells_possible(nr_feat, capacity, table_format)) return 0;
    const size_t slice = slice_bytes(capacity, nr_feat, table_format);
    size_t levels = kCellChunkBytes / slice;
    if (levels < 1) levels = 1;
    if (levels > static_cast<size_t>(nr_levels)) levels = static_cast<size_t>(nr_levels);
    return levels * slice + 256;
}

// Gathers from a copy of at least 64 KiB a level are faster in cells by 2 to 15 ps a point and level (forward, 12 levels in binary16, 2^18
// points, table -> copy: D = 2, 2^16 slots 28.7 -> 19.5 us; D = 3, 2^16 39.4 -> 27.1, 2^20 54.8 -> 40.8, with four features 80.0 -> 51.3; D = 5,
// 2^20 84.0 -> 73.2; D = 8, 2^16 87.4 -> 79.8, with eight features 2^20 285 -> 247; 24 levels of 2^22 slots in bfloat16, 500003 points near a
// surface 315 -> 160), from a smaller one, which the first-level cache holds, slower (2^12 slots: D = 3 19.5 -> 19.8, D = 8 41.6 -> 43.8).  Making
// it takes longer than rounding the table does (24 levels, 2^18 slots 22.5 and 11.7 us, 2^20 87 and 48, 2^22 337 and 206).  The line is where a
// first pass on a new table, its copy made, takes as long either way; from 1.5 to 14 MiB a level that is about the same number of points.  24 levels in
// bfloat16, D = 3, the copy in the table's order -> in cells, us:
//   2^16 slots   32768 points 30.7 -> 34.8   65536 40.0 -> 40.3   131072 56.7 -> 52.9
//   2^18         131072 73.8 -> 78.7, along rays 62.7 -> 69.1   262144 108 -> 105, 85.0 -> 86.4   524288 179 -> 156, 131 -> 123
//   2^20         262144 190 -> 205, near a surface 184 -> 202   524288 282 -> 272, 272 -> 262
//   2^21         299593 329 -> 331, 305 -> 325   419430 395 -> 370, 363 -> 358   599186 498 -> 422, 455 -> 410
//   2^22         419430 552 -> 577, 520 -> 563   599186 678 -> 639, 626 -> 619   838860 834 -> 724, 767 -> 708
//   (16 levels: D = 4, 2^22 slots 299593 388 -> 404   419430 466 -> 447;  D = 2, four features, 2^20 419430 219 -> 222   599186 259 -> 248)
int64_t penc_table_cells_points(int nr_feat, int capacity, int table_format) {
    if ((nr_feat != 2 && nr_feat != 4 && nr_feat != 8) || capacity <= 0 || !known_half_format(table_format) ||
        strip_cells(table_format) != table_format || !cells_possible(nr_feat, capacity, table_format))
        return -1;
    const size_t slice = slice_bytes(capacity, nr_feat, table_format);
    if (slice < (size_t{64} << 10)) return -1;
    const size_t points = slice / 3 < (size_t{1} << 19) ? slice / 3 : size_t{1} << 19;
    return static_cast<int64_t>(points > slice / 28 ? points : slice / 28);
}

int penc_table_cells(int pos_dim, int nr_feat, int nr_levels, int capacity, const void* lattice_values, int source_format, int table_format,
                     void* cells, void* workspace, size_t workspace_bytes, void* stream) {
    if (int rc = check_geometry(pos_dim, nr_feat, 1, nr_levels, capacity, 0)) return rc;
    if (strip_cells(table_format) != table_format || !known_half_format(table_format) || !cells_possible(nr_feat, capacity, table_format) ||
        (source_format != 0 && source_format != table_format))
        return PENC_ERR_UNSUPPORTED_TABLE_FORMAT;
    if (!lattice_values || !cells) return PENC_ERR_NULL_POINTER;
    if (!table_aligned(TableRef{lattice_values, source_format}, nr_feat) || (reinterpret_cast<uintptr_t>(cells) & 15u) != 0) return PENC_ERR_MISALIGNED;
    const size_t slice = slice_bytes(capacity, nr_feat, table_format);
    const uintptr_t base = (reinterpret_cast<uintptr_t>(workspace) + 255u) & ~uintptr_t{255};
    const size_t lost = base - reinterpret_cast<uintptr_t>(workspace);
    if (workspace == nullptr || workspace_bytes < lost + slice) return PENC_ERR_WORKSPACE_TOO_SMALL;
    void* const columns = reinterpret_cast<void*>(base);
    const size_t room = (workspace_bytes - lost) / slice;
    const int slots = slots_per_line(nr_feat, table_format), most = room < static_cast<size_t>(nr_levels) ? static_cast<int>(room) : nr_levels;
    const uint32_t lines = static_cast<uint32_t>(capacity / slots);
    const CellMap map = cell_map(pos_dim, slots);
    hipStream_t st = static_cast<hipStream_t>(stream);
    for (int level = 0; level < nr_levels; level += most) {
        const dim3 grid((lines + kCellLines - 1) / kCellLines, nr_levels - level < most ? nr_levels - level : most);
        const void* const from = static_cast<const char*>(lattice_values) + static_cast<size_t>(level) * slice_bytes(capacity, nr_feat, source_format);
        void* const to = static_cast<char*>(cells) + static_cast<size_t>(level) * slice;
#define PENC_LAUNCH_COLUMNS(F_, T_, RAW_) hipLaunchKernelGGL((cell_columns_kernel<F_, T_, RAW_>), grid, dim3(kCellBlock), 0, st, from, lines, columns)
#define PENC_LAUNCH_COLUMNS_OF(T_, RAW_)                     \
    if (nr_feat == 2) PENC_LAUNCH_COLUMNS(2, T_, RAW_);      \
    else if (nr_feat == 4) PENC_LAUNCH_COLUMNS(4, T_, RAW_); \
    else PENC_LAUNCH_COLUMNS(8, T_, RAW_)
        if (source_format != 0) {
            PENC_LAUNCH_COLUMNS_OF(bfloat16_bits, true);  // (either format: the bits are moved)
        } else if (table_format == PENC_TABLE_BF16) {
            PENC_LAUNCH_COLUMNS_OF(bfloat16_bits, false);
        } else {
            PENC_LAUNCH_COLUMNS_OF(__half, false);
        }
#undef PENC_LAUNCH_COLUMNS_OF
#undef PENC_LAUNCH_COLUMNS
        if (int rc = check_launch()) return rc;
        switch (kLineBytes / slots / 4) {
            case 1: hipLaunchKernelGGL(cell_lines_kernel<1>, grid, dim3(kCellBlock), 0, st, columns, lines, map, to); break;
            case 2: hipLaunchKernelGGL(cell_lines_kernel<2>, grid, dim3(kCellBlock), 0, st, columns, lines, map, to); break;
            default: hipLaunchKernelGGL(cell_lines_kernel<4>, grid, dim3(kCellBlock), 0, st, columns, lines, map, to); break;
        }
        if (int rc = check_launch()) return rc;
    }
    return PENC_OK;
}

// Where one forward is worth a copy of the fp32 table in cells: from 16 M points times levels on, on levels of 64 KiB to 2 MiB with at most a slot for
// every two or three points.  What is gained depends on the points, which only the device sees: a call whose levels are not worth a copy has
// looked in vain (5 us, 9 with 2^18 slots), and one along rays to a coarse finest level loses 4 to 10%, at the line up to 15%, where unordered points, and
// points near a surface, gain up to 28%.  Below the line the loss is a larger share (up to a third) and the gain a smaller one.  Forward without -> with, us, D = 3, 24
// levels, two features, at 6.3 / 12.6 / 16.8 / 25.2 M (2^18 to 2^20 points):
//   2^14 slots, finest scale 1e-4   unordered 71 -> 63  123 -> 104  164 -> 134  241 -> 192   along rays 50 -> 50  78 -> 76  101 ->  97  147 -> 139
//                            1e-2             43 -> 48   79 ->  81  106 -> 104  154 -> 149              27 -> 31  50 -> 55   66 ->  72   96 -> 102
//   2^16                     1e-4             75 -> 69  139 -> 117  185 -> 149  273 -> 212              48 -> 52  88 -> 85  116 -> 107  170 -> 150
//                            1e-2             50 -> 53   88 ->  84  117 -> 106  170 -> 151              27 -> 32  48 -> 56   68 ->  72   97 -> 102
//   2^18                     1e-4             83 -> 91  145 -> 139  193 -> 173  283 -> 239              51 -> 65  94 -> 102 123 -> 128  179 -> 175
//                            1e-3             76 -> 81  134 -> 120  176 -> 149  261 -> 203              38 -> 54  69 -> 81   90 -> 100  133 -> 137
//                            1e-2             53 -> 70   90 -> 100  118 -> 123  172 -> 167              27 -> 36  51 -> 59   69 ->  75   98 -> 106
//   2^19         2^20 points, unordered 360 -> 375, 1e-3 286 -> 299, 1e-2 173 -> 203 (an L2 holds no such level beside what it gathers)
//   16 levels, 1e-3, 2^18 slots, 2^20 points     D = 2 115 -> 101   D = 4 230 -> 204   D = 5 291 -> 277   D = 6 337 -> 325   D = 7 387 -> 376   (D = 8, 2^19 271 -> 309)
// Four features, D = 3, 16 levels: 2^14 slots 163 -> 144, 2^16 176 -> 152, 2^17 179 -> 172, 2^18 217 -> 235; eight: 2^16 243 -> 267.
constexpr int64_t kForwardCellsMinWork = 16000000;
constexpr size_t kForwardCellsMaxSlice = size_t{2} << 20;
static bool forward_cells_serve(int pos_dim, int nr_feat, int64_t n, int levels, int capacity) {
    if (pos_dim > 7 || nr_feat == 8 || !cells_possible(nr_feat, capacity, 0) || n * levels < kForwardCellsMinWork) return false;
    const size_t slice = slice_bytes(capacity, nr_feat, 0);
    return slice >= (size_t{64} << 10) && slice <= kForwardCellsMaxSlice && slice <= static_cast<size_t>(n) * 3;
}
// What the workspace holds: the flags of the levels, then the copy.
static size_t forward_cells_flags(int levels) { return (static_cast<size_t>(levels) * sizeof(uint32_t) + 255u) & ~size_t{255}; }

size_t penc_forward_cells_workspace_bytes(int pos_dim, int nr_feat, int64_t nr_positions, int nr_levels, int capacity, int row_columns) {
    if (check_geometry(pos_dim, nr_feat, nr_positions, nr_levels, capacity, 0) != PENC_OK) return 0;
    // (rows that a workgroup of 64 points and all levels writes need no transpose)
    if (row_columns != 0 && takes_point_blocks(pos_dim, nr_positions, nr_levels, capacity, nr_feat, row_columns, 0)) return 0;
    if (!forward_cells_serve(pos_dim, nr_feat, nr_positions, nr_levels, capacity)) return 0;
    return forward_cells_flags(nr_levels) + slice_bytes(capacity, nr_feat, 0) * static_cast<size_t>(nr_levels) + 256;
}

int penc_forward_cells(int pos_dim, int nr_feat, int64_t nr_positions, int nr_levels, int capacity, const float* positions,
                       const float* lattice_values, const float* scale_factor, const float* random_shift, const float* anneal_window,
                       float* sliced_values, float* sliced_rows, int64_t row_stride, float* slopes, int concat_points, float points_scaling,
                       void* workspace, size_t workspace_bytes, void* stream) {
    const int extra = penc_extra_levels(pos_dim, nr_feat, concat_points), cols = nr_feat * (nr_levels + extra);
    if (int rc = check_geometry(pos_dim, nr_feat, nr_positions, nr_levels, capacity, extra)) return rc;
    if (sliced_rows != nullptr && (cols > 255 || row_stride < cols || row_stride * nr_positions >= (int64_t{1} << 31))) return PENC_ERR_BAD_SIZE;
    if (nr_feat == 8 || !cells_possible(nr_feat, capacity, 0)) return PENC_ERR_UNSUPPORTED_TABLE_FORMAT;
    if (!positions || !lattice_values || !scale_factor || !random_shift || !anneal_window || !sliced_values) return PENC_ERR_NULL_POINTER;
    const TableRef table{lattice_values, 0};
    if (!table_aligned(table, nr_feat)) return PENC_ERR_MISALIGNED;
    const size_t flags = forward_cells_flags(nr_levels);
    const uintptr_t base = (reinterpret_cast<uintptr_t>(workspace) + 255u) & ~uintptr_t{255};
    if (workspace == nullptr || workspace_bytes < (base - reinterpret_cast<uintptr_t>(workspace)) + flags +
                                                      slice_bytes(capacity, nr_feat, 0) * static_cast<size_t>(nr_levels))
        return PENC_ERR_WORKSPACE_TOO_SMALL;
    uint32_t* const chosen = reinterpret_cast<uint32_t*>(base);
    float* const cells = reinterpret_cast<float*>(base + flags);
    const int slots = slots_per_line(nr_feat, 0);
    const uint32_t lines = static_cast<uint32_t>(capacity / slots), levels = static_cast<uint32_t>(nr_levels), dies = dies_of_current_device();
    const uint32_t per_level = (lines + kCellLines * kCellsPerWorkgroup - 1) / (kCellLines * kCellsPerWorkgroup);
    const CellMap map = cell_map(pos_dim, slots);
    const dim3 grid(dies * per_level * ((levels + dies - 1) / dies));
    hipStream_t st = static_cast<hipStream_t>(stream);
#define PENC_LAUNCH_CHOSEN(F_)                                                                                                              \
    PENC_DISPATCH_D(pos_dim, hipLaunchKernelGGL((chosen_cells_kernel<DD, F_>), grid, dim3(kCellBlock), 0, st, lattice_values, lines, levels, \
                                                per_level, dies, map, nr_positions, positions, scale_factor, random_shift, anneal_window,    \
                                                chosen, cells))
    if (nr_feat == 4) {
        PENC_LAUNCH_CHOSEN(4);
    } else {
        PENC_LAUNCH_CHOSEN(2);
    }
#undef PENC_LAUNCH_CHOSEN
    if (int rc = check_launch()) return rc;
    if (int rc = forward_impl(pos_dim, nr_feat, nr_positions, nr_levels, capacity, positions, table, scale_factor, random_shift, anneal_window,
                              sliced_values, concat_points, points_scaling, stream, slopes, ChosenCells{cells, chosen}))
        return rc;
    return sliced_rows == nullptr ? PENC_OK : transpose_to_rows(sliced_values, sliced_rows, row_stride, nr_positions, cols, st);
}

int penc_upload(const float* host_values, float* dst, int n, void* stream) {
    if (!host_values || !dst) return PENC_ERR_NULL_POINTER;
    if (n <= 0) return PENC_ERR_BAD_SIZE;
    for (int first = 0; first < n; first += kUploadValues) {
        UploadValues values;
        const int count = n - first < kUploadValues ? n - first : kUploadValues;
        __builtin_memcpy(values.v, host_values + first, static_cast<size_t>(count) * sizeof(float));
        hipLaunchKernelGGL(upload_kernel, dim3(1), dim3(kUploadValues), 0, static_cast<hipStream_t>(stream), values, count, dst + first);
        if (int rc = check_launch()) return rc;
    }
    return PENC_OK;
}

int penc_transpose(const float* src, float* dst, int64_t rows, int cols, void* stream) {
    if (!src || !dst) return PENC_ERR_NULL_POINTER;
    if (rows <= 0 || cols <= 0 || cols > 255 || rows > ((int64_t{1} << 31) - 1) / cols) return PENC_ERR_BAD_SIZE;
    return transpose_rows(src, cols, dst, rows, cols, static_cast<hipStream_t>(stream));
}

int penc_simplex_debug(int pos_dim, int64_t nr_positions, int nr_levels, int capacity,
                       const float* positions, const float* scale_factor, const float* random_shift,
                       int gather_path, int* rem0, int* rank, int* slot, float* barycentric, void* stream) {
    if (int rc = check_geometry(pos_dim, 2, nr_positions, nr_levels, capacity, 0)) return rc;
    if (nr_positions > ((int64_t{1} << 31) - 1) / (pos_dim + 1) / nr_levels) return PENC_ERR_BAD_SIZE;
    if (!positions || !scale_factor || !random_shift) return PENC_ERR_NULL_POINTER;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const dim3 grid(tiles(nr_positions), nr_levels);
#define PENC_LAUNCH_DEBUG(ROUTINE)                                                                                   \
    PENC_DISPATCH_D(pos_dim, hipLaunchKernelGGL((simplex_debug_kernel<DD, ROUTINE>), grid, dim3(kBlock), 0, st,       \
                                                static_cast<int>(nr_positions), static_cast<uint32_t>(capacity),     \
                                                mask_of(capacity), positions, scale_factor, random_shift, rem0, rank, \
                                                slot, barycentric))
    switch (gather_path) {
        case kBySelects: PENC_LAUNCH_DEBUG(kBySelects); break;
        case kByNetwork: PENC_LAUNCH_DEBUG(kByNetwork); break;
        case kByNetworkBothOrders: PENC_LAUNCH_DEBUG(kByNetworkBothOrders); break;
        default: PENC_LAUNCH_DEBUG(kByLds); break;
    }
#undef PENC_LAUNCH_DEBUG
    return check_launch();
}

}  // extern "C"
