// The scattering and the sorting kernel of the table gradient, for the input dimension PENC_DIM (see penc_table_backward.hpp).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "penc_group_sort.hpp"
#include "penc_lattice.hpp"
#include "penc_scatter.hpp"
#include "penc_table_backward.hpp"

namespace penc {

// ------------------------------------------------------------------------------------------
// backward w.r.t. the table (EncodingGPU.cuh:259-414)

// Wavefronts per SIMD the scattering kernel is compiled for: six (three workgroups per compute unit, at
// most 80 vector registers) where that costs a few spilled registers at most, else four (two
// workgroups, 128 registers).  Measured at 2^19 points, 24 levels: table backward 0.367 -> 0.338 ms
// at D = 4 (84 -> 80 registers, 3 spilled); the second-order kernel
// 0.577 -> 0.552 ms at D = 4; at D = 8 the second-order kernel needed 130 registers and ran one workgroup per compute
// unit: held to 128, 1.334 -> 1.113 ms.  At D = 5 two workgroups whose staging space takes all six vertices of a point are better than three
// that sort a tile in two chunks (16 levels of 2^18 slots, 2^19 points, scatter and reduction 323 -> 314 us, second order 327 -> 315).
// Workgroups of 1024 threads, the wide bins' among them, are alone on their compute unit: four.
// (The register counts are of the search by ranks.  With the sorting network the first order takes 80 at D = 4 and none is spilled, 125 at D = 8; of both orders a few
// addresses are spilled, before the first tile, at D = 3 and from D = 6 on: ParkedWeights.)
constexpr int scatter_waves_per_simd(int pos_dim, int threads) { return pos_dim <= 4 && threads == kScatterBlock ? 6 : 4; }

constexpr int both_orders_waves_per_simd(int pos_dim, int threads) { return pos_dim <= 3 && threads == kScatterBlock ? 6 : 4; }

// kRowMajor: the upstream gradient is read as rows grad[n][2*level + feature] of `grad_row_stride`
// floats (what the layer after the encoding produces) instead of [level][feature][n].  A die walks
// all levels of a group of points back to back, so that part of the rows' many reads comes from its L2, although every level only uses
// 8 bytes of each: one L2 request per lane and level where the other layout has one per 16 lanes.  Measured at 2^20 points, 24
// levels, D = 3, in groups of 16 tiles (a die holds 6 MB of rows at a time): 711 MiB read, the 192 MiB of rows 3.6 times, 42.9 M L2
// requests, 375 us; in groups of eight 280 MiB, the rows 1.4 times, 45.2 M requests, 366 us; from [level][feature][n] 221 MiB, 17.8 M, 311 us.  At
// 2^19 points, 16 levels, D = 8 (8 tiles, rows of 128 bytes) 328 us from rows, 316 from [level][feature][n].
// With `grad_level_major` the kernel also leaves the values it read in [level][feature][n] order
// (for the position-gradient kernel, which gathers level by level and wants its upstream gradient
// coalesced): the layout change rides on reads this kernel makes anyway.
// Second order: the table-gradient half of the double backward (EncodingGPU.cuh:1016-1257): the
// vertex weights are the derivatives of the barycentric weights along `double_pos_grad` instead of
// the barycentric weights themselves; everything else is the same scatter.
// feat_pairs: with four or eight features per level the pairs (0,1), (2,3), ... are scattered like levels that
// share their geometry: "levels" below (first_level, n_pass_levels, the grid, the bins) count pairs,
// `pair_level` = level * feat_pairs + pair.  The upstream gradient needs no special case: [L][F][N]
// is [L * F/2][2][N], and in a row the pair sits at column 2 * pair_level.
// kBins: what the bins are.  Many: the records go to more than kStageBins bins (stream_tile_many), so that neither sort's registers are spilled
// for the other's sake.  Wide: of more than kBinSlots slots (tables above 2^22 slots), narrow: of fewer (small tables).  A parameter of the kernel
// rather than a value read from its arguments, because with the bin width a variable the usual instances
// need up to eight more vector registers (at D = 4, held to 80 registers, 27 spilled instead of 5).
enum BinKind : int { kBinsFew = 0, kBinsNarrow = 1, kBinsMany = 2, kBinsWide = 3 };
template <int kBins>
using ClearTargetOf = std::conditional_t<(kBins >= kBinsMany), ClearTarget, std::conditional_t<kBins == kBinsFew, LateTarget, NoLateTarget>>;
// kOrder: kFirstOrder, kSecondOrder (above), or kBothOrders: the table gradient of a loss on the encoded values and of
// a loss on the position gradient of the same points in one pass (`second_grad`, always [level][feature][n], is the upstream
// gradient of the latter).  Both are sums over the same simplices, so they share the search, the records and the
// reducer; apart, the second pass and the dense sum of the two gradients were a third of an SDF training step.
enum TableOrder : int { kFirstOrder = 1, kSecondOrder = 2, kBothOrders = 3 };
// From which dimension on the weights are parked (ParkedWeights): below, nothing is spilled without.
constexpr int park_min_dim(int order) { return order == kBothOrders ? 3 : (order == kFirstOrder ? 4 : 5); }
template <int D, bool kRowMajor, int kOrder, int kBins, int kThreads>
__device__ __forceinline__ void
scatter_group_of_points(int n_points, int first_level, uint32_t n_pass_levels, uint32_t feat_pairs, uint32_t dies, int tiles_per_group,
                        uint32_t capacity, uint32_t cap_mask,
                        const float* __restrict__ positions, const float* __restrict__ scale_factor,
                        const float* __restrict__ random_shift, const float* __restrict__ window,
                        const float* __restrict__ grad_sliced, int64_t grad_row_stride,
                        const float* __restrict__ double_pos_grad, const float* __restrict__ second_grad,
                        float* __restrict__ table_grad, float* __restrict__ grad_level_major, const BinTarget& pass_bins,
                        const ClearTargetOf<kBins>& clear) {
    constexpr bool kNeedsQ = kOrder != kFirstOrder, kBoth = kOrder == kBothOrders, kManyBins = kBins >= kBinsMany;
    __shared__ ScatterStateT<stage_chunk(D), kThreads> state;
    // Workgroups are dealt round-robin to the chip's `dies` dies, each with an L2 of its own.  The j-th
    // workgroup of a die takes level j % levels of one group of points: a die works through all
    // levels of a group before the next group, so the points are fetched from memory once, and
    // compute-bound coarse levels and store-bound fine levels share the chip at all times (this
    // kernel never reads the table: there is no slice to keep cache-resident by running a level at
    // a time).
    const uint32_t die = blockIdx.x % dies;
    uint32_t j = blockIdx.x / dies;
    if constexpr (kManyBins) {
        if (clear.kept != nullptr) {
            const uint32_t workgroups = clear.rows != 0u ? clear.rows * dies : gridDim.x;
            if (blockIdx.x < workgroups) {
                typedef float Quad __attribute__((ext_vector_type(4)));
                const uint64_t quads = clear.pairs / 2, share = (quads + workgroups - 1) / workgroups, from = share * blockIdx.x;
                const uint64_t to = from + share < quads ? from + share : quads;
                for (uint64_t i = from + threadIdx.x; i < to; i += kThreads) __builtin_nontemporal_store(Quad(0.0f), reinterpret_cast<Quad*>(table_grad) + i);
                if ((clear.pairs & 1u) != 0u && blockIdx.x == 0 && threadIdx.x == 0) reinterpret_cast<float2*>(table_grad)[clear.pairs - 1] = make_float2(0.0f, 0.0f);
                for (uint32_t flag = blockIdx.x * kThreads + threadIdx.x; flag < clear.flags; flag += workgroups * kThreads) pass_bins.direct[flag] = 0u;
                if (clear.rows != 0u) return;
            }
            j -= clear.rows;
        }
    }
    const uint32_t level_in_pass = j % n_pass_levels, group = (j / n_pass_levels) * dies + die;
    const int64_t group_base = static_cast<int64_t>(group) * tiles_per_group * kThreads;
    if (group_base >= n_points) return;
    const uint32_t pair_level = static_cast<uint32_t>(first_level) + level_in_pass;
    const int level = static_cast<int>(pair_level / feat_pairs);  // the geometry's level
    const float w_level = window[level];
    if (w_level == 0.0f) return;
    BinRecord* deferred = nullptr;
    if constexpr (kBins != kBinsNarrow) {
        if (clear.kept != nullptr) deferred = clear.kept + (static_cast<size_t>(level_in_pass) * pass_bins.n_groups + group) * clear.room;
        if (threadIdx.x == 0) state.deferred = 0u;
    }
    BinTarget bins = bins_of_level(pass_bins, level_in_pass);
    if constexpr (kBins == kBinsFew || kBins == kBinsMany) bins.bin_shift = kBinSlotsLog2;  // a constant from here on
    const GradSlice level_grad{table_grad + (static_cast<size_t>(level) * capacity * feat_pairs + pair_level % feat_pairs) * 2,
                               2 * feat_pairs, bins.direct, bins.bin_shift, deferred, &state.deferred};
    // Everything a thread reads lies within its group of at most 16 x 512 points, so the addresses are
    // wave-uniform 64-bit bases (scalar registers) plus 32-bit per-thread offsets in bytes: the form the load instructions take.
    const uint32_t last_in_group = static_cast<uint32_t>(n_points - 1 - group_base);
    const float* const group_positions = positions + group_base * D;
    const float* const group_q = kNeedsQ ? double_pos_grad + group_base * D : nullptr;
    const float* const group_grad0 =
        kRowMajor ? grad_sliced + group_base * grad_row_stride + 2 * pair_level
                  : grad_sliced + (static_cast<size_t>(pair_level) * 2) * n_points + group_base;
    const float* const group_grad1 = group_grad0 + n_points;
    const auto at_byte = [](const float* base, uint32_t offset) { return reinterpret_cast<const float*>(reinterpret_cast<const char*>(base) + offset); };
    const auto load_grad = [&](uint32_t i, float& g0, float& g1) {
        if constexpr (kRowMajor) {
            const float2 g = *reinterpret_cast<const float2*>(group_grad0 + static_cast<int64_t>(i) * grad_row_stride);
            g0 = g.x;
            g1 = g.y;
        } else {
            g0 = *at_byte(group_grad0, i * 4u);
            g1 = *at_byte(group_grad1, i * 4u);
        }
    };
    const float* const group_second0 = kBoth ? second_grad + (static_cast<size_t>(pair_level) * 2) * n_points + group_base : nullptr;
    const float* const group_second1 = group_second0 + n_points;
    const auto load_group_point = [&](const float* base, uint32_t i) {
        const float* const p = at_byte(base, i * static_cast<uint32_t>(D * sizeof(float)));
        fvec<D> v;
        static_for<D>(PENC_BODY(k) {
            PENC_INDEX(k); v[k] = p[k]; });
        return v;
    };
    // A tile's inputs are fetched one tile ahead: their latency then overlaps the previous tile's
    // scatter instead of stalling the wave at the top of every iteration.
    const auto point_of = [&](int t) {  // the point this thread handles in tile t, within the group (clamped: the tail re-reads the last point)
        const uint32_t i = static_cast<uint32_t>(t) * kThreads + threadIdx.x;
        return i < last_in_group ? i : last_in_group;
    };
    uint32_t nn = point_of(0);
    fvec<D> pos = load_group_point(group_positions, nn);
    fvec<D> q = 0.0f;
    if constexpr (kNeedsQ) q = load_group_point(group_q, nn);
    float g0, g1;
    load_grad(nn, g0, g1);
    float s0 = 0.0f, s1 = 0.0f;
    if constexpr (kBoth) {
        s0 = group_second0[nn];
        s1 = group_second1[nn];
    }
    scatter_begin(state);  // (while the first tile is on its way)
    int mode = kModeCache;
    uint32_t id_bits = 0, cursor = 0;
    for (int t = 0; t < tiles_per_group; ++t) {
        const int64_t tile_base = group_base + static_cast<int64_t>(t) * kThreads;
        if (tile_base >= n_points) break;
        const bool active = tile_base + threadIdx.x < n_points;
        const uint32_t nn_next = point_of(t + 1);
        const fvec<D> pos_next = load_group_point(group_positions, nn_next);
        fvec<D> q_next = 0.0f;
        if constexpr (kNeedsQ) q_next = load_group_point(group_q, nn_next);
        float g0_next, g1_next;
        load_grad(nn_next, g0_next, g1_next);
        float s0_next = 0.0f, s1_next = 0.0f;
        if constexpr (kBoth) {
            s0_next = *at_byte(group_second0, nn_next * 4u);
            s1_next = *at_byte(group_second1, nn_next * 4u);
        }
        if constexpr (kRowMajor) {
            if (grad_level_major != nullptr && active) {
                float* out = grad_level_major + (static_cast<size_t>(pair_level) * 2) * n_points + tile_base + threadIdx.x;
                out[0] = g0;
                out[n_points] = g1;
            }
        }
        CyclicSimplex<D> s = scatter_simplex<D, kOrder != kSecondOrder, kNeedsQ>(pos, q, random_shift + level * D, scale_factor + level * D, capacity, cap_mask);
        if (t == 0) {
            // the next tile's slots, should the decision want to know whether its points use the slots this tile uses
            // (its point is already here).  This tile's weights wait in the LDS meanwhile (ParkedWeights).
            constexpr bool kPark = D >= park_min_dim(kOrder);
            const auto slots_of_next_tile = [&]() {
                const ParkedWeights<D, kBoth ? 2 : 1, ScatterStateT<stage_chunk(D), kThreads>> parked{state};
                if constexpr (kPark) {
                    parked.template put<0>(kOrder == kSecondOrder ? s.dB : s.w);
                    if constexpr (kBoth) parked.template put<1>(s.dB);
                    wave_lds_fence();
                }
                const uvec<D + 1> next_slot = scatter_simplex<D, false, false>(pos_next, q, random_shift + level * D, scale_factor + level * D, capacity, cap_mask).slot;
                if constexpr (kPark) {
                    wave_lds_fence();
                    parked.template take<0>(kOrder == kSecondOrder ? s.dB : s.w);
                    if constexpr (kBoth) parked.template take<1>(s.dB);
                }
                return next_slot;
            };
            const bool next_active = tile_base + kThreads + threadIdx.x < n_points && tiles_per_group > 1;
            const uint32_t points = last_in_group < static_cast<uint32_t>(kThreads) ? last_in_group + 1u : kThreads;
            mode = scatter_mode_decide<D>(state, bins, active, points, s.slot, id_bits, next_active, slots_of_next_tile, tiles_per_group);
        }
        // b_r * w_level (:405), or dB[r] * w_level (:1244-1245)
        fvec<D + 1> w = (kOrder == kSecondOrder ? s.dB : s.w) * w_level;
        fvec<D + 1> w2 = 0.0f;
        if constexpr (kBoth) w2 = s.dB * w_level;
        if (mode == kModeCache) {  // which folds lanes by vertex: the same vertex of a simplex in the same place in all lanes
            s.slot = turn_back<D + 1>(s.slot, s.turned);
            w = turn_back<D + 1>(w, s.turned);
            if constexpr (kBoth) w2 = turn_back<D + 1>(w2, s.turned);
        }
        fvec<D + 1> a0 = w * g0, a1 = w * g1;  // g_f * (b_r * w_level), :405-410
        if constexpr (kBoth) {
            a0 += w2 * s0;
            a1 += w2 * s1;
        }
        const uint32_t hits = scatter_tile<D, kManyBins>(state, level_grad, bins, group, static_cast<uint32_t>(t), active, cache_pays<D>(state, t), mode, id_bits, s.slot, a0, a1, cursor);
        // the first tile finds the lines its own look-up has claimed: no evidence of reuse
        if ((threadIdx.x & 63) == 0 && hits && t > 0) atomicAdd(&state.hits, hits);
        pos = pos_next;
        q = q_next;
        g0 = g0_next;
        g1 = g1_next;
        s0 = s0_next;
        s1 = s1_next;
    }
    scatter_end<D, kManyBins>(state, level_grad, bins, group, mode, id_bits, cursor);
    if constexpr (kBins != kBinsNarrow) {
        if (deferred != nullptr && threadIdx.x == 0) clear.counts[static_cast<size_t>(level_in_pass) * pass_bins.n_groups + group] = state.deferred;
    }
}

#define PENC_TABLE_PARAMETERS                                                                                                          \
    int n_points, int first_level, uint32_t n_pass_levels, uint32_t feat_pairs, uint32_t dies, int tiles_per_group, uint32_t capacity, \
        uint32_t cap_mask, const float *__restrict__ positions, const float *__restrict__ scale_factor,                                \
        const float *__restrict__ random_shift, const float *__restrict__ window, const float *__restrict__ grad_sliced,               \
        int64_t grad_row_stride, const float *__restrict__ double_pos_grad, const float *__restrict__ second_grad,                     \
        float *__restrict__ table_grad, float *__restrict__ grad_level_major, BinTarget pass_bins, ClearTargetOf<kBins> clear
#define PENC_TABLE_ARGUMENTS                                                                                                        \
    n_points, first_level, n_pass_levels, feat_pairs, dies, tiles_per_group, capacity, cap_mask, positions, scale_factor,           \
        random_shift, window, grad_sliced, grad_row_stride, double_pos_grad, second_grad, table_grad, grad_level_major, pass_bins, clear
template <int D, bool kRowMajor, bool kSecond, int kBins, int kThreads>
__global__ void __launch_bounds__(kThreads, scatter_waves_per_simd(D, kThreads))
backward_table_kernel(PENC_TABLE_PARAMETERS) {
    scatter_group_of_points<D, kRowMajor, kSecond ? kSecondOrder : kFirstOrder, kBins, kThreads>(PENC_TABLE_ARGUMENTS);
}
template <int D, bool kRowMajor, int kBins, int kThreads>
__global__ void __launch_bounds__(kThreads, both_orders_waves_per_simd(D, kThreads))
backward_table_both_kernel(PENC_TABLE_PARAMETERS) {
    scatter_group_of_points<D, kRowMajor, kBothOrders, kBins, kThreads>(PENC_TABLE_ARGUMENTS);
}
#undef PENC_TABLE_PARAMETERS
#undef PENC_TABLE_ARGUMENTS

// ------------------------------------------------------------------------------------------
// the same for batches that do not fill the chip for long (see penc_group_sort.hpp)

// Levels whose points share a hundred slots or so are summed in an LDS table first (lines of a tag and two fp64 sums, kept
// where the records are staged later) and leave one record per line: else every group leaves hundreds of records on the same
// few slots, which the one range_sum_kernel workgroup that owns those slots adds one after the other (2 to 3 clocks per lane and add).
// A level with a handful of slots spreads each over several lines, by lane, so that the lanes of a wave rarely meet.
constexpr uint32_t kGroupLinesLog2 = 9, kGroupLines = 1u << kGroupLinesLog2, kGroupProbes = 8;
// Not for a few thousand points, whose records on one slot are a few hundred at most: the table's barriers cost more.
constexpr int kGroupLinesMinPoints = 4096;
static_assert(kGroupLines == kGroupPoints, "a thread per line");
constexpr int group_sort_waves_per_simd(int pos_dim) { return pos_dim <= 3 ? 6 : (pos_dim == 4 ? 5 : 4); }

template <int D, bool kRowMajor, int kOrder>
__global__ void __launch_bounds__(kGroupPoints, group_sort_waves_per_simd(D))
group_sort_kernel(int n_points, uint32_t n_levels, uint32_t feat_pairs, uint32_t dies, uint32_t capacity, uint32_t cap_mask,
                  const float* __restrict__ positions, const float* __restrict__ scale_factor, const float* __restrict__ random_shift,
                  const float* __restrict__ window, const float* __restrict__ grad, int64_t grad_row_stride,
                  const float* __restrict__ double_pos_grad, const float* __restrict__ second_grad, float* __restrict__ grad_level_major,
                  GroupSort sort) {
    constexpr bool kNeedsQ = kOrder != kFirstOrder, kBoth = kOrder == kBothOrders;
    constexpr int kRecords = (D + 1) * kGroupPoints, kWaves = kGroupPoints / 64;
    __shared__ RecordValues stage_values[kRecords];
    __shared__ uint16_t stage_slots[kRecords];
    __shared__ uint32_t count[kGroupMaxRanges + 1];  // records per range, then where each range starts
    __shared__ uint32_t wave_total[kWaves];
    __shared__ uint32_t repeats;
    struct Lines {
        double sum[2][kGroupLines];
        int tag[kGroupLines];
    };
    static_assert(sizeof(Lines) <= sizeof(stage_values), "the table of lines lives where the values are staged");
    static_assert(kGroupMaxRanges == kGroupPoints, "a thread per range");
    Lines& lines = *reinterpret_cast<Lines*>(stage_values);
    // all levels of a group of points on one die, as in the scatter: rows then come from its L2 after the first level
    uint32_t level, group;
    if (dies != 0u) {
        const uint32_t j = blockIdx.x / dies;
        level = j % n_levels;
        group = j / n_levels * dies + blockIdx.x % dies;
    } else {
        level = blockIdx.x % n_levels;
        group = blockIdx.x / n_levels;
    }
    if (group >= sort.n_groups) return;
    const float w_level = window[level];
    if (w_level == 0.0f) return;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t mine = static_cast<int64_t>(group) * kGroupPoints + tid;
    const bool active = mine < n_points;
    const int64_t n = active ? mine : n_points - 1;
    const auto load_vector = [&](const float* base) {
        fvec<D> v;
        static_for<D>(PENC_BODY(k) {
            PENC_INDEX(k); v[k] = base[n * D + k]; });
        return v;
    };
    const auto load_upstream = [&](size_t pair_level, float& g0, float& g1, float& s0, float& s1) {
        if constexpr (kRowMajor) {
            const float2 g = *reinterpret_cast<const float2*>(grad + n * grad_row_stride + 2 * pair_level);
            g0 = g.x;
            g1 = g.y;
        } else {
            g0 = grad[2 * pair_level * n_points + n];
            g1 = grad[(2 * pair_level + 1) * n_points + n];
        }
        if constexpr (kBoth) {
            s0 = second_grad[2 * pair_level * n_points + n];
            s1 = second_grad[(2 * pair_level + 1) * n_points + n];
        }
    };
    const fvec<D> pos = load_vector(positions);
    fvec<D> q = 0.0f;
    if constexpr (kNeedsQ) q = load_vector(double_pos_grad);
    float g0, g1, s0 = 0.0f, s1 = 0.0f;
    load_upstream(static_cast<size_t>(level) * feat_pairs, g0, g1, s0, s1);
    count[tid] = 0u;
    if (tid == 0) repeats = 0u;
    lines.tag[tid] = -1;
    lines.sum[0][tid] = 0.0;
    lines.sum[1][tid] = 0.0;
    const float* const sf = scale_factor + level * D;
    uvec<D + 1> slot;
    fvec<D + 1> w, w2;
    {
        const Located<D> s = locate<D>(pos, random_shift + level * D, sf);
        const uvec<D + 1> h = vertex_hashes<D>(s.rank, s.hash0);
        if constexpr (kOrder == kSecondOrder) {
            w = pos_grad_grad_to_bary<D>(s.rank, q, sf) * w_level;
        } else {
            w = barycentric<D>(s.rank, s.delta) * w_level;
            if constexpr (kBoth) w2 = pos_grad_grad_to_bary<D>(s.rank, q, sf) * w_level;
        }
        static_for<D + 1>(PENC_BODY(r) {
            PENC_INDEX(r);
            slot[r] = to_slot(h[r], capacity, cap_mask);
        });
    }
    const bool ordered = neighbours_share_slots(slot[0], active);
    // (each lane but the last points' against those 16, 32 and 48 away)
    uint32_t same = 0;
#pragma unroll
    for (int away = 16; away < 64; away += 16) {
        const uint32_t other = static_cast<uint32_t>(__shfl_xor(static_cast<int>(slot[0]), away));
        same += __popcll(__ballot((lane & (away == 16 ? 16u : 32u)) == 0u && mine + 48 < n_points && other == slot[0]));
    }
    __syncthreads();  // the counters and lines are cleared
    if (lane == 0 && same != 0u) atomicAdd(&repeats, same);
    __syncthreads();
    // of 768 pairs of lanes, about 768 / (distinct slots) meet, and the level's other vertices have as many slots each: lines for
    // up to 384 slots of a group, which then fit, and as many copies of a slot as leave its lines room (about 300 of 512)
    const uint32_t met = repeats;
    const bool few = met >= 2u * (D + 1) && n_points > kGroupLinesMinPoints;
    uint32_t copies_log2 = 0;
#pragma unroll
    for (uint32_t c = 1; c <= 4; ++c) copies_log2 += 2u * met >= (5u * (D + 1) << c) ? 1u : 0u;
    const uint32_t my_copy = lane & ((1u << copies_log2) - 1u);
    // where each contribution goes: kNone (it has none), kLine | its line, or its place among the group's records
    constexpr uint32_t kNone = 0xFFFFFFFFu, kLine = 0x80000000u;
    uvec<D + 1> to = kNone;
    uint32_t total = 0, line_slot = 0, line_to = kNone;
    const size_t group_at = static_cast<size_t>(level) * sort.n_groups + group;
    const uint32_t slot_mask = (1u << sort.range_shift) - 1u;
#pragma unroll 1
    for (uint32_t pair = 0; pair < feat_pairs; ++pair) {
        const size_t pair_level = static_cast<size_t>(level) * feat_pairs + pair;
        if (pair != 0) {
            load_upstream(pair_level, g0, g1, s0, s1);
            if (few) {
                lines.sum[0][tid] = 0.0;
                lines.sum[1][tid] = 0.0;
                __syncthreads();
            }
        }
        if constexpr (kRowMajor) {
            if (grad_level_major != nullptr && active) {
                grad_level_major[2 * pair_level * n_points + n] = g0;
                grad_level_major[(2 * pair_level + 1) * n_points + n] = g1;
            }
        }
        fvec<D + 1> a0 = w * g0, a1 = w * g1;
        if constexpr (kBoth) {
            a0 += w2 * s0;
            a1 += w2 * s1;
        }
        // (which lanes are folded into which, and which line takes a slot, depends on the slots alone: the same for every pair)
        if (ordered) {
            static_for<D + 1>(PENC_BODY(r) {
                PENC_INDEX(r);
                float x0 = a0[r], x1 = a1[r];
                bool keep = active;
                fold_adjacent_runs(slot[r], keep, x0, x1);
                a0[r] = x0;
                a1[r] = x1;
                if (pair == 0) to[r] = keep ? 0u : kNone;
            });
        } else if (pair == 0) {
            static_for<D + 1>(PENC_BODY(r) {
                PENC_INDEX(r); to[r] = active ? 0u : kNone; });
        }
        float line0 = 0.0f, line1 = 0.0f;
        if (few) {
            static_for<D + 1>(PENC_BODY(r) {
                PENC_INDEX(r);
                if (pair == 0 && to[r] != kNone) {
                    const int want = static_cast<int>((slot[r] << copies_log2) | my_copy);  // slots stay below 2^22
                    uint32_t e = (static_cast<uint32_t>(want) * 0x9E3779B1u) >> (32 - kGroupLinesLog2);
#pragma unroll 1
                    for (uint32_t probe = 0; probe < kGroupProbes; ++probe) {
                        int owner = lines.tag[e];
                        if (owner == -1) owner = atomicCAS(&lines.tag[e], -1, want);
                        if (owner == -1 || owner == want) {
                            to[r] = kLine | e;
                            break;
                        }
                        e = (e + 1u) & (kGroupLines - 1u);
                    }
                }
                if (to[r] != kNone && (to[r] & kLine) != 0u) {
                    const uint32_t e = to[r] & ~kLine;
                    __hip_atomic_fetch_add(&lines.sum[0][e], static_cast<double>(a0[r]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    __hip_atomic_fetch_add(&lines.sum[1][e], static_cast<double>(a1[r]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                }
            });
            __syncthreads();  // all contributions are in
            if (pair == 0) {
                const int tag = lines.tag[tid];
                if (tag != -1) {
                    line_slot = static_cast<uint32_t>(tag) >> copies_log2;
                    line_to = atomicAdd(&count[line_slot >> sort.range_shift], 1u);
                }
            }
            line0 = static_cast<float>(lines.sum[0][tid]);
            line1 = static_cast<float>(lines.sum[1][tid]);
        }
        if (pair == 0) {
            static_for<D + 1>(PENC_BODY(r) {
                PENC_INDEX(r);
                if ((to[r] & kLine) == 0u) to[r] = atomicAdd(&count[slot[r] >> sort.range_shift], 1u);
            });
        }
        __syncthreads();  // the records are counted, the lines read
        if (pair == 0) {
            const uint32_t records = count[tid];
            uint32_t in_wave;
            uint32_t before = wave_exclusive_scan(records, in_wave);
            if (lane == 0) wave_total[wave] = in_wave;
            __syncthreads();
#pragma unroll
            for (uint32_t v = 0; v < kWaves; ++v) {
                const uint32_t t = wave_total[v];
                before += v < wave ? t : 0u;
                total += t;
            }
            count[tid] = before;
            uint16_t* const starts = sort.starts + group_at * (sort.n_ranges + 1);
            if (tid < sort.n_ranges) starts[tid] = static_cast<uint16_t>(before);
            if (tid == 0) starts[sort.n_ranges] = static_cast<uint16_t>(total);
            __syncthreads();
        }
        const auto stage = [&](uint32_t& at, uint32_t of_slot, float v0, float v1) {
            if (pair == 0) {
                at += count[of_slot >> sort.range_shift];
                stage_slots[at] = static_cast<uint16_t>(of_slot & slot_mask);
            }
            RecordValues v;
            v.x = v0;
            v.y = v1;
            stage_values[at] = v;
        };
        static_for<D + 1>(PENC_BODY(r) {
            PENC_INDEX(r);
            uint32_t at = to[r];
            if ((at & kLine) == 0u) stage(at, slot[r], a0[r], a1[r]);
            to[r] = at;
        });
        if (line_to != kNone) stage(line_to, line_slot, line0, line1);
        __syncthreads();
        RecordValues* const values_out = sort.values + (pair_level * sort.n_groups + group) * sort.records;
        for (uint32_t i = tid; i < total; i += kGroupPoints) values_out[i] = stage_values[i];
        if (pair == 0) {
            uint16_t* const slots_out = sort.slots + group_at * sort.records;
            for (uint32_t i = tid; i < total; i += kGroupPoints) slots_out[i] = stage_slots[i];
        }
        if (pair + 1 < feat_pairs) __syncthreads();  // the staged values are read
    }
}

template <int D>
void launch_group_sort(const TableLaunch& t, const GroupSort& sort, uint32_t n_levels) {
#define PENC_LAUNCH(ROWS, ORDER)                                                                                                     \
    hipLaunchKernelGGL((group_sort_kernel<D, ROWS, ORDER>), t.grid, dim3(kGroupPoints), 0, t.stream, t.n_points, n_levels, t.feat_pairs, \
                       t.dies, t.capacity, t.cap_mask, t.positions, t.scale_factor, t.random_shift, t.window, t.grad, t.grad_row_stride, \
                       t.double_pos_grad, t.second_grad, t.grad_level_major, sort)
#define PENC_LAUNCH_ORDER(ROWS)                \
    if (t.second_grad != nullptr) {            \
        PENC_LAUNCH(ROWS, kBothOrders);        \
    } else if (t.second_order) {               \
        PENC_LAUNCH(ROWS, kSecondOrder);       \
    } else {                                   \
        PENC_LAUNCH(ROWS, kFirstOrder);        \
    }
    if (t.rows) {
        PENC_LAUNCH_ORDER(true)
    } else {
        PENC_LAUNCH_ORDER(false)
    }
#undef PENC_LAUNCH_ORDER
#undef PENC_LAUNCH
}

template void launch_group_sort<PENC_DIM>(const TableLaunch& t, const GroupSort& sort, uint32_t n_levels);

template <int D>
void launch_table_backward(const TableLaunch& t) {
    // (a group of points is the same for all instances: half the tiles of twice the points)
#define PENC_LAUNCH(THREADS, BINS, ...)                                                                                                \
    hipLaunchKernelGGL((__VA_ARGS__, BINS, THREADS>), t.grid, dim3(THREADS), 0, t.stream, t.n_points, t.first_level, t.n_pass_levels,  \
                       t.feat_pairs, t.dies, t.tiles_per_group / (THREADS / kScatterBlock), t.capacity, t.cap_mask, t.positions,       \
                       t.scale_factor, t.random_shift, t.window, t.grad, t.grad_row_stride, t.double_pos_grad, t.second_grad,          \
                       t.table_grad, t.grad_level_major, t.bins, ClearTargetOf<BINS>(t.clear))
#define PENC_LAUNCH_WIDTH(KERNEL, ...)                                          \
    if (t.wide_bins) {                                                          \
        PENC_LAUNCH(kScatterBlockManyBins, kBinsWide, KERNEL<D, __VA_ARGS__);   \
    } else if (t.most_bins) {                                                   \
        PENC_LAUNCH(kScatterBlockManyBins, kBinsMany, KERNEL<D, __VA_ARGS__);   \
    } else if (t.many_bins) {                                                   \
        PENC_LAUNCH(kScatterBlock, kBinsMany, KERNEL<D, __VA_ARGS__);           \
    } else if (t.bins.records != nullptr && t.bins.bin_shift < static_cast<uint32_t>(kBinSlotsLog2)) { \
        PENC_LAUNCH(kScatterBlock, kBinsNarrow, KERNEL<D, __VA_ARGS__);         \
    } else {                                                                    \
        PENC_LAUNCH(kScatterBlock, kBinsFew, KERNEL<D, __VA_ARGS__);            \
    }
    if (t.second_grad != nullptr) {
        if (t.rows) {
            PENC_LAUNCH_WIDTH(backward_table_both_kernel, true);
        } else {
            PENC_LAUNCH_WIDTH(backward_table_both_kernel, false);
        }
    } else if (t.second_order) {
        if (t.rows) {
            PENC_LAUNCH_WIDTH(backward_table_kernel, true, true);
        } else {
            PENC_LAUNCH_WIDTH(backward_table_kernel, false, true);
        }
    } else if (t.rows) {
        PENC_LAUNCH_WIDTH(backward_table_kernel, true, false);
    } else {
        PENC_LAUNCH_WIDTH(backward_table_kernel, false, false);
    }
#undef PENC_LAUNCH_WIDTH
#undef PENC_LAUNCH
}

template void launch_table_backward<PENC_DIM>(const TableLaunch& t);

}  // namespace penc
