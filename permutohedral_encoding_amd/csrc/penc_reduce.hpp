// The reducers of the table gradient: they sum the records the scattering kernel has left in its slot-range bins
// (penc_scatter.hpp), or the sorted groups of penc_group_sort.hpp, into the gradient.
#pragma once

#include "penc_group_sort.hpp"
#include "penc_scatter.hpp"

namespace penc {

// Second kernel of stage 2: a workgroup sums the records of one (bin, level) in LDS (fp64,
// ds_add_f64: a few hot slots must not serialise the whole bin, which rules out a compare-and-swap
// loop) and adds the bin's slot range into the gradient.  gridDim.z workgroups share a bin, each
// taking a contiguous range of the scattering workgroups' segments (a launch over few bins and levels would
// otherwise leave most of the chip idle).  Each wavefront takes whole segments, so its loads are
// contiguous.  With one workgroup per bin nothing else touches the bin's slots while this kernel
// runs (the scattering kernel before it has completed, and bins do not overlap), so the final add is
// a plain coalesced read-modify-write; workgroups that share a bin add with atomics (consecutive
// addresses: one request per 64 bytes).
constexpr int reduce_threads(int slots_log2) { return slots_log2 >= 12 ? kReduceBlock : kReduceBlock / 2; }
template <bool kSplit, int kSlotsLog2>  // whether the records are split (the host knows: BinTarget::slots), and the slots per bin
__global__ void __launch_bounds__(reduce_threads(kSlotsLog2))
bin_reduce_kernel(BinTarget pass_bins, const float* __restrict__ window, uint32_t capacity, uint32_t feat_pairs,
                  float* __restrict__ table_grad, int first_level, LateTarget late) {
    constexpr int kSlots = 1 << kSlotsLog2, kThreads = reduce_threads(kSlotsLog2);
    // one array per feature: lanes that hit different slots then spread over all bank pairs (interleaved
    // features would leave every other pair idle in each of the two adds)
    __shared__ double acc0[kSlots];
    __shared__ double acc1[kSlots];
    __shared__ uint32_t wave_ran_over[kThreads / 64];
    const uint32_t bin = blockIdx.x;
    // last level first: with the usual coarse-to-fine level list the bins with the most records are
    // started first and the nearly empty ones fill the tail of the launch
    const uint32_t level_in_pass = gridDim.y - 1 - blockIdx.y;
    // with more than two features per level, every pair of features is scattered and reduced like a level of its own
    const uint32_t pair_level = static_cast<uint32_t>(first_level) + level_in_pass;
    const uint32_t level = pair_level / feat_pairs, pair = pair_level % feat_pairs;
    // With lists of late adds (LateTarget) nobody has cleared the gradient, and nobody else adds to it: the workgroup, alone with its bin,
    // writes all of the bin's slot range.
    const bool whole = kSlotsLog2 == kBinSlotsLog2 && late.kept != nullptr;
    const uint32_t slot0 = bin << kSlotsLog2;
    const GradSlice level_grad{table_grad + (static_cast<size_t>(level) * capacity * feat_pairs + pair) * 2, 2 * feat_pairs, nullptr, 0u, nullptr, nullptr};
    // Its sums, two slots to a store where they lie together (16 bytes of 8-byte alignment).
    const auto write_whole = [&](auto&& sum_of) {
        typedef float Quad __attribute__((ext_vector_type(4), aligned(8)));
        if (feat_pairs == 1u) {
#pragma unroll 2
            for (uint32_t s = 2 * threadIdx.x; s < static_cast<uint32_t>(kSlots); s += 2 * kThreads) {
                const float2 a = sum_of(s), b = sum_of(s + 1);
                float* const to = level_grad.at(slot0 + s);
                if (slot0 + s + 1 < capacity) *reinterpret_cast<Quad*>(to) = Quad{a.x, a.y, b.x, b.y};
                else if (slot0 + s < capacity) *reinterpret_cast<float2*>(to) = a;
            }
        } else {
#pragma unroll 4
            for (uint32_t s = threadIdx.x; s < static_cast<uint32_t>(kSlots); s += kThreads)
                if (slot0 + s < capacity) *reinterpret_cast<float2*>(level_grad.at(slot0 + s)) = sum_of(s);
        }
    };
    const auto write_zeros = [&]() { write_whole([](uint32_t) { return make_float2(0.0f, 0.0f); }); };
    if (window[level] == 0.0f) {  // masked level: its scattering workgroups wrote no counts
        if (whole && feat_pairs == 2u) {
            // half of the bin's slots to each of the level's two pairs of features, whole slots of 16 bytes (forward and table gradient, D = 3, 16 levels of 2^18 slots, the window
            // on 0.4 of them, us: 131072 points along rays 79.0 -> 77.1, 2^18 points 99.6 -> 97.3;  with a fill 76.9 and 97.5)
            typedef float Quad __attribute__((ext_vector_type(4), aligned(8)));
            const uint32_t half0 = slot0 + pair * (kSlots / 2);
            float* const to = table_grad + (static_cast<size_t>(level) * capacity + half0) * 4;
            for (uint32_t s = threadIdx.x; s < static_cast<uint32_t>(kSlots / 2); s += kThreads)
                if (half0 + s < capacity) *reinterpret_cast<Quad*>(to + 4 * s) = Quad{0.0f, 0.0f, 0.0f, 0.0f};
        } else if (whole) {
            write_zeros();
        }
        return;
    }
    const BinTarget bins = bins_of_level(pass_bins, level_in_pass);
    constexpr uint32_t kWaves = kThreads / 64;
    constexpr uint32_t kUnroll = 4;  // even
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const uint32_t per_split = (bins.n_groups + gridDim.z - 1) / gridDim.z;
    const uint32_t group_begin = blockIdx.z * per_split;
    const uint32_t group_end = group_begin + per_split < bins.n_groups ? group_begin + per_split : bins.n_groups;
    const uint32_t* counts = bins.counts + static_cast<size_t>(bin) * bins.n_groups;
    const size_t first = static_cast<size_t>(bin) * bins.n_groups * bins.segment_capacity;  // the bin's first record
    // A bin nothing was appended to (the levels whose scattering workgroups summed in columns, a slot
    // range no point touches) ends here: the look at the counts overlaps the clearing of the sums,
    // and the barrier that follows the clearing carries the vote.
    bool any = false;
    for (uint32_t g = group_begin + threadIdx.x; g < group_end; g += kThreads) any = any || counts[g] != 0u;
    bool ran_over = false;
    if (whole)
        for (uint32_t g = threadIdx.x; g < bins.n_groups; g += kThreads) ran_over = ran_over || counts[g] > bins.segment_capacity;
    ran_over = __any(ran_over);
    if (lane == 0) wave_ran_over[wave] = ran_over ? 1u : 0u;
    for (int s = threadIdx.x; s < kSlots; s += kThreads) {
        acc0[s] = 0.0;
        acc1[s] = 0.0;
    }
    if (!__syncthreads_or(any)) {
        if (whole) write_zeros();
        return;
    }
    // segments g = group_begin + wave, + kWaves, ...; their record counts are fetched 64 at a time
    // (one per lane) so that no segment has to wait for its own count.  The records are walked in
    // chunks of kUnroll wave-widths, and the next chunk's loads are issued before the current
    // chunk's LDS atomics, so a wave always has loads in flight.
    constexpr uint32_t kChunk = 64 * kUnroll;
    // Short segments (a large table has hundreds of bins, so a scattering workgroup leaves only a few
    // dozen records in each): a quarter of the wave per segment, four segments at a time, each taken
    // whole in one step of kShortUnroll loads per lane.
    constexpr uint32_t kShortLanes = 16, kShortUnroll = 8, kShortMax = kShortLanes * kShortUnroll;
    for (uint32_t g0 = group_begin + wave; g0 < group_end; g0 += kWaves * 64) {
        const uint32_t mine = g0 + lane * kWaves;
        const uint32_t wanted = mine < group_end ? counts[mine] : 0u;
        const uint32_t my_count = wanted < bins.segment_capacity ? wanted : bins.segment_capacity;
        const uint32_t n_segments = (group_end - g0 + kWaves - 1) / kWaves < 64u ? (group_end - g0 + kWaves - 1) / kWaves : 64u;
        if (__ballot(my_count > kShortMax) == 0ull) {
            const uint32_t quarter = lane / kShortLanes, l = lane % kShortLanes;
            const uint32_t n_steps = (n_segments + 3) / 4;
            const auto fetch4 = [&](uint32_t step, BinRecord (&rec)[kShortUnroll]) {
                const uint32_t k = 4 * step + quarter;  // < 64; lanes past the last segment hold a count of 0
                const uint32_t count = static_cast<uint32_t>(__shfl(static_cast<int>(my_count), static_cast<int>(k)));
                const uint32_t seg = (g0 + k * kWaves) * bins.segment_capacity;  // within the bin: below 2^29 like the level's records
#pragma unroll
                for (uint32_t u = 0; u < kShortUnroll; ++u) {
                    const uint32_t i = u * kShortLanes + l;
                    // (normal loads: neighbouring short segments share cache lines)
                    rec[u] = load_record<kSplit>(bins, first, i < count ? seg + i : 0u);  // the bin's first record stands in where there is none
                }
                return count;
            };
            BinRecord cur[kShortUnroll], next[kShortUnroll];
            uint32_t cur_count = fetch4(0, cur), next_count = 0;
            for (uint32_t step = 0; step < n_steps; ++step) {
                if (step + 1 < n_steps) next_count = fetch4(step + 1, next);
#pragma unroll
                for (uint32_t u = 0; u < kShortUnroll; ++u)
                    if (u * kShortLanes + l < cur_count) {
                        const uint32_t cell = cur[u].slot_in_bin;
                        __hip_atomic_fetch_add(&acc0[cell], static_cast<double>(cur[u].a0), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                        __hip_atomic_fetch_add(&acc1[cell], static_cast<double>(cur[u].a1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    }
#pragma unroll
                for (uint32_t u = 0; u < kShortUnroll; ++u) cur[u] = next[u];
                cur_count = next_count;
            }
            continue;
        }
        const auto count_of = [&](uint32_t k) { return static_cast<uint32_t>(__builtin_amdgcn_readlane(my_count, k)); };
        // What a lane holds of one chunk, as loaded: split records are read two to a lane (16 bytes of
        // values, 4 of slots: a quarter of the load instructions) and taken apart only when they are
        // added, so that nothing between the loads and the previous chunk's adds waits for them.
        typedef float ValuePair __attribute__((ext_vector_type(4)));
        struct Loaded {
            ValuePair values[kSplit ? kUnroll / 2 : 1];
            uint32_t slots[kSplit ? kUnroll / 2 : 1];
            RecordWords whole[kSplit ? 1 : kUnroll];
        };
        // record u of a lane's kUnroll is record index_of(base, u) of the segment
        const auto index_of = [&](uint32_t base, uint32_t u) {
            return kSplit ? base + ((u >> 1) * 64 + lane) * 2 + (u & 1) : base + u * 64 + lane;
        };
        struct Cursor {
            uint32_t k, base;  // segment (of this wave's n_segments), first record of the chunk
        };
        // (Past the last chunk the loads are issued all the same, from the wave's first segment: with loads
        // behind a branch the compiler cannot tell how many are on their way when the other chunk is added, and
        // makes the adds wait for all of them.)
        const auto fetch = [&](const Cursor& at, Loaded& got) {
            const bool any = at.k < n_segments;
            const uint32_t count = any ? count_of(at.k) : 0u;
            const size_t seg = first + (g0 + (any ? at.k : 0u) * kWaves) * bins.segment_capacity;
            if constexpr (kSplit) {
                const RecordValues* values = static_cast<const RecordValues*>(bins.records) + seg;  // 16-byte aligned:
                const uint16_t* slots = bins.slots + seg;                                         // segments are multiples of four records
#pragma unroll
                for (uint32_t u = 0; u < kUnroll; u += 2) {
                    const uint32_t i = index_of(at.base, u);
                    const uint32_t from = i < count ? i : 0u;  // even; an odd count's last pair reads one record of the segment's slack
                    got.values[u / 2] = __builtin_nontemporal_load(reinterpret_cast<const ValuePair*>(values + from));
                    got.slots[u / 2] = __builtin_nontemporal_load(reinterpret_cast<const uint32_t*>(slots + from));
                }
            } else {
                const BinRecord* recs = static_cast<const BinRecord*>(bins.records) + seg;
#pragma unroll
                for (uint32_t u = 0; u < kUnroll; ++u) {
                    const uint32_t i = index_of(at.base, u);
                    got.whole[u] = __builtin_nontemporal_load(reinterpret_cast<const RecordWords*>(recs + (i < count ? i : 0u)));
                }
            }
        };
        const auto add = [&](const Cursor& at, const Loaded& got) {
            const uint32_t count = count_of(at.k);
#pragma unroll
            for (uint32_t u = 0; u < kUnroll; ++u) {
                uint32_t cell;
                float a0, a1;
                if constexpr (kSplit) {
                    const ValuePair v = got.values[u / 2];
                    const float v0 = v.x, v1 = v.y, v2 = v.z, v3 = v.w;  // copies first: a bit cast applied directly to a vector element reads element 0
                    cell = (u & 1) ? got.slots[u / 2] >> 16 : got.slots[u / 2] & 0xFFFFu;
                    a0 = (u & 1) ? v2 : v0;
                    a1 = (u & 1) ? v3 : v1;
                } else {
                    const RecordWords w = got.whole[u];
                    const uint32_t w0 = w.x, w1 = w.y, w2 = w.z;
                    cell = w0;
                    a0 = __builtin_bit_cast(float, w1);
                    a1 = __builtin_bit_cast(float, w2);
                }
                if (index_of(at.base, u) < count) {
                    __hip_atomic_fetch_add(&acc0[cell], static_cast<double>(a0), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    __hip_atomic_fetch_add(&acc1[cell], static_cast<double>(a1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                }
            }
        };
        // the chunk after `at`: the next kChunk records of its segment, or the start of the next segment that has any
        const auto after = [&](Cursor at) {
            at.base += kChunk;
            if (at.base >= count_of(at.k)) {
                at.base = 0;
                do ++at.k; while (at.k < n_segments && count_of(at.k) == 0u);
            }
            return at;
        };
        // two sets of registers take turns, so a chunk's loads stay in flight over the other chunk's adds
        Cursor a{0u, 0u};
        while (a.k < n_segments && count_of(a.k) == 0u) ++a.k;
        Loaded got_a, got_b;
        if (a.k < n_segments) fetch(a, got_a);
        while (a.k < n_segments) {
            const Cursor b = after(a);
            fetch(b, got_b);
            add(a, got_a);
            if (b.k >= n_segments) break;
            a = after(b);
            fetch(a, got_a);
            add(b, got_b);
        }
    }
    if (whole) {
        // Late adds: of this bin where its segment was to have more records than it has room for, in the list of that group, with others.  A full bin's reducer is what
        // the launch waits for: eight loads on their way at once.  (Every list of the level by every reducer, a load at a time -> so, forward and table gradient, us: D = 3, 24 levels
        // of 2^18 slots, a third of the points in one simplex, 2^18 points 518 -> 397, 2^20 2011 -> 1493;  D = 8, 16 levels of 2^19, three quarters of 131072 points in a small
        // box 403 -> 349.  With a fill and direct adds 1389, 5571 and 598.)
        bool any_ran_over = false;
#pragma unroll
        for (uint32_t w = 0; w < kWaves; ++w) any_ran_over = any_ran_over || wave_ran_over[w] != 0u;
        if (any_ran_over) {
            constexpr uint32_t kAtOnce = 8;
            for (uint32_t g = wave; g < bins.n_groups; g += kWaves) {
                if (counts[g] <= bins.segment_capacity) continue;
                const size_t list = static_cast<size_t>(level_in_pass) * bins.n_groups + g;
                const BinRecord* const kept = late.kept + list * late.room;
                const uint32_t count = late.counts[list];
                for (uint32_t base = 0; base < count; base += 64 * kAtOnce) {
                    BinRecord rec[kAtOnce];
#pragma unroll
                    for (uint32_t u = 0; u < kAtOnce; ++u) {
                        const uint32_t i = base + u * 64 + lane;
                        rec[u] = kept[i < count ? i : 0u];
                    }
#pragma unroll
                    for (uint32_t u = 0; u < kAtOnce; ++u) {
                        const uint32_t cell = rec[u].slot_in_bin - slot0;  // (a late add's slot is that in the level)
                        if (base + u * 64 + lane < count && cell < static_cast<uint32_t>(kSlots)) {
                            __hip_atomic_fetch_add(&acc0[cell], static_cast<double>(rec[u].a0), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                            __hip_atomic_fetch_add(&acc1[cell], static_cast<double>(rec[u].a1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                        }
                    }
                }
            }
        }
        __syncthreads();
        write_whole([&](uint32_t s) { return make_float2(static_cast<float>(acc0[s]), static_cast<float>(acc1[s])); });
        return;
    }
    // nothing has been added to the bin's slots since the gradient was cleared (or, for a caller who keeps the gradient
    // across calls, since that caller last cleared this slot range): the sums are the result.  Read before the barrier:
    // thread 0 sets the flag at the end.
    const bool untouched_so_far = bins.direct[bin] == 0u;
    __syncthreads();
    const bool alone = gridDim.z == 1;
    if (alone) {
        // all of a thread's read-modify-writes at once: the loads are issued together, not one per trip
        constexpr int kMine = kSlots / kThreads;
        float2 sum[kMine], g[kMine];
        bool touched[kMine];
#pragma unroll
        for (int k = 0; k < kMine; ++k) {
            const uint32_t s = static_cast<uint32_t>(k) * kThreads + threadIdx.x;
            const double v0 = acc0[s], v1 = acc1[s];
            sum[k] = make_float2(static_cast<float>(v0), static_cast<float>(v1));
            touched[k] = (v0 != 0.0 || v1 != 0.0) && slot0 + s < capacity;
        }
#pragma unroll
        for (int k = 0; k < kMine; ++k) {
            const uint32_t s = static_cast<uint32_t>(k) * kThreads + threadIdx.x;
            g[k] = make_float2(0.0f, 0.0f);
            if (touched[k] && !untouched_so_far) g[k] = *reinterpret_cast<const float2*>(level_grad.at(slot0 + s));
        }
#pragma unroll
        for (int k = 0; k < kMine; ++k) {
            const uint32_t s = static_cast<uint32_t>(k) * kThreads + threadIdx.x;
            if (touched[k]) {
                g[k].x += sum[k].x;
                g[k].y += sum[k].y;
                *reinterpret_cast<float2*>(level_grad.at(slot0 + s)) = g[k];
            }
        }
        if (threadIdx.x == 0 && untouched_so_far) bins.direct[bin] = 1u;  // this slot range now holds sums
        return;
    }
    if (threadIdx.x == 0 && untouched_so_far) bins.direct[bin] = 1u;  // (the workgroups that share the bin all store the same value)
    // Both features of a slot by two neighbouring lanes, so that an instruction's adds fall into half as many 64-byte segments (16 levels
    // of 2^16 slots, four features, 2^18 points: 48 -> 34 us).
    const double* const acc = (threadIdx.x & 1u) != 0u ? acc1 : acc0;
#pragma unroll 4
    for (uint32_t s = threadIdx.x >> 1; s < static_cast<uint32_t>(kSlots); s += kThreads / 2) {
        const double v = acc[s];
        if (v != 0.0 && slot0 + s < capacity) global_add(level_grad.at(slot0 + s) + (threadIdx.x & 1u), static_cast<float>(v));
    }
}

// Adds what a scattering kernel that cleared the gradient has kept (ClearTarget::kept): a workgroup to a group of points and a level.
__global__ void __launch_bounds__(kBlock)
add_deferred_kernel(ClearTarget clear, const float* __restrict__ window, uint32_t capacity, uint32_t feat_pairs, float* __restrict__ table_grad) {
    const uint32_t group = blockIdx.x, pair_level = blockIdx.y, level = pair_level / feat_pairs, pair = pair_level % feat_pairs;
    if (window[level] == 0.0f) return;  // masked level: its scattering workgroups wrote no counts
    const size_t list = static_cast<size_t>(pair_level) * gridDim.x + group;
    const uint32_t count = clear.counts[list];
    const BinRecord* const kept = clear.kept + list * clear.room;
    const GradSlice level_grad{table_grad + (static_cast<size_t>(level) * capacity * feat_pairs + pair) * 2, 2 * feat_pairs, nullptr, 0u, nullptr, nullptr};
    for (uint32_t first = 0; first < count; first += kBlock) {
        const uint32_t i = first + threadIdx.x;
        BinRecord rec{0u, 0.0f, 0.0f};
        if (i < count) rec = kept[i];
        global_add_pairs(level_grad, i < count, rec.slot_in_bin, rec.a0, rec.a1);
    }
}

// The reducer of tables with hundreds of bins.  There a scattering workgroup leaves only a few
// dozen records in each of its segments and a (bin, level) has a few thousand in all, so a workgroup of
// bin_reduce_kernel is a chain of latencies (launch, counts, records, gradient) with nothing to overlap
// them: its 128 KiB of sums allow one workgroup per compute unit.  Here a workgroup keeps its bin and walks
// several levels (blockIdx.y, + gridDim.y, ...): the counts of all its levels are fetched at once and kept in LDS
// (levels that left no records cost nothing more), and over the sequence of (level, 64 segments)
// steps that remain the records are fetched two steps ahead of the adds.
// What it would wait for otherwise is its own stores: a wait for records counts every memory operation issued after them, and how
// many stores a write-out makes is not known when the code is compiled, so a wait that follows a write-out waits for the stores as well, a trip
// to memory for every level.  So the next step's records are waited for before the write-out, and those of the step after it
// are on their way over it.
// (16 live levels of 2^22 slots, 2^20 points near a surface, 340 MB of records: 152 -> 134 us; 200001 points 80 -> 63 us; 8 levels of random
// slots, 49 segments of 32 records 98 -> 95, 128 of 64 207 -> 212, of which the records alone 123 -> 87.)
// A wave reads four segments at a time, their records counted through, so that every lane of a load has one (with a quarter of the
// wave to a segment of 64 records in room for 101 half of the lanes had none).  Needs segments of at
// most kLevelsMaxSegment records, whole (12-byte) records, at most kReduceBlock groups and
// at most kLevelsMaxPerWorkgroup levels per workgroup (the host checks all four).
constexpr uint32_t kLevelsUnroll = 6, kLevelsShortUnroll = 3;
constexpr uint32_t kLevelsMaxSegment = 128, kLevelsShortSegment = 64;
constexpr uint32_t kLevelsMaxPerWorkgroup = 24;
static_assert(kLevelsMaxSegment < 256, "a segment's count is kept in a byte");
template <uint32_t kUnroll>
__global__ void __launch_bounds__(kReduceBlock)
bin_reduce_levels_kernel(BinTarget pass_bins, const float* __restrict__ window, uint32_t capacity, uint32_t feat_pairs,
                         float* __restrict__ table_grad, int first_level, uint32_t n_levels_in_pass) {
    __shared__ __align__(16) double acc0[kBinSlots];
    __shared__ __align__(16) double acc1[kBinSlots];
    __shared__ __align__(4) uint8_t counts[kLevelsMaxPerWorkgroup][kReduceBlock];  // records of the workgroup's i-th level in each group's segment
    __shared__ uint32_t masks[2];  // bit i: the workgroup's i-th level [0] has records in this bin, [1] got direct adds in this bin's slots
    const uint32_t bin = blockIdx.x, my_first = blockIdx.y, my_stride = gridDim.y;
    const uint32_t n_mine = (n_levels_in_pass - my_first + my_stride - 1) / my_stride;  // blockIdx.y < n_levels_in_pass
    const uint32_t n_bins = pass_bins.n_bins, n_groups = pass_bins.n_groups, seg_cap = pass_bins.segment_capacity;
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    // the workgroup's i-th level within the pass, and where its segments of this bin start (counted in segments)
    const auto level_in_pass = [&](uint32_t i) { return my_first + i * my_stride; };
    const auto first_segment = [&](uint32_t i) { return (static_cast<size_t>(level_in_pass(i)) * n_bins + bin) * n_groups; };
    if (threadIdx.x < 2) masks[threadIdx.x] = 0u;
    for (int s = threadIdx.x; s < kBinSlots; s += kReduceBlock) {
        acc0[s] = 0.0;
        acc1[s] = 0.0;
    }
    // which of the levels have records here (thread g looks at group g's count of every level, all loads at once)
    uint32_t seen[kLevelsMaxPerWorkgroup];
#pragma unroll
    for (uint32_t i = 0; i < kLevelsMaxPerWorkgroup; ++i) {
        seen[i] = 0u;
        if (i < n_mine) {
            const uint32_t pair_level = static_cast<uint32_t>(first_level) + level_in_pass(i);
            // (a masked level's scattering workgroups wrote no counts)
            if (window[pair_level / feat_pairs] != 0.0f && threadIdx.x < n_groups) seen[i] = pass_bins.counts[first_segment(i) + threadIdx.x];
        }
    }
    uint32_t direct = 0u;
    if (threadIdx.x < n_mine) direct = pass_bins.direct[static_cast<size_t>(level_in_pass(threadIdx.x)) * n_bins + bin];
    __syncthreads();  // the masks are cleared
    uint32_t found = 0u;
#pragma unroll
    for (uint32_t i = 0; i < kLevelsMaxPerWorkgroup; ++i) {
        if (i < n_mine) counts[i][threadIdx.x] = static_cast<uint8_t>(seen[i]);
        if (__ballot(seen[i] != 0u) != 0ull) found |= 1u << i;
    }
    if (lane == 0 && found != 0u) atomicOr(&masks[0], found);
    if (direct != 0u) atomicOr(&masks[1], 1u << threadIdx.x);
    __syncthreads();
    const uint32_t todo = masks[0], direct_mask = masks[1];
    if (todo == 0u) return;

    // a step: 64 segments of one level, four to a wave
    constexpr uint32_t kEnd = 32;
    // Bins wider than the LDS sums (tables above 2^22 slots) are summed one range of kBinSlots slots after
    // the other: every range walks all the bin's records and takes those that fall into it.
    const uint32_t n_ranges = 1u << (pass_bins.bin_shift - kBinSlotsLog2);
    struct Cursor {
        uint32_t i, range, step;  // the workgroup's i-th level (kEnd: past the last), the range of the bin, segments 64 * step ...
    };
    const uint32_t n_steps = (n_groups + 63) / 64;
    const auto after = [&](Cursor at) {
        if (at.i == kEnd || ++at.step < n_steps) return at;
        at.step = 0u;
        if (++at.range < n_ranges) return at;
        const uint32_t rest = at.i + 1 < 32 ? todo >> (at.i + 1) : 0u;
        return Cursor{rest != 0u ? at.i + 1 + static_cast<uint32_t>(__builtin_ctz(rest)) : kEnd, 0u, 0u};
    };
    struct Loaded {
        RecordWords rec[kUnroll];
        uint32_t total, range, counts4;
    };
    const BinRecord* const records = static_cast<const BinRecord*>(pass_bins.records);
    // Record j of the wave's four segments, counted through, in the order of the segments.
    const auto index_of = [&](uint32_t counts4, uint32_t j) {
        const uint32_t c0 = counts4 & 255u, c1 = (counts4 >> 8) & 255u, c2 = (counts4 >> 16) & 255u;
        uint32_t i = j;
        i += j >= c0 ? seg_cap - c0 : 0u;
        i += j >= c0 + c1 ? seg_cap - c1 : 0u;
        i += j >= c0 + c1 + c2 ? seg_cap - c2 : 0u;
        return i;
    };
    // (Every load is issued whether or not its result is wanted, from an address that is valid
    // either way: with loads behind branches the compiler cannot tell how many are on their way and
    // makes every use wait for all of them, those of the next step included.)
    const auto fetch = [&](const Cursor& at, Loaded& got) {
        const uint32_t i = at.i != kEnd ? at.i : 0u, g = at.step * 64 + wave * 4;  // (the counts reach to the end of the last step)
        uint32_t counts4 = *reinterpret_cast<const uint32_t*>(&counts[i][g]);
        counts4 = at.i != kEnd ? __builtin_amdgcn_readfirstlane(counts4) : 0u;
        got.counts4 = counts4;
        got.total = (counts4 & 255u) + ((counts4 >> 8) & 255u) + ((counts4 >> 16) & 255u) + (counts4 >> 24);
        got.range = at.range;
        const BinRecord* seg = records + (first_segment(i) + g) * seg_cap;
#pragma unroll
        for (uint32_t u = 0; u < kUnroll; ++u) {
            const uint32_t j = u * 64 + lane;
            got.rec[u] = *reinterpret_cast<const RecordWords*>(j < got.total ? seg + index_of(counts4, j) : records);
        }
    };
    // waits for a step's records
    const auto arrive = [&](Loaded& got) {
#pragma unroll
        for (uint32_t u = 0; u < kUnroll; ++u) asm volatile("" : "+v"(got.rec[u]));
    };
    const auto add_one = [&](const RecordWords& w, uint32_t range) {
        const uint32_t w0 = w.x, w1 = w.y, w2 = w.z;  // copies first: a bit cast applied directly to a vector element reads element 0
        if ((w0 >> kBinSlotsLog2) != range) return;
        const uint32_t cell = w0 & (kBinSlots - 1);
        __hip_atomic_fetch_add(&acc0[cell], static_cast<double>(__builtin_bit_cast(float, w1)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        __hip_atomic_fetch_add(&acc1[cell], static_cast<double>(__builtin_bit_cast(float, w2)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    };
    const auto add = [&](const Cursor& at, const Loaded& got) {
#pragma unroll
        for (uint32_t u = 0; u < kUnroll; ++u)
            if (u * 64 + lane < got.total) add_one(got.rec[u], got.range);
        // (more records than the registers take are rare: a segment's share is its mean)
        if (got.total > kUnroll * 64) {
            const BinRecord* seg = records + (first_segment(at.i) + at.step * 64 + wave * 4) * seg_cap;
            for (uint32_t j = kUnroll * 64 + lane; j < got.total; j += 64)
                add_one(*reinterpret_cast<const RecordWords*>(seg + index_of(got.counts4, j)), got.range);
        }
    };
    // Adds the sums of one range of the bin at the workgroup's i-th level into the gradient and clears them; waits for the records of
    // `next` in between.  Nothing else touches the bin's slots of that level while this kernel runs, so the add is a plain
    // read-modify-write, or a store where nothing was added since the gradient was cleared.  Two slots to a thread at a time.
    typedef double Pair __attribute__((ext_vector_type(2)));
    typedef float Quad __attribute__((ext_vector_type(4), aligned(8)));  // (the gradient is aligned to 8 bytes)
    const auto flush = [&](uint32_t i, uint32_t range, Loaded& next) {
        lds_barrier();
        const uint32_t pair_level = static_cast<uint32_t>(first_level) + level_in_pass(i);
        const uint32_t level = pair_level / feat_pairs, pair = pair_level % feat_pairs;
        const GradSlice level_grad{table_grad + (static_cast<size_t>(level) * capacity * feat_pairs + pair) * 2, 2 * feat_pairs, nullptr, 0u, nullptr, nullptr};
        const uint32_t slot0 = (bin << pass_bins.bin_shift) + (range << kBinSlotsLog2);
        const bool untouched_so_far = ((direct_mask >> i) & 1u) == 0u;
        constexpr int kMine = kBinSlots / kReduceBlock / 2;
        Pair v0[kMine], v1[kMine];
#pragma unroll
        for (int k = 0; k < kMine; ++k) {
            const uint32_t at = static_cast<uint32_t>(k) * kReduceBlock + threadIdx.x;
            v0[k] = reinterpret_cast<const Pair*>(acc0)[at];
            v1[k] = reinterpret_cast<const Pair*>(acc1)[at];
        }
        arrive(next);
        if (threadIdx.x == 0 && untouched_so_far) pass_bins.direct[static_cast<size_t>(level_in_pass(i)) * n_bins + bin] = 1u;  // this slot range now holds sums
#pragma unroll
        for (int k = 0; k < kMine; ++k) {
            const uint32_t at = static_cast<uint32_t>(k) * kReduceBlock + threadIdx.x, slot = slot0 + 2 * at;
            const bool one = v0[k].x != 0.0 || v1[k].x != 0.0, two = v0[k].y != 0.0 || v1[k].y != 0.0;
            if (!one && !two) continue;
            reinterpret_cast<Pair*>(acc0)[at] = Pair{0.0, 0.0};
            reinterpret_cast<Pair*>(acc1)[at] = Pair{0.0, 0.0};
            Quad sum = {static_cast<float>(v0[k].x), static_cast<float>(v1[k].x), static_cast<float>(v0[k].y), static_cast<float>(v1[k].y)};
            if (untouched_so_far && feat_pairs == 1u && slot + 1 < capacity) {  // (a slot without sums holds zeros)
                *reinterpret_cast<Quad*>(level_grad.at(slot)) = sum;
                continue;
            }
            if (one && slot < capacity) {
                float2* const cell = reinterpret_cast<float2*>(level_grad.at(slot));
                const float2 g = untouched_so_far ? make_float2(0.0f, 0.0f) : *cell;
                *cell = make_float2(g.x + sum.x, g.y + sum.y);
            }
            if (two && slot + 1 < capacity) {
                float2* const cell = reinterpret_cast<float2*>(level_grad.at(slot + 1));
                const float2 g = untouched_so_far ? make_float2(0.0f, 0.0f) : *cell;
                *cell = make_float2(g.x + sum.z, g.y + sum.w);
            }
        }
        lds_barrier();
    };
    // three sets of registers take turns for the records; past the last step the loads fetch the stand-in
    Cursor it0{static_cast<uint32_t>(__builtin_ctz(todo)), 0u, 0u};
    Cursor it1 = after(it0), it2 = after(it1);
    Loaded a, b, c;
    fetch(it0, a);
    fetch(it1, b);
    const auto turn = [&](Loaded& now, Loaded& next, Loaded& last) {
        fetch(it2, last);
        add(it0, now);
        if (it1.i != it0.i || it1.range != it0.range) flush(it0.i, it0.range, next);
        it0 = it1;
        it1 = it2;
        it2 = after(it2);
        return it0.i != kEnd;
    };
    while (turn(a, b, c) && turn(b, c, a) && turn(c, a, b)) {
    }
}

// A workgroup takes one slot range of one pair of features: every reader of `lanes` threads sums the range's stretches of its groups
// of points, then the range is written.  (Workgroups that stay and take one range after the other, their stores on the way while
// the next is summed, were slower: 2^15 points 29.7 us instead of 20.6; 8192-slot ranges, one workgroup per compute unit, 24.)
// `touched` (the sparse entry points; nullptr otherwise): nothing is written where a range got no record, sums are added where the
// caller's map says that the range's bin holds anything, and the map is marked.
constexpr int kRangeBlock = 1024;
__global__ void __launch_bounds__(kRangeBlock)
range_sum_kernel(GroupSort sort, const float* __restrict__ window, uint32_t capacity, uint32_t feat_pairs, uint32_t n_levels,
                 uint32_t lanes_log2, uint32_t dies, uint32_t* __restrict__ touched, uint32_t bins_per_level, uint32_t bin_shift,
                 float* __restrict__ table_grad) {
    extern __shared__ double sums[];  // [2][slots per range]
    // the pairs of a range, whose slots share cache lines, on one die and side by side
    const uint32_t j = blockIdx.x / dies, at_range = j / feat_pairs * dies + blockIdx.x % dies;
    if (at_range >= n_levels * sort.n_ranges) return;
    const uint32_t pair = j % feat_pairs, range = at_range % sort.n_ranges, level = at_range / sort.n_ranges;
    const uint32_t slots = 1u << sort.range_shift, slot0 = range << sort.range_shift;
    const uint32_t readers = kRangeBlock >> lanes_log2, lanes = 1u << lanes_log2;
    const uint32_t reader = threadIdx.x >> lanes_log2, l = threadIdx.x & (lanes - 1);
    const auto stretch = [&](uint32_t g, uint32_t& first, uint32_t& end) {
        const uint16_t* const s = sort.starts + (static_cast<size_t>(level) * sort.n_groups + (g < sort.n_groups ? g : 0u)) * (sort.n_ranges + 1) + range;
        first = s[0];
        end = s[1];
    };
    // (the first look at where the records are overlaps the look at the window and the clearing of the sums; of a masked level
    // it reads what nobody has written, and the result is not used)
    uint32_t first, end;
    stretch(reader, first, end);
    float* const out = table_grad + (static_cast<size_t>(level) * capacity * feat_pairs + pair) * 2;
    if (window[level] == 0.0f) {
        if (touched != nullptr) return;
        for (uint32_t s = threadIdx.x; s < slots && slot0 + s < capacity; s += kRangeBlock)
            *reinterpret_cast<float2*>(out + static_cast<size_t>(slot0 + s) * 2 * feat_pairs) = make_float2(0.0f, 0.0f);
        return;
    }
    double* const acc0 = sums;
    double* const acc1 = sums + slots;
    for (uint32_t s = threadIdx.x; s < slots; s += kRangeBlock) {
        acc0[s] = 0.0;
        acc1[s] = 0.0;
    }
    bool any = false;
    __syncthreads();
    for (uint32_t g = reader; g < sort.n_groups; g += readers) {
        if (g != reader) stretch(g, first, end);
        any = any || end > first;
        const uint16_t* const slot_of = sort.slots + (static_cast<size_t>(level) * sort.n_groups + g) * sort.records;
        const RecordValues* const value_of = sort.values + ((static_cast<size_t>(level) * feat_pairs + pair) * sort.n_groups + g) * sort.records;
        constexpr uint32_t kTogether = 4;
        for (uint32_t k = first + l; k < end; k += kTogether * lanes) {
            uint32_t cell[kTogether];
            RecordValues v[kTogether];
#pragma unroll
            for (uint32_t u = 0; u < kTogether; ++u) {
                const uint32_t at = k + u * lanes < end ? k + u * lanes : k;
                cell[u] = slot_of[at];
                v[u] = value_of[at];
            }
#pragma unroll
            for (uint32_t u = 0; u < kTogether; ++u) {
                if (k + u * lanes < end) {
                    __hip_atomic_fetch_add(&acc0[cell[u]], static_cast<double>(v[u].x), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    __hip_atomic_fetch_add(&acc1[cell[u]], static_cast<double>(v[u].y), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                }
            }
        }
    }
    uint32_t* flag = nullptr;
    bool holds_sums = false;
    if (touched != nullptr) {
        flag = touched + (static_cast<size_t>(level) * feat_pairs + pair) * bins_per_level + (slot0 >> bin_shift);
        holds_sums = *flag != 0u;
        if (!__syncthreads_or(any)) return;
    } else {
        __syncthreads();
    }
    for (uint32_t s = threadIdx.x; s < slots; s += kRangeBlock) {
        if (slot0 + s >= capacity) break;
        float2* const cell = reinterpret_cast<float2*>(out + static_cast<size_t>(slot0 + s) * 2 * feat_pairs);
        float2 sum = make_float2(static_cast<float>(acc0[s]), static_cast<float>(acc1[s]));
        if (holds_sums) {
            const float2 before = *cell;
            sum.x += before.x;
            sum.y += before.y;
        }
        *cell = sum;
    }
    // (ranges that share a bin each see the flag set or not: where it was not, the gradient is zero and adding to it is the same)
    if (flag != nullptr && threadIdx.x == 0) *flag = 1u;
}

}  // namespace penc
