// The reducers of the table gradient: they sum the records the scattering kernel has left in its slot-range bins
// (penc_scatter.hpp), or the sorted groups of penc_group_sort.hpp, into the gradient.
#pragma once

#include "penc_group_sort.hpp"
#include "penc_scatter.hpp"

namespace penc {

// Second kernel of stage 2: a workgroup sums the records of one (bin, level) in LDS (fp64,
// ds_add_f64: a few hot slots must not serialise the whole bin, which rules out a compare-and-swap
// loop) and adds the bin's slot range into the gradient.  gridDim.z workgroups share a bin, each
// taking a contiguous range of the scattering workgroups' segments (a launch over few levels would
// otherwise leave most of the chip idle).  Each wavefront takes whole segments, so its loads are
// contiguous.  With one workgroup per bin nothing else touches the bin's slots while this kernel
// runs (the scattering kernel before it has completed, and bins do not overlap), so the final add is
// a plain coalesced read-modify-write; workgroups that share a bin add with atomics (consecutive
// addresses: one request per 64 bytes).
template <bool kSplit>  // whether the records are split (the host knows: BinTarget::slots)
__global__ void __launch_bounds__(kReduceBlock)
bin_reduce_kernel(BinTarget pass_bins, const float* __restrict__ window, uint32_t capacity, uint32_t feat_pairs,
                  float* __restrict__ table_grad, int first_level) {
    // one array per feature: lanes that hit different slots then spread over all bank pairs (interleaved
    // features would leave every other pair idle in each of the two adds)
    __shared__ double acc0[kBinSlots];
    __shared__ double acc1[kBinSlots];
    const uint32_t bin = blockIdx.x;
    // last level first: with the usual coarse-to-fine level list the bins with the most records are
    // started first and the nearly empty ones fill the tail of the launch
    const uint32_t level_in_pass = gridDim.y - 1 - blockIdx.y;
    // with more than two features per level, every pair of features is scattered and reduced like a level of its own
    const uint32_t pair_level = static_cast<uint32_t>(first_level) + level_in_pass;
    const uint32_t level = pair_level / feat_pairs, pair = pair_level % feat_pairs;
    if (window[level] == 0.0f) return;  // masked level: its scattering workgroups wrote no counts
    const BinTarget bins = bins_of_level(pass_bins, level_in_pass);
    constexpr uint32_t kWaves = kReduceBlock / 64;
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
    for (uint32_t g = group_begin + threadIdx.x; g < group_end; g += kReduceBlock) any = any || counts[g] != 0u;
    for (int s = threadIdx.x; s < kBinSlots; s += kReduceBlock) {
        acc0[s] = 0.0;
        acc1[s] = 0.0;
    }
    if (!__syncthreads_or(any)) return;
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
        const uint32_t my_count = mine < group_end ? counts[mine] : 0u;
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
    // nothing has been added to the bin's slots since the gradient was cleared (or, for a caller who keeps the gradient
    // across calls, since that caller last cleared this slot range): the sums are the result.  Read before the barrier:
    // thread 0 sets the flag at the end.
    const bool untouched_so_far = bins.direct[bin] == 0u;
    __syncthreads();
    const GradSlice level_grad{table_grad + (static_cast<size_t>(level) * capacity * feat_pairs + pair) * 2, 2 * feat_pairs, nullptr, 0u};
    const uint32_t slot0 = bin << kBinSlotsLog2;  // (this kernel serves bins of kBinSlots slots only)
    const bool alone = gridDim.z == 1;
    if (alone) {
        // all of a thread's read-modify-writes at once: the loads are issued together, not one per trip
        constexpr int kMine = kBinSlots / kReduceBlock;
        float2 sum[kMine], g[kMine];
        bool touched[kMine];
#pragma unroll
        for (int k = 0; k < kMine; ++k) {
            const uint32_t s = static_cast<uint32_t>(k) * kReduceBlock + threadIdx.x;
            const double v0 = acc0[s], v1 = acc1[s];
            sum[k] = make_float2(static_cast<float>(v0), static_cast<float>(v1));
            touched[k] = (v0 != 0.0 || v1 != 0.0) && slot0 + s < capacity;
        }
#pragma unroll
        for (int k = 0; k < kMine; ++k) {
            const uint32_t s = static_cast<uint32_t>(k) * kReduceBlock + threadIdx.x;
            g[k] = make_float2(0.0f, 0.0f);
            if (touched[k] && !untouched_so_far) g[k] = *reinterpret_cast<const float2*>(level_grad.at(slot0 + s));
        }
#pragma unroll
        for (int k = 0; k < kMine; ++k) {
            const uint32_t s = static_cast<uint32_t>(k) * kReduceBlock + threadIdx.x;
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
    for (uint32_t s = threadIdx.x; s < static_cast<uint32_t>(kBinSlots); s += kReduceBlock) {
        const double v0 = acc0[s], v1 = acc1[s];
        if ((v0 != 0.0 || v1 != 0.0) && slot0 + s < capacity) {
            float2* cell = reinterpret_cast<float2*>(level_grad.at(slot0 + s));
            global_add(&cell->x, static_cast<float>(v0));
            global_add(&cell->y, static_cast<float>(v1));
        }
    }
}

// The reducer of tables with hundreds of bins.  There a scattering workgroup leaves only a few
// dozen records in each of its segments and a (bin, level) has a few thousand in all, so a workgroup of
// bin_reduce_kernel is a chain of latencies (launch, counts, records, gradient) with nothing to overlap
// them: its 128 KiB of sums allow one workgroup per compute unit.  Here a workgroup keeps its bin and walks
// several levels (blockIdx.y, + gridDim.y, ...): the counts of all its levels are fetched at once
// (levels that left no records cost nothing more), and over the sequence of (level, 64 segments)
// steps that remain the counts are fetched two steps and the records one step ahead of the adds, so the
// loads of the next level are in flight while this level's sums are added and written out
// (measured on a 2^22-slot table, 16 levels, per call: bin_reduce_kernel 0.207 ms; this kernel 0.170 ms;
// with every load issued unconditionally, LDS-only barriers and a store-only write-out, so that nothing
// waits for the loads of the next step, 0.157 ms; with one workgroup per bin instead of two 0.146 ms).
// A quarter of a wave reads a segment, kLevelsShortUnroll records per lane: needs segments of at
// most kLevelsMaxSegment records, whole (12-byte) records, at most kReduceBlock groups and
// at most kLevelsMaxPerWorkgroup levels per workgroup (the host checks all four).
constexpr uint32_t kLevelsShortLanes = 16, kLevelsShortUnroll = 8;
constexpr uint32_t kLevelsMaxSegment = kLevelsShortLanes * kLevelsShortUnroll;
constexpr uint32_t kLevelsMaxPerWorkgroup = 24;
__global__ void __launch_bounds__(kReduceBlock)
bin_reduce_levels_kernel(BinTarget pass_bins, const float* __restrict__ window, uint32_t capacity, uint32_t feat_pairs,
                         float* __restrict__ table_grad, int first_level, uint32_t n_levels_in_pass) {
    __shared__ double acc0[kBinSlots];
    __shared__ double acc1[kBinSlots];
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
    for (uint32_t i = 0; i < kLevelsMaxPerWorkgroup; ++i)
        if (__ballot(seen[i] != 0u) != 0ull) found |= 1u << i;
    if (lane == 0 && found != 0u) atomicOr(&masks[0], found);
    if (direct != 0u) atomicOr(&masks[1], 1u << threadIdx.x);
    __syncthreads();
    const uint32_t todo = masks[0], direct_mask = masks[1];
    if (todo == 0u) return;

    // a step: 64 segments of one level, one per quarter wave
    constexpr uint32_t kEnd = 32;
    // Bins wider than the LDS sums (tables above 2^22 slots) are summed one range of kBinSlots slots after
    // the other: every range walks all the bin's records and takes those that fall into it.
    const uint32_t n_ranges = 1u << (pass_bins.bin_shift - kBinSlotsLog2);
    struct Cursor {
        uint32_t i, range, step;  // the workgroup's i-th level (kEnd: past the last), the range of the bin, segments 64 * step ...
    };
    const uint32_t n_steps = (n_groups + 63) / 64;
    const auto after = [&](Cursor at) {
        if (++at.step < n_steps) return at;
        at.step = 0u;
        if (++at.range < n_ranges) return at;
        const uint32_t rest = at.i + 1 < 32 ? todo >> (at.i + 1) : 0u;
        return Cursor{rest != 0u ? at.i + 1 + static_cast<uint32_t>(__builtin_ctz(rest)) : kEnd, 0u, 0u};
    };
    const uint32_t reader = wave * 4 + lane / kLevelsShortLanes, l = lane % kLevelsShortLanes;
    // (Every load below is issued whether or not its result is wanted, from an address that is valid
    // either way: with loads behind branches the compiler cannot tell how many are on their way and
    // makes every use wait for all of them, those of the next step included.)
    const auto load_count = [&](const Cursor& at) {
        const uint32_t g = at.step * 64 + reader;
        const uint32_t i = at.i != kEnd ? at.i : 0u;
        const uint32_t count = pass_bins.counts[first_segment(i) + (g < n_groups ? g : 0u)];
        return at.i != kEnd && g < n_groups ? count : 0u;
    };
    struct Loaded {
        RecordWords rec[kLevelsShortUnroll];
        uint32_t count, range;
    };
    const BinRecord* const records = static_cast<const BinRecord*>(pass_bins.records);
    const auto fetch = [&](const Cursor& at, uint32_t count, Loaded& got) {
        const uint32_t g = at.step * 64 + reader;
        const BinRecord* seg = records + (first_segment(at.i != kEnd ? at.i : 0u) + (g < n_groups ? g : 0u)) * seg_cap;
        got.count = count;
        got.range = at.range;
#pragma unroll
        for (uint32_t u = 0; u < kLevelsShortUnroll; ++u) {
            const uint32_t idx = u * kLevelsShortLanes + l;
            // (normal loads: neighbouring short segments share cache lines); the pass's first record stands in where there is none
            got.rec[u] = *reinterpret_cast<const RecordWords*>(idx < count ? seg + idx : records);
        }
    };
    const auto add = [&](const Loaded& got) {
#pragma unroll
        for (uint32_t u = 0; u < kLevelsShortUnroll; ++u) {
            const RecordWords w = got.rec[u];
            const uint32_t w0 = w.x, w1 = w.y, w2 = w.z;  // copies first: a bit cast applied directly to a vector element reads element 0
            if (u * kLevelsShortLanes + l < got.count && (w0 >> kBinSlotsLog2) == got.range) {
                const uint32_t cell = w0 & (kBinSlots - 1);
                __hip_atomic_fetch_add(&acc0[cell], static_cast<double>(__builtin_bit_cast(float, w1)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                __hip_atomic_fetch_add(&acc1[cell], static_cast<double>(__builtin_bit_cast(float, w2)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            }
        }
    };
    // Adds the sums of one range of the bin at the workgroup's i-th level into the gradient and clears them.  Nothing else touches
    // the bin's slots of that level while this kernel runs, so the add is a plain read-modify-write, or a
    // store where nothing was added since the gradient was cleared.
    const auto flush = [&](uint32_t i, uint32_t range) {
        lds_barrier();
        const uint32_t pair_level = static_cast<uint32_t>(first_level) + level_in_pass(i);
        const uint32_t level = pair_level / feat_pairs, pair = pair_level % feat_pairs;
        const GradSlice level_grad{table_grad + (static_cast<size_t>(level) * capacity * feat_pairs + pair) * 2, 2 * feat_pairs, nullptr, 0u};
        const uint32_t slot0 = (bin << pass_bins.bin_shift) + (range << kBinSlotsLog2);
        const bool untouched_so_far = ((direct_mask >> i) & 1u) == 0u;
        if (threadIdx.x == 0 && untouched_so_far) pass_bins.direct[static_cast<size_t>(level_in_pass(i)) * n_bins + bin] = 1u;  // this slot range now holds sums
        constexpr int kMine = kBinSlots / kReduceBlock;
        // (two loops, so that the usual one has no load to wait for: a wait would also be one for the
        // records of the next step, which are on their way)
        if (untouched_so_far) {
#pragma unroll
            for (int k = 0; k < kMine; ++k) {
                const uint32_t s = static_cast<uint32_t>(k) * kReduceBlock + threadIdx.x;
                const double v0 = acc0[s], v1 = acc1[s];
                if (v0 != 0.0 || v1 != 0.0) {
                    acc0[s] = 0.0;
                    acc1[s] = 0.0;
                    if (slot0 + s < capacity)
                        *reinterpret_cast<float2*>(level_grad.at(slot0 + s)) = make_float2(static_cast<float>(v0), static_cast<float>(v1));
                }
            }
        } else {
#pragma unroll
            for (int k = 0; k < kMine; ++k) {
                const uint32_t s = static_cast<uint32_t>(k) * kReduceBlock + threadIdx.x;
                const double v0 = acc0[s], v1 = acc1[s];
                if (v0 != 0.0 || v1 != 0.0) {
                    acc0[s] = 0.0;
                    acc1[s] = 0.0;
                    if (slot0 + s < capacity) {
                        float2* cell = reinterpret_cast<float2*>(level_grad.at(slot0 + s));
                        float2 g = *cell;
                        g.x += static_cast<float>(v0);
                        g.y += static_cast<float>(v1);
                        *cell = g;
                    }
                }
            }
        }
        lds_barrier();
    };
    // two sets of registers take turns for the records, two registers for the counts; past the last step the
    // counts are zero and the loads fetch the stand-in
    Cursor it0{static_cast<uint32_t>(__builtin_ctz(todo)), 0u, 0u};
    Cursor it1 = after(it0);
    uint32_t count_x = load_count(it0), count_y = load_count(it1);
    Loaded got_a, got_b;
    fetch(it0, count_x, got_a);
    while (true) {
        const Cursor it2 = it1.i != kEnd ? after(it1) : it1;
        count_x = load_count(it2);
        fetch(it1, count_y, got_b);
        add(got_a);
        if (it1.i != it0.i || it1.range != it0.range) flush(it0.i, it0.range);
        if (it1.i == kEnd) break;
        const Cursor it3 = it2.i != kEnd ? after(it2) : it2;
        count_y = load_count(it3);
        fetch(it2, count_x, got_a);
        add(got_b);
        if (it2.i != it1.i || it2.range != it1.range) flush(it1.i, it1.range);
        if (it2.i == kEnd) break;
        it0 = it2;
        it1 = it3;
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
