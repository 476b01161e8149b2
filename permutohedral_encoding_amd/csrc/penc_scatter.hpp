// Scatter-add of (slot, value pair) contributions into one level's slice of the table gradient.
//
// What the memory system of gfx950 gives (measured with purpose-built probes):
//   * a global fp32 atomic costs one request per 64-byte segment touched by a wave instruction,
//     whatever the number of lanes in the segment (1..16), the scope or the footprint; the chip
//     retires about 21 G such requests/s.  A level with many distinct slots is therefore bound
//     by requests, not bytes.
//   * ds_add_f32 retires about one lane every 3 clocks per CU, whatever the addresses: 30 times
//     slower than integer LDS atomics (ds_add_u32, ds_cmpst_b32/b64) and plain LDS accesses, and
//     5-20 times slower than ds_add_f64 (1.5 lanes/clock when 8 addresses take all the traffic,
//     3 for random addresses, 7.5 without bank conflicts).
//
// Hence three stages, each taking what the previous one could not combine:
//   1. Accumulate cache in LDS.  Every workgroup keeps a small open-addressed table
//      (tag = slot) for the level it works on.  Coarse levels, where thousands of points share
//      a handful of vertices, are absorbed here completely; the table is flushed once at the end.
//      When the first tile shows that the level has only a few dozen distinct slots, the cache's
//      LDS is re-laid as one column of per-lane cells for each slot (column mode): lanes then
//      add without meeting each other, and the wave-wide folding that a handful of hot lines
//      needs, which is what bounds those levels (vector ALU), is not needed at all.
//   2. Slot-range bins (optional, needs a workspace).  A contribution that finds no line in the
//      cache is appended, as a record of 12 or 10 bytes, to the bin of its slot range (each workgroup has a
//      private segment in every bin, so appending costs one LDS counter increment and one
//      store); a second kernel (bin_reduce_kernel) reads each bin back coalesced, sums it in
//      LDS (fp64), and adds the range into the gradient with coalesced read-modify-writes.  This
//      turns the random scatter of the fine levels into streaming traffic.  A workgroup whose
//      look-up of the first tile's slots shows that the cache would not hit at its level never
//      fills it: the cache's LDS becomes staging space in which the records of a tile are sorted by
//      bin, so that records of one bin leave in runs of consecutive addresses (whole cache lines)
//      instead of one small store each.
//   3. Direct global atomics, with the two features of a slot in one instruction (lane pairs),
//      for whatever is left: no workspace, capacity too large for binning, or a full bin.
// The result never depends on a stage hitting: every stage falls through to the next.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "penc_lattice.hpp"

namespace penc {

constexpr uint32_t kDefaultDies = 8;   // accelerator dies (XCDs) of an MI355X, for when the runtime does not tell
constexpr int kBlock = 256;            // threads per workgroup of the gather-type kernels (4 wavefronts)
#ifndef PENC_SCATTER_BLOCK
#define PENC_SCATTER_BLOCK 512
#define PENC_SCATTER_TILES 8
#define PENC_SCATTER_TILES_LARGE 16
#define PENC_CACHE_LINES_LOG2 11
#endif
constexpr int kScatterBlock = PENC_SCATTER_BLOCK;  // threads per scattering workgroup (its wavefronts share one accumulate cache)
constexpr int kScatterBlockManyBins = 2 * kScatterBlock;  // ... for tables of more than kFewerOpenLinesMinBins bins (see stream_tile_many)
constexpr uint32_t kFewerOpenLinesMinBins = 256;
constexpr int kScatterTiles = PENC_SCATTER_TILES;  // tiles of kScatterBlock points a scattering workgroup walks (a "group" of points) ...
constexpr int kScatterTilesLarge = PENC_SCATTER_TILES_LARGE;  // ... or this many, when the launch still has workgroups to spare
constexpr int kCacheLinesLog2 = PENC_CACHE_LINES_LOG2;
constexpr int kCacheLines = 1 << kCacheLinesLog2;  // accumulate-cache lines per workgroup
constexpr int kWaveGroups = 6;         // same-slot groups a wave folds with DPP before it touches the cache
constexpr int kMinWaveGroup = 8;       // ... as long as the groups have at least this many lanes
constexpr int kColumnMinIdsLog2 = 5;   // column mode: the cache's kCacheLines cells per feature are 32 columns of 64 cells (one per lane) ...
#ifndef PENC_COLUMN_MAX_IDS_LOG2
#define PENC_COLUMN_MAX_IDS_LOG2 7
#endif
constexpr int kColumnMaxIdsLog2 = PENC_COLUMN_MAX_IDS_LOG2;   // ... up to 128 columns of 16 cells, by the number of distinct slots the first tile has shown
constexpr int kColumnProbes = 16;      // entries a contribution looks at before it gives up on a column
enum ScatterMode : int { kModeCache = 0, kModeStream = 1, kModeColumns = 2 };
// vertices per thread a wave sorts by bin in one go (256 to 384 records): all D+1 of them up to D = 5
constexpr int stage_chunk(int pos_dim) { return pos_dim + 1 <= 4 ? 4 : (pos_dim == 5 ? 6 : 5); }
constexpr int kStageBins = 64;         // a wave counts one bin per lane: staging needs n_bins <= 64
constexpr int kWorkgroupSortMaxDim = 5;  // up to this input dimension a streaming workgroup sorts a tile's records across all its waves
constexpr int kBinSlotsLog2 = 13;      // slots per bin: 8192 (128 KiB of fp64 sums in LDS)
constexpr int kBinSlots = 1 << kBinSlotsLog2;
constexpr int kFinestBinSlotsLog2 = 10;  // small tables get narrower bins, down to this
constexpr int kMaxBins = 512;          // bins per level
constexpr int kMaxBinSlotsLog2 = 16;   // tables of more than kMaxBins * kBinSlots slots (2^22) get bins of up to 2^16 slots, which their
                                       // reducer sums one range of kBinSlots slots after the other; above 2^25 slots nothing is binned
constexpr int kReduceBlock = 1024;     // threads of a bin_reduce_kernel workgroup

// A contribution on its way through a bin: the slot within the bin's range and the two values.
// In memory the records of a level are either one array of these 12-byte structures, or 10 bytes in
// two arrays indexed alike, the values (8 bytes) and the slots (2 bytes: a bin spans 2^13 slots).
// The fine levels move nothing but records through the HBM, twice, so the split form saves a sixth
// of their traffic (measured on a 2^18-slot table: the reducer 0.163 -> 0.150 ms, the scattering
// kernel unchanged); it takes two stores per record, which pays only where a tile's records leave in long
// runs, i.e. where the workgroup-wide sort of stream_tile applies (measured on a 2^22-slot table, whose runs are
// about four records: the scattering kernel 0.313 -> 0.355 ms, the reducer 0.207 -> 0.218 ms; at
// D = 8, whose waves sort on their own and leave runs of eight: 0.343 -> 0.356 ms, 0.137 -> 0.129 ms).
struct BinRecord {
    uint32_t slot_in_bin;
    float a0, a1;
};
static_assert(kBinSlotsLog2 <= 16, "a split record keeps its slot within the bin in 16 bits");
typedef float RecordValues __attribute__((ext_vector_type(2)));
typedef uint32_t RecordWords __attribute__((ext_vector_type(3), aligned(4)));
constexpr size_t kSplitRecordBytes = sizeof(RecordValues) + sizeof(uint16_t);

// Where the misses of the levels of one launch go.  Every scattering workgroup (a "group" of
// points at one level) owns a private segment of `segment_capacity` records in every
// bin, so appending needs no global atomics and no synchronisation: the cursor is an LDS counter.
//   records [level_in_pass][bin][group][segment_capacity]   12-byte records, or the 8-byte values of split ones
//   slots   [level_in_pass][bin][group][segment_capacity]   the 2-byte slots of split records; nullptr otherwise
//   counts  [level_in_pass][bin][group]            records actually written (<= segment_capacity); with late adds of few bins (LateTarget) those there were to be
//   direct  [level_in_pass][bin]                   nonzero once anything has been added into the gradient in the
//                                                  bin's slot range: straight from the scattering kernel (see
//                                                  GradSlice), or by the bin's reducer.  Cleared with the gradient, or,
//                                                  for a caller who keeps gradient and flags across calls (the sparse
//                                                  entry points), the caller's map of touched slot ranges.
// `records` == nullptr disables binning (`direct`, `n_bins` and `bin_shift` may still be set: flags without bins).
// (Every kernel of a small batch begins with a fetch of its arguments, a cache line at a time: with the fields of ClearTarget in here too, a third
// line for the same code, bin_reduce_kernel took 14.4 us where it took 14.1, and the table gradient of 131007 points along rays 0.6 us longer in all.  The lists of late adds
// are given to the kernels that read them, bin_reduce_kernel among them, as an argument of their own.)
struct BinTarget {
    void* records;
    uint16_t* slots;
    uint32_t* counts;
    uint32_t* direct;
    uint32_t n_bins;
    uint32_t n_groups;
    uint32_t segment_capacity;
    uint32_t bin_shift;  // log2 of the slots per bin: kBinSlotsLog2, more only with more than kStageBins bins (whole records), less for small tables
};
// Where nothing may be added to a gradient that has not been cleared or written yet, what would go straight into it is kept:
//   kept    [level_in_pass][group][room]   {slot in the level, values}; there is room for all a group can leave
//   counts  [level_in_pass][group]
// kept == nullptr: nothing is.  Few bins of kBinSlots slots (written_whole) have no gradient cleared before: their reducers, one to a bin, write all of its slot range,
// and take what was kept from the lists of their level themselves.
struct LateTarget {
    BinRecord* kept;
    uint32_t* counts;
    uint32_t room;
};
// What the instances for narrow bins, which are never written whole, are given instead (for the look whether there are lists, and what follows from it, the scatter of 16
// levels of 2^14 slots, 2^18 points, took up to 3% longer: D = 2 53.6 -> 51.9 us, D = 3 62.1 -> 60.6, D = 5 118 -> 113).
struct NoLateTarget {
    NoLateTarget() = default;
    explicit NoLateTarget(const LateTarget&) {}
};
// Large tables (more than kStageBins bins, all levels in one launch): the scattering kernel clears the gradient and the flags
// itself, because those writes pass while it waits for other things.  The first `rows` rows of its grid, a workgroup to a die, do nothing else; rows == 0: every
// workgroup clears a share when it starts.  So many rows that they write at about half of the memory's rate: with more the loads of
// the others wait behind them, and where a share each is cleared by little more than one round of workgroups at once, fill and scatter might as
// well be apart (table gradient with a fill / a share each / rows, D = 3, 24 levels unless given, us):
//   2^21 slots  95077 points 227 / 201 / 167, 19 levels 158 / 161 / 133;  70000 points 196 / 192 / 155;  200001 points along rays, 1e-2, 208 / 185 / 145;  400000
//               459 / 428 / 400
//   2^20        70000 points 122 / 112 / 103, 16 levels 88 / 87 / 83;  200001 points 204 / 189 / 179;  D = 8, 50000 points 161 / 153 / 152
//   2^22        200001 points 524 / 431 / 383, near a surface with 16 levels live 324 / 246 / 246;  500003 points 784 / 719 / 666, near a surface, 1e-2,
//               498 / 414 / 423, 1e-3 631 / 566 / 523
// (4, 6, 8 and 12 rows of 512 threads for 95077 points 190 / 175 / 167 / 174; 3, 4, 6, 8 of 1024 for 500003 686 / 666 / 683 / 678.)  With many points the two are
// as good on average and apart by point order (kClearApartMaxWork).  Nothing may
// be added to a gradient that another workgroup is still to clear, so what would go straight into it is kept until the reducers have ended, and
// add_deferred_kernel adds it (5 to 7 us, up to 22 with more segments that have run over).
struct ClearTarget : LateTarget {
    uint32_t rows;    // of workgroups that clear and do nothing else
    uint64_t pairs;   // 8-byte units of the gradient,
    uint32_t flags;   // and its flags
};
// What a group of points can leave for later at a level: all its contributions, and the lines its cache claimed.
constexpr uint32_t deferred_room(int pos_dim, int tiles_per_group) {
    return static_cast<uint32_t>(tiles_per_group * kScatterBlock * (pos_dim + 1) + kCacheLines);
}

// `pass` describes the first level of a launch; level k of the launch follows k bin arrays later.
__device__ __forceinline__ BinTarget bins_of_level(const BinTarget& pass, uint32_t k) {
    BinTarget t = pass;
    if (pass.records != nullptr) {
        const size_t segments = static_cast<size_t>(k) * pass.n_bins * pass.n_groups;
        const size_t records = segments * pass.segment_capacity;
        t.records = static_cast<char*>(pass.records) + records * (pass.slots != nullptr ? sizeof(RecordValues) : sizeof(BinRecord));
        if (pass.slots != nullptr) t.slots += records;
        t.counts += segments;
    }
    if (pass.direct != nullptr) t.direct += static_cast<size_t>(k) * pass.n_bins;
    return t;
}

// Writes record `i` of a level (32-bit byte offsets: the host plans for that).
__device__ __forceinline__ void store_record(const BinTarget& bins, uint32_t i, uint32_t slot_in_bin, float a0, float a1) {
    char* const bytes = static_cast<char*>(bins.records);
    if (bins.slots != nullptr) {
        RecordValues v;
        v.x = a0;
        v.y = a1;
        *reinterpret_cast<RecordValues*>(bytes + i * static_cast<uint32_t>(sizeof(RecordValues))) = v;
        *reinterpret_cast<uint16_t*>(reinterpret_cast<char*>(bins.slots) + i * 2u) = static_cast<uint16_t>(slot_in_bin);
    } else {
        BinRecord rec;
        rec.slot_in_bin = slot_in_bin;
        rec.a0 = a0;
        rec.a1 = a1;
        *reinterpret_cast<BinRecord*>(bytes + i * static_cast<uint32_t>(sizeof(BinRecord))) = rec;
    }
}

// Writes a staged record {slot in its bin, values, index of the record in the level's array}, where records are whole.
__device__ __forceinline__ void store_whole_record(const BinTarget& bins, uint4 e) {
    BinRecord rec;
    rec.slot_in_bin = e.x;
    rec.a0 = __builtin_bit_cast(float, e.y);
    rec.a1 = __builtin_bit_cast(float, e.z);
    *reinterpret_cast<BinRecord*>(static_cast<char*>(bins.records) + e.w * static_cast<uint32_t>(sizeof(BinRecord))) = rec;
}

// Record `i` of a bin whose first record is `first` (of the level's arrays), with ordinary loads.
template <bool kSplit>
__device__ __forceinline__ BinRecord load_record(const BinTarget& bins, size_t first, uint32_t i) {
    BinRecord rec;
    if constexpr (kSplit) {
        const RecordValues v = static_cast<const RecordValues*>(bins.records)[first + i];
        rec.slot_in_bin = bins.slots[first + i];
        rec.a0 = v.x;
        rec.a1 = v.y;
    } else {
        rec = static_cast<const BinRecord*>(bins.records)[first + i];
    }
    return rec;
}

// The same with the non-temporal hint: the reducer reads every record once, and a normal
// load would make room for it in the caches by evicting records the scatter has just written and
// that are still waiting there to be read (measured: the reducer of 2^18-slot tables 0.213 ->
// 0.168 ms; non-temporal *stores* of the records cost the scatter more than they save here).
template <bool kSplit>
__device__ __forceinline__ BinRecord load_record_once(const BinTarget& bins, size_t first, uint32_t i) {
    BinRecord rec;
    if constexpr (kSplit) {
        const RecordValues v = __builtin_nontemporal_load(static_cast<const RecordValues*>(bins.records) + first + i);
        rec.slot_in_bin = __builtin_nontemporal_load(bins.slots + first + i);
        rec.a0 = v.x;
        rec.a1 = v.y;
    } else {
        const RecordWords w = __builtin_nontemporal_load(reinterpret_cast<const RecordWords*>(static_cast<const BinRecord*>(bins.records) + first + i));
        const uint32_t w0 = w.x, w1 = w.y, w2 = w.z;  // copies first: a bit cast applied directly to a vector element reads element 0
        rec.slot_in_bin = w0;
        rec.a0 = __builtin_bit_cast(float, w1);
        rec.a1 = __builtin_bit_cast(float, w2);
    }
    return rec;
}

// One level's slice of the table gradient as the scatter sees it: a pair of features per slot,
// `slot_floats` floats from one slot to the next (2 when a level has two features; with four, the
// slice of features (0,1) or (2,3) of an array whose slots are four floats apart).
// `direct` (the level's BinTarget::direct, or nullptr without bins) is told about every add that goes
// straight into the gradient: a bin whose slot range received none still holds the zeros it was
// cleared to when its reducer workgroup arrives, which can then store its sums without reading
// the gradient first (on a 2^22-slot table, whose gradient no cache holds, that read is a third
// of the reducer's traffic).
struct GradSlice {
    float* base;
    uint32_t slot_floats;
    uint32_t* direct;
    uint32_t bin_shift;  // of the bins `direct` belongs to
    BinRecord* deferred;       // nullptr: adds go into the gradient; else the workgroup's list of them (see LateTarget),
    uint32_t* deferred_count;  // in LDS: how many are in it
    __device__ __forceinline__ float* at(uint32_t slot) const { return base + static_cast<size_t>(slot) * slot_floats; }
    // A plain store on purpose: many workgroups may set the same flag at once, all to 1, and nobody reads it before the
    // kernel has ended.  (As a relaxed atomic store of device scope, a store that writes through the L2, the levels that
    // sum in columns took up to 2.5 times as long and the kernel 8% longer.)
    __device__ __forceinline__ void mark_direct(uint32_t slot) const {
        if (direct != nullptr) direct[slot >> bin_shift] = 1u;
    }
    __device__ __forceinline__ void defer(uint32_t slot, float a0, float a1) const { deferred[atomicAdd(deferred_count, 1u)] = BinRecord{slot, a0, a1}; }
};

__device__ __forceinline__ void global_add(float* addr, float v) {
    __hip_atomic_fetch_add(addr, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Sum over the 64 lanes of a wavefront; the total is valid in lane 63.
__device__ __forceinline__ float wave_sum_to_last_lane(float v) {
    // row_shr:1,2,4,8 build the total of each row of 16 in its last lane (lanes shifted in from
    // outside the row read 0); row_bcast:15 adds it into rows 1 and 3, row_bcast:31 into rows 2 and 3
    constexpr int kShr1 = 0x111, kShr2 = 0x112, kShr4 = 0x114, kShr8 = 0x118, kBcast15 = 0x142, kBcast31 = 0x143;
#define PENC_DPP_ADD(CTRL, ROW_MASK) \
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, ROW_MASK, 0xf, true))
    PENC_DPP_ADD(kShr1, 0xf);
    PENC_DPP_ADD(kShr2, 0xf);
    PENC_DPP_ADD(kShr4, 0xf);
    PENC_DPP_ADD(kShr8, 0xf);
    PENC_DPP_ADD(kBcast15, 0xa);
    PENC_DPP_ADD(kBcast31, 0xc);
#undef PENC_DPP_ADD
    return v;
}

// The value `v` has in lane `lane` (wave-uniform index), broadcast to all lanes.
__device__ __forceinline__ float lane_value(float v, int lane) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}

// Exclusive prefix sum over the 64 lanes of a wavefront; `total` is the sum of all lanes.
__device__ __forceinline__ uint32_t wave_exclusive_scan(uint32_t v, uint32_t& total) {
    // row_shr:1,2,4,8 scan each row of 16 (lanes shifted in from outside the row read 0);
    // row_bcast:15 adds the total of rows 0 and 2 to rows 1 and 3, row_bcast:31 that of rows 0-1 to rows 2-3
    int s = static_cast<int>(v);
    s += __builtin_amdgcn_update_dpp(0, s, 0x111, 0xf, 0xf, true);
    s += __builtin_amdgcn_update_dpp(0, s, 0x112, 0xf, 0xf, true);
    s += __builtin_amdgcn_update_dpp(0, s, 0x114, 0xf, 0xf, true);
    s += __builtin_amdgcn_update_dpp(0, s, 0x118, 0xf, 0xf, true);
    s += __builtin_amdgcn_update_dpp(0, s, 0x142, 0xa, 0xf, true);
    s += __builtin_amdgcn_update_dpp(0, s, 0x143, 0xc, 0xf, true);
    total = static_cast<uint32_t>(__builtin_amdgcn_readlane(s, 63));
    return static_cast<uint32_t>(s) - v;
}

// Orders the LDS accesses of one wavefront: what its lanes wrote before is visible to all of them
// after (LDS executes a wave's instructions in order; this keeps the compiler from reordering them).
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// A barrier that orders the workgroup's LDS accesses only.  __syncthreads() also makes the global stores
// issued so far visible, i.e. waits for the counter that loads share with them: after a store, it
// would wait for every load that is still on its way.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Stage 3.  Lanes are paired (2p, 2p+1): first both lanes of a pair add the two features of the
// even lane's slot, then those of the odd lane's slot, so that each 8-byte slot is one request.
// Must be called with all 64 lanes of the wave active.
__device__ __forceinline__ void global_add_pairs(const GradSlice& level_grad, bool need, uint32_t slot,
                                                 float a0, float a1) {
    constexpr int kFromEven = 0xA0;  // quad_perm:[0,0,2,2]
    constexpr int kFromOdd = 0xF5;   // quad_perm:[1,1,3,3]
    if (level_grad.deferred != nullptr) {
        if (need) level_grad.defer(slot, a0, a1);
        return;
    }
    if (need) level_grad.mark_direct(slot);
    const int odd = threadIdx.x & 1;
    const int slot_i = static_cast<int>(slot), need_i = need ? 1 : 0;
    const int a0_i = __builtin_bit_cast(int, a0), a1_i = __builtin_bit_cast(int, a1);
    {   // the even lane's contribution: even lane adds feature 0, odd lane feature 1
        const int s = __builtin_amdgcn_update_dpp(0, slot_i, kFromEven, 0xf, 0xf, true);
        const int n = __builtin_amdgcn_update_dpp(0, need_i, kFromEven, 0xf, 0xf, true);
        const int hi = __builtin_amdgcn_update_dpp(0, a1_i, kFromEven, 0xf, 0xf, true);
        const float v = __builtin_bit_cast(float, odd ? hi : a0_i);
        if (n) global_add(level_grad.at(static_cast<uint32_t>(s)) + odd, v);
    }
    {   // the odd lane's contribution
        const int s = __builtin_amdgcn_update_dpp(0, slot_i, kFromOdd, 0xf, 0xf, true);
        const int n = __builtin_amdgcn_update_dpp(0, need_i, kFromOdd, 0xf, 0xf, true);
        const int lo = __builtin_amdgcn_update_dpp(0, a0_i, kFromOdd, 0xf, 0xf, true);
        const float v = __builtin_bit_cast(float, odd ? a1_i : lo);
        if (n) global_add(level_grad.at(static_cast<uint32_t>(s)) + odd, v);
    }
}

// Folds runs of neighbouring lanes that add to the same slot, within each row of 16 lanes: a segmented
// inclusive scan over the row (DPP row shifts, four steps), after which the last lane of every run
// holds the run's sums and is the only one of it still `live`.  Batches whose consecutive points are
// neighbours in space (samples along a ray) make such runs at every level whose cells are wider than the
// sampling distance: left alone they are what LDS atomics are slowest at (a few lanes on each of many
// addresses, too few per address for the wave-wide fold below).  Returns the number of lanes folded away.
// Must be called with all 64 lanes of the wave active.  Worth its 45 instructions only where many lanes have such a
// neighbour: neighbours_share_slots() asks that of one vertex per tile, for all the tile's vertices.
__device__ __forceinline__ bool neighbours_share_slots(uint32_t slot, bool live) {
    const int key = live ? static_cast<int>(slot) : -1 - static_cast<int>(threadIdx.x & 63);
    const int prev = __builtin_amdgcn_update_dpp(0, key, 0x111 /* row_shr:1 */, 0xf, 0xf, true);
    return __popcll(__ballot((threadIdx.x & 15) != 0 && prev == key)) >= 16;
}
__device__ __forceinline__ uint32_t fold_adjacent_runs(uint32_t slot, bool& live, float& x0, float& x1) {
    constexpr int kShr1 = 0x111, kShl1 = 0x101;  // row_shr:1, row_shl:1; row_shr:n is 0x110 + n
    const uint32_t lane = threadIdx.x & 63, in_row = lane & 15;
    // a lane that adds nothing gets a key of its own, so it joins no run
    const int key = live ? static_cast<int>(slot) : -1 - static_cast<int>(lane);
    const int prev = __builtin_amdgcn_update_dpp(0, key, kShr1, 0xf, 0xf, true);
    // `open`: the partial sum of this lane does not reach back to the first lane of its run yet
    int open = (in_row != 0 && prev == key) ? 1 : 0;
#define PENC_SCAN_STEP(SHIFT)                                                                                              \
    {                                                                                                                      \
        const float s0 = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x0), 0x110 + SHIFT, 0xf, 0xf, true)); \
        const float s1 = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x1), 0x110 + SHIFT, 0xf, 0xf, true)); \
        const int so = __builtin_amdgcn_update_dpp(0, open, 0x110 + SHIFT, 0xf, 0xf, true);  /* 0 from beyond the row: a run ends there */      \
        x0 += open ? s0 : 0.0f;                                                                                            \
        x1 += open ? s1 : 0.0f;                                                                                            \
        open = open ? so : 0;                                                                                              \
    }
    PENC_SCAN_STEP(1)
    PENC_SCAN_STEP(2)
    PENC_SCAN_STEP(4)
    PENC_SCAN_STEP(8)
#undef PENC_SCAN_STEP
    const int next = __builtin_amdgcn_update_dpp(0, key, kShl1, 0xf, 0xf, true);
    const bool last_of_run = in_row == 15 || next != key;
    const bool was_live = live;
    live = live && last_of_run;
    return __popcll(__ballot(was_live && !live));
}

// Folds the contributions of lanes that share a slot, wherever they are in the wave.  At the coarsest levels the 64 lanes of a
// wave hit two to six distinct slots, and LDS atomics on one address serialise (about 5 clocks per lane): so up to
// kWaveGroups times, take the slot of the first pending lane, sum the contributions of
// all lanes that share it with DPP, and leave the sum with that lane alone.  A group
// of fewer than kMinWaveGroup lanes means the wave's slots are spread out: stop.  Returns the number of lanes folded away.
__device__ __forceinline__ uint32_t fold_shared_slots(uint32_t slot, bool& live, float& x0, float& x1) {
    uint32_t folded = 0;
    unsigned long long pending = __ballot(live);
#pragma unroll 1
    for (int round = 0; round < kWaveGroups && pending != 0ull; ++round) {
        const int leader = __builtin_ctzll(pending);
        const uint32_t leader_slot = __builtin_amdgcn_readlane(slot, leader);
        const bool in_group = live && slot == leader_slot;
        const unsigned long long members = __ballot(in_group);
        if (__popcll(members) < kMinWaveGroup) break;
        const float s0 = lane_value(wave_sum_to_last_lane(in_group ? x0 : 0.0f), 63);
        const float s1 = lane_value(wave_sum_to_last_lane(in_group ? x1 : 0.0f), 63);
        const bool is_leader = static_cast<int>(threadIdx.x & 63) == leader;
        x0 = is_leader ? s0 : x0;
        x1 = is_leader ? s1 : x1;
        live = live && (!in_group || is_leader);
        folded += __popcll(members) - 1;
        pending &= ~members;
    }
    return folded;
}

// LDS state of a scattering workgroup.  The accumulate cache sums in fp64 with ds_add_f64: its
// lines are hit by many lanes at once (that is what the cache is for), where a compare-and-swap
// loop degrades quadratically (measured: 10-40x slower on the coarsest levels) and ds_add_f32 is
// slow on this chip.  The fp64 partial sums are rounded to fp32 once, when the cache is flushed.
template <int kStageChunk, int kBlockThreads>
struct ScatterStateT {
    static constexpr int kChunk = kStageChunk, kThreads = kBlockThreads;
    static constexpr int kTail = (kThreads / 64) * kStageChunk * 64 - kCacheLines;
    static_assert(kTail >= 0, "the staging slices cover the cache's values");
    int tag[kCacheLines];
    double val[2][kCacheLines];  // one array per feature: random lines then spread over all LDS bank pairs
    // when the workgroup streams, val and this tail together are its waves' staging slices
    uint4 stage_tail[kTail > 0 ? kTail : 1];
    uint32_t bin_count[kMaxBins];  // records this workgroup has appended to each bin so far
    uint32_t hits;                 // contributions the cache has absorbed into existing lines since the first tile
    // what the look at the first tile's slots showed (see scatter_mode_decide)
    uint32_t distinct;             // of them, as far as the bits they were marked in tell them apart
    uint32_t wanted;               // contributions of the first tile,
    uint32_t first_hits;           // and how many of them find a line that an earlier one has claimed
    uint32_t columns;              // columns given away (kModeColumns)
    uint32_t deferred;             // entries of the workgroup's list of deferred adds
    uint32_t strangers;            // slots of the second tile that the first tile did not touch (counted for levels with few slots)
};

// The bits in which the first tile's slots are marked: 128 to a thread of the workgroup (2^16 or 2^17 of them), where the values will be.
template <typename State>
__device__ __forceinline__ uint32_t* seen_bits(State& c) { return reinterpret_cast<uint32_t*>(c.val); }
template <typename State>
__device__ __forceinline__ uint32_t seen_bit(uint32_t slot) {
    return (slot * 0x9E3779B1u) >> (32 - __builtin_ctz(static_cast<unsigned>(State::kThreads) * 128u));
}

// Where the weights of a thread's first point (kSets arrays of D+1) wait while the slots of its second one are found for scatter_mode_decide: in the staging
// space past the marked bits, and in the tags, neither of which holds anything yet.  A cell is its thread's own.  With both points' values in registers at
// once the kernels of both orders were held to 128 with up to 24 of them spilled, the next tile's point among them, which every tile then waited for
// (scatter of both orders from [level][feature][n], 16 levels, 2^18 points, before -> with ranks, as it was -> so, us: D = 8, 2^14 slots 202 -> 188 -> 182,
// 2^18 195 -> 178 -> 180, 2^20 235 -> 216 -> 212, 2^22 373 -> 302 -> 294;  D = 7, 2^20 231 -> 217 -> 197;  D = 3, 2^20 105 -> 101 -> 102;  first order, D = 4, 2^18 82 -> 83 -> 79).
template <int D, int kSets, typename State>
struct ParkedWeights {
    static constexpr int kInStage = 4 * State::kChunk - 4;  // words a thread has there
    static_assert((kSets * (D + 1) - kInStage) * State::kThreads <= kCacheLines, "they fit");
    State& c;
    template <int i>
    __device__ __forceinline__ float& cell() const {
        if constexpr (i < kInStage) return reinterpret_cast<float*>(c.val)[(4 + i) * State::kThreads + threadIdx.x];
        else return reinterpret_cast<float*>(c.tag)[(i - kInStage) * State::kThreads + threadIdx.x];
    }
    template <int kSet>
    __device__ __forceinline__ void put(fvec<D + 1> w) const {
        static_for<D + 1>(PENC_BODY(r) {
            PENC_INDEX(r); cell<kSet * (D + 1) + r>() = w[r]; });
    }
    template <int kSet>
    __device__ __forceinline__ void take(fvec<D + 1>& w) const {
        static_for<D + 1>(PENC_BODY(r) {
            PENC_INDEX(r); w[r] = cell<kSet * (D + 1) + r>(); });
    }
};

// Clears what the look at the first tile needs, and the bins' cursors.
template <typename State>
__device__ __forceinline__ void scatter_begin(State& c) {
    static_assert(State::kThreads * sizeof(uint4) <= sizeof(c.val), "the bits fit");
    reinterpret_cast<uint4*>(seen_bits(c))[threadIdx.x] = make_uint4(0u, 0u, 0u, 0u);
    for (int b = threadIdx.x; b < kMaxBins; b += State::kThreads) c.bin_count[b] = 0u;
    if (threadIdx.x == 0) {
        c.hits = 0u;
        c.distinct = 0u;
        c.strangers = 0u;
        c.columns = 0u;
    }
    __syncthreads();
}

// Stage 2 for one contribution: append a record to this workgroup's segment of the slot's bin.
// Returns false when the segment is full.
template <typename State>
__device__ __forceinline__ bool append_record(State& c, const BinTarget& bins, uint32_t group, uint32_t slot,
                                              float a0, float a1) {
    const uint32_t b = slot >> bins.bin_shift;
    const uint32_t pos = atomicAdd(&c.bin_count[b], 1u);
    if (pos >= bins.segment_capacity) return false;
    store_record(bins, (b * bins.n_groups + group) * bins.segment_capacity + pos, slot & ((1u << bins.bin_shift) - 1u), a0, a1);
    return true;
}

// From D = 4 on a third candidate line: every contribution of a slot that finds no line becomes
// a record, and tens of thousands of records on a handful of slots serialise in the LDS of
// the one reducer workgroup that owns their bin.  At D = 3 the low 11 bits of a coarse level's
// slots are all distinct and two candidates leave no slot out while the level fits; at D = 4
// they collide (levels 6 and 7 of 24: 350 and 1000 slots, 4 and 110 of them left out; those
// levels' reducer workgroups took 0.05-0.11 ms each, and with a third candidate the
// double backward's table half went from 0.73 to 0.65 ms; at D = 3 it would add 2% to the
// scattering kernel for nothing).
constexpr int cache_probes(int pos_dim) { return pos_dim >= 4 ? 3 : 2; }

// Looks `slot` up in the accumulate cache, claiming a free line if there is one.  Two candidate
// lines per slot (two-choice hashing): with one, a level with a few hundred distinct slots already
// loses several of them to collisions, and those are exactly the slots every wave keeps hitting.
// Returns the line, or -1 when both candidates belong to other slots; `found` tells whether the
// line already held the slot (a hit, as opposed to a claim).
// (Spreading the lanes that share a slot over replicated sub-tables, instead of folding them in
// registers first, was measured 30% slower on the coarse levels, and no faster on top of folding.)
template <int kProbes, typename State>
__device__ __forceinline__ int cache_find(State& c, uint32_t slot, bool& found) {
    const int want = static_cast<int>(slot);
    int e = static_cast<int>(slot & (kCacheLines - 1));
    found = false;
    constexpr uint32_t kMix[3] = {0x9E3779B1u, 0x85EBCA6Bu, 0xC2B2AE35u};
    static_assert(kProbes >= 1 && kProbes <= 4, "one mixing constant per probe after the first");
#pragma unroll
    for (int probe = 0; probe < kProbes; ++probe) {
        int owner = c.tag[e];
        if (owner == want) {
            found = true;
            return e;
        }
        if (owner == -1) {
            owner = atomicCAS(&c.tag[e], -1, want);
            if (owner == -1 || owner == want) return e;
        }
        if (probe + 1 < kProbes) e = static_cast<int>((slot * kMix[probe]) >> (32 - kCacheLinesLog2));
    }
    return -1;
}

// Stage 2 for a whole tile once the workgroup streams (see scatter_mode_decide): the cache's LDS is
// staging space for a counting sort of the tile's records by bin, all vertices at a time
// (1536 to 3072 records of 512 threads).  The workgroup counts its records per bin; then every wave, lane b looking after bin b, turns the
// counts into where each bin's run starts in the staging space and in the workgroup's segment, and lays its records out in that order;
// and then all threads store the records in staging order: a wave instruction writes 64 consecutive records
// of (mostly) one bin, i.e. whole cache lines, where the records of a single wave would leave in
// runs of eight.  How far the workgroup's segment of a bin is filled (`cursor`, lane b's is bin b's) every wave
// knows from the same sums.  (With the offsets made by the first wave for all, and a cursor in LDS, the others waited for it at a
// barrier of its own.  Scatter and reduction of the finest 12 of 24 levels of 2^18 slots, D = 3, 2^20 points: 348 -> 322 us, of the finest four
// 149 -> 119; D = 4, second order, 12 levels 437 -> 412; with the coarse levels beside them, which keep the vector units busy, the same.)
// A staged record carries its destination (its index in the level's record
// array), so the store needs no search.  When a run does not fit its segment any more (rare: the
// segments hold the mean plus three standard deviations) the tile checks every record against
// the room left and sends the excess to stage 3, in code of its own: without a branch in them, a thread's trips to the LDS
// for its D+1 records are made together, not one after the other.
// What it waits for are those trips and the barriers, not the vector units (53% of their slots), the LDS or the stores.  With counters of every wave's own, summed by all
// of them, and a branch for every record (scatter of 2^20 points, 24 levels of 2^18 slots, before -> after, us): D = 3 from rows 371 -> 356, D = 4 472 -> 430,
// second order 450 -> 428, D = 2 307 -> 296; 16 levels, 2^19 points, D = 5 236 -> 229; 131007 points along rays 53 -> 51.  With four dimensions all five records
// of a point together would spill: three.
// Two arrays of counters take turns (`tile` says which): the other one is cleared between this tile's barriers.  Both are
// zero before the first tile.
// Needs bins.n_bins <= kStageBins, split records and a level's record array below 2^32 bytes (the host plans
// for all three); all threads of the workgroup must call it together.
template <int D, typename State>
__device__ __forceinline__ void stream_tile(State& c, const GradSlice& level_grad, const BinTarget& bins,
                                            uint32_t group, uint32_t tile, bool active, uvec<D + 1> slot, fvec<D + 1> a0,
                                            fvec<D + 1> a1, uint32_t& cursor) {
    constexpr int kWaves = State::kThreads / 64;
    constexpr int kStageChunk = State::kChunk;
    static_assert(D + 1 <= kStageChunk, "all vertices of a tile are staged at a time");
    static_assert(kCacheLines >= 2 * kStageBins + 2 * kWaves * kStageBins, "the sort's index arrays live in the tag array");
    static_assert(offsetof(State, stage_tail) == offsetof(State, val) + sizeof(c.val) &&
                      (sizeof(c.val) + (State::kTail > 0 ? sizeof(c.stage_tail) : 0)) == kStageChunk * State::kThreads * sizeof(uint4),
                  "val and stage_tail are one contiguous staging array");
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    uint32_t* const words = reinterpret_cast<uint32_t*>(c.tag);
    uint32_t* const count = words + (tile & 1u) * kStageBins;  // [bin] records of this tile
    uint32_t* const next_count = words + (~tile & 1u) * kStageBins;
    // [bin], every wave's own: where the bin's run starts in the staging array, and the index of the run's first record in the level's record array
    uint2* const run = reinterpret_cast<uint2*>(words + 2 * kStageBins) + wave * kStageBins;
    uint4* const stage = reinterpret_cast<uint4*>(c.val);
    constexpr int kTogether = D == 4 ? 3 : D + 1;
    uvec<D + 1> place = 0u;  // rank of each record within its bin's run
    if (active) {
        static_for<D + 1>(PENC_BODY(j) {
            PENC_INDEX(j); place[j] = atomicAdd(&count[slot[j] >> bins.bin_shift], 1u); });
    }
    __syncthreads();  // all waves have counted, and have left the staging array of the tile before
    const uint32_t mine = count[lane];
    if (wave == 0u) next_count[lane] = 0u;  // (last read before the last tile's second barrier, counted in after the next one here)
    uint32_t total;
    const uint32_t first = wave_exclusive_scan(mine, total);
    run[lane] = make_uint2(first, (lane * bins.n_groups + group) * bins.segment_capacity + cursor);
    cursor += mine;
    const bool all_fit = __all(cursor <= bins.segment_capacity);
    wave_lds_fence();
    RecordValues* const values_out = static_cast<RecordValues*>(bins.records);
    const auto record_of = [&](uint32_t slot_in_bin, float v0, float v1, uint32_t to) {
        uint4 e;
        e.x = slot_in_bin;
        e.y = __builtin_bit_cast(uint32_t, v0);
        e.z = __builtin_bit_cast(uint32_t, v1);
        e.w = to;
        return e;
    };
    const auto store = [&](const uint4& e) {
        RecordValues v;
        v.x = __builtin_bit_cast(float, e.y);
        v.y = __builtin_bit_cast(float, e.z);
        *reinterpret_cast<RecordValues*>(reinterpret_cast<char*>(values_out) + e.w * static_cast<uint32_t>(sizeof(RecordValues))) = v;
        *reinterpret_cast<uint16_t*>(reinterpret_cast<char*>(bins.slots) + e.w * 2u) = static_cast<uint16_t>(e.x);
    };
    if (all_fit) {
        if (active) {
            static_for<(D + kTogether) / kTogether>(PENC_BODY(part) {
                PENC_INDEX(part);
                constexpr int kFirst = part * kTogether, kCount = D + 1 - kFirst < kTogether ? D + 1 - kFirst : kTogether;
                uint2 at[kCount];
                static_for<kCount>(PENC_BODY(k) {
                    PENC_INDEX(k); at[k] = run[slot[kFirst + k] >> bins.bin_shift]; });
                static_for<kCount>(PENC_BODY(k) {
                    PENC_INDEX(k);
                    constexpr int j = kFirst + k;
                    const float v0 = a0[j], v1 = a1[j];  // copies first: a bit cast applied directly to a vector element reads element 0
                    stage[at[k].x + place[j]] = record_of(slot[j] & ((1u << bins.bin_shift) - 1u), v0, v1, at[k].y + place[j]);
                });
            });
        }
        __syncthreads();
        static_for<(D + kTogether) / kTogether>(PENC_BODY(part) {
            PENC_INDEX(part);
            constexpr int kFirst = part * kTogether, kCount = D + 1 - kFirst < kTogether ? D + 1 - kFirst : kTogether;
            uint4 e[kCount];  // (past the tile's last record: what an earlier one left there)
            static_for<kCount>(PENC_BODY(k) {
                PENC_INDEX(k); e[k] = stage[(kFirst + k) * State::kThreads + threadIdx.x]; });
            static_for<kCount>(PENC_BODY(k) {
                PENC_INDEX(k);
                if ((kFirst + k) * State::kThreads + threadIdx.x < total) store(e[k]);
            });
        });
    } else {
        constexpr uint32_t kNoRoom = 0xFFFFFFFFu;
        if (active) {
            static_for<D + 1>(PENC_BODY(j) {
                PENC_INDEX(j);
                const uint32_t b = slot[j] >> bins.bin_shift;
                const float v0 = a0[j], v1 = a1[j];
                const uint2 at = run[b];
                const uint32_t to = at.y + place[j];
                stage[at.x + place[j]] = record_of(slot[j], v0, v1, to < (b * bins.n_groups + group + 1u) * bins.segment_capacity ? to : kNoRoom);
            });
        }
        __syncthreads();
#pragma unroll 1
        for (int j = 0; j <= D; ++j) {
            const uint32_t i = j * State::kThreads + threadIdx.x;
            bool spill = false;
            uint4 e = {0u, 0u, 0u, 0u};
            if (i < total) {
                e = stage[i];
                spill = e.w == kNoRoom;  // the segment is full: stage 3
                if (!spill) store(make_uint4(e.x & ((1u << bins.bin_shift) - 1u), e.y, e.z, e.w));
            }
            if (__any(spill)) global_add_pairs(level_grad, spill, e.x, __builtin_bit_cast(float, e.y), __builtin_bit_cast(float, e.z));
        }
    }
    // the next tile counts in the other array, and writes the staging array after its own first barrier: nothing here is
    // overwritten while another wave reads it
    wave_lds_fence();
}

// The same sort for tables with more bins than a wave has lanes (up to one bin per thread of the
// workgroup: capacities up to 2^22).  One LDS counter per bin for the whole workgroup gives every
// record its place in the bin's run; thread b then looks after bin b: one block-wide prefix sum
// over the counts, one reservation per bin.  With hundreds of bins a tile leaves only a handful of
// records in each, but even runs of four records are worth it: appended one at a time, every
// 12-byte record is a store of its own to one of hundreds of open cache lines (measured on a
// 2^22-slot table: 42 us per level against 13 us for the sorted stores of a 2^18-slot one).
// What it waits for with the most bins is the lines the records go to: a workgroup leaves a line open in every bin, and of 512 bins and the 96
// workgroups of a die those are 6 MB, which its L2 writes out part by part.  So workgroups of twice the threads serve them, of which
// a compute unit holds one: a third of the open lines, and twice the records in a run.  (Scatter, reduction and fill, us: 2^22 slots, D = 3, 2^20
// points, 24 levels 1203 -> 1046, the finest eight 664 -> 604; 200001 points 537 -> 512; D = 4, 16 levels, 2^19 points 579 -> 533; D = 8, 2^17 points
// 427 -> 423.  With 256 bins, whose open lines nearly fit, 24 levels 855 -> 780 but 16 coarser ones from rows 502 -> 566; with 128 599 -> 661.)
// The counters must be zero on entry (scatter_mode_decide clears them; every call leaves them so).
template <int D, typename State>
__device__ __forceinline__ void stream_tile_many(State& c, const GradSlice& level_grad, const BinTarget& bins,
                                                 uint32_t group, bool active, uvec<D + 1> slot, fvec<D + 1> a0,
                                                 fvec<D + 1> a1) {
    constexpr int kWaves = State::kThreads / 64;
    constexpr int kStageChunk = State::kChunk;
    static_assert(kMaxBins <= State::kThreads, "one thread per bin");
    static_assert(kCacheLines >= 3 * kMaxBins + kWaves, "the sort's index arrays live in the tag array");
    const uint32_t wave = threadIdx.x >> 6;
    uint32_t* const words = reinterpret_cast<uint32_t*>(c.tag);
    uint32_t* const count = words;                       // [bin] records of this chunk
    uint32_t* const offset = words + kMaxBins;           // [bin] where the bin's run starts in the staging array
    uint32_t* const dest = words + 2 * kMaxBins;         // [bin] index of the run's first record in the level's record array
    uint32_t* const wave_total = words + 3 * kMaxBins;   // [wave] records of the wave's 64 bins
    uint4* const stage = reinterpret_cast<uint4*>(c.val);
    constexpr uint32_t kNoRoom = 0xFFFFFFFFu;
    constexpr int kChunks = (D + 1 + kStageChunk - 1) / kStageChunk;
    const uint32_t my_bin = threadIdx.x;  // the bin this thread looks after
    const uint32_t my_segment = (my_bin * bins.n_groups + group) * bins.segment_capacity;
    static_for<kChunks>(PENC_BODY(chunk) {
        PENC_INDEX(chunk);
        constexpr int kFirst = chunk * kStageChunk;
        constexpr int kCount = D + 1 - kFirst < kStageChunk ? D + 1 - kFirst : kStageChunk;
        uvec<kStageChunk> place = 0u;  // rank of each record within the workgroup's run for its bin
        static_for<kCount>(PENC_BODY(j) {
            PENC_INDEX(j);
            if (active) place[j] = atomicAdd(&count[slot[kFirst + j] >> bins.bin_shift], 1u);
        });
        __syncthreads();
        uint32_t mine = 0u;
        if (my_bin < bins.n_bins) {
            mine = count[my_bin];
            count[my_bin] = 0u;  // for the next chunk; nobody counts again before the barriers below
        }
        uint32_t in_wave;
        const uint32_t before_in_wave = wave_exclusive_scan(mine, in_wave);
        if ((threadIdx.x & 63) == 0) wave_total[wave] = in_wave;
        __syncthreads();
        uint32_t before = before_in_wave, total = 0u;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            const uint32_t t = wave_total[w];
            before += w < static_cast<int>(wave) ? t : 0u;
            total += t;
        }
        bool fits = true;
        if (my_bin < bins.n_bins) {
            const uint32_t taken = c.bin_count[my_bin];  // only this thread touches its bin's cursor while the workgroup streams
            if (mine != 0u) c.bin_count[my_bin] = taken + mine;
            offset[my_bin] = before;
            dest[my_bin] = my_segment + taken;
            fits = taken + mine <= bins.segment_capacity;
        }
        const bool all_fit = __syncthreads_and(fits);
        static_for<kCount>(PENC_BODY(j) {
            PENC_INDEX(j);
            if (active) {
                const uint32_t b = slot[kFirst + j] >> bins.bin_shift;
                // copies first: a bit cast applied directly to a vector element reads element 0
                const float v0 = a0[kFirst + j], v1 = a1[kFirst + j];
                const uint32_t to = dest[b] + place[j];
                const uint32_t segment_end = (b * bins.n_groups + group + 1u) * bins.segment_capacity;
                uint4 e;
                e.x = slot[kFirst + j];
                e.y = __builtin_bit_cast(uint32_t, v0);
                e.z = __builtin_bit_cast(uint32_t, v1);
                e.w = all_fit || to < segment_end ? to : kNoRoom;
                stage[offset[b] + place[j]] = e;
            }
        });
        __syncthreads();
        static_for<kCount>(PENC_BODY(j) {
            PENC_INDEX(j);
            const uint32_t i = j * State::kThreads + threadIdx.x;
            bool spill = false;
            uint4 e = {0u, 0u, 0u, 0u};
            if (i < total) {
                e = stage[i];
                if (e.w != kNoRoom) {
                    store_record(bins, e.w, e.x & ((1u << bins.bin_shift) - 1u), __builtin_bit_cast(float, e.y), __builtin_bit_cast(float, e.z));
                } else {
                    spill = true;  // the segment is full: stage 3
                }
            }
            if (!all_fit && __any(spill))
                global_add_pairs(level_grad, spill, e.x, __builtin_bit_cast(float, e.y), __builtin_bit_cast(float, e.z));
        });
        // The next chunk (or tile) counts into counters this chunk has cleared, overwrites offset/dest after its
        // first two barriers and what other threads read of the staging array after its third.
    });
}

// The same sort with every wave on its own (no barriers), for the higher dimensions: their D+1
// vertices take two chunks, the waves of a workgroup drift apart over their longer tiles, and
// waiting for each other in every chunk then costs more than the longer runs save
// (measured: 5-7% slower at D = 6, 7, 8).
// The staging space is a 4 or 5 KiB slice per wave.  For stage_chunk(D) vertices per thread at a time, the wave
// counts its records per bin (one LDS counter per bin, owned by one lane), reserves room for each
// bin's run in the workgroup's segment with one add per bin, lays the records out bin by bin in
// its slice, and then stores them in that order: neighbouring lanes write neighbouring addresses.
// A staged record carries its destination (its index in the level's record array), so the
// store needs no search.  When a run does not fit its segment any more (rare: the segments hold
// the mean plus three standard deviations) the whole chunk takes the careful path, which checks
// every record against the room left and sends the excess to stage 3.
// Needs bins.n_bins <= kStageBins, whole records and a level's record array below 2^32 bytes (the host plans
// for all three); all 64 lanes of the wave must call it together.
template <int D, typename State>
__device__ __forceinline__ void stream_tile_wave(State& c, const GradSlice& level_grad, const BinTarget& bins,
                                            uint32_t group, bool active, uvec<D + 1> slot, fvec<D + 1> a0,
                                            fvec<D + 1> a1) {
    constexpr int kWaves = State::kThreads / 64;
    constexpr int kStageChunk = State::kChunk;
    static_assert(kCacheLines / kWaves >= 4 * 64, "four 64-entry arrays per wave live in the tag array");
    static_assert(offsetof(State, stage_tail) == offsetof(State, val) + sizeof(c.val) &&
                      (sizeof(c.val) + (State::kTail > 0 ? sizeof(c.stage_tail) : 0)) / kWaves == kStageChunk * 64 * sizeof(uint4),
                  "val and stage_tail are one contiguous array of staging slices");
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    uint32_t* count = reinterpret_cast<uint32_t*>(c.tag) + wave * (kCacheLines / kWaves);  // records per bin
    uint2* run = reinterpret_cast<uint2*>(count + 64);  // where a bin's run starts in the wave's slice, and the index of its first record in the level's record array
    uint32_t* room = count + 192;   // records the workgroup's segment of the bin can still take
    uint4* stage = reinterpret_cast<uint4*>(c.val) + wave * (kStageChunk * 64);
    constexpr uint32_t kNoRoom = 0xFFFFFFFFu;
    constexpr int kChunks = (D + 1 + kStageChunk - 1) / kStageChunk;
    static_for<kChunks>(PENC_BODY(chunk) {
        PENC_INDEX(chunk);
        constexpr int kFirst = chunk * kStageChunk;
        constexpr int kCount = D + 1 - kFirst < kStageChunk ? D + 1 - kFirst : kStageChunk;
        count[lane] = 0u;
        wave_lds_fence();
        uvec<kStageChunk> place = 0u;  // rank of each record within its bin's run
        if (active) {
            static_for<kCount>(PENC_BODY(j) {
                PENC_INDEX(j); place[j] = atomicAdd(&count[slot[kFirst + j] >> bins.bin_shift], 1u); });
        }
        wave_lds_fence();
        // lane b looks after bin b: one reservation and one index computation per bin, not per record
        const uint32_t mine = count[lane];
        const uint32_t taken = mine != 0u ? atomicAdd(&c.bin_count[lane], mine) : 0u;
        uint32_t total;
        const uint32_t before = wave_exclusive_scan(mine, total);
        run[lane] = make_uint2(before, (lane * bins.n_groups + group) * bins.segment_capacity + taken);
        const bool fits = taken + mine <= bins.segment_capacity;
        if (__all(fits)) {  // (no branch for single records: a thread's trips to the LDS are made together)
            wave_lds_fence();
            if (active) {
                uint2 at[kCount];
                static_for<kCount>(PENC_BODY(j) {
                    PENC_INDEX(j); at[j] = run[slot[kFirst + j] >> bins.bin_shift]; });
                static_for<kCount>(PENC_BODY(j) {
                    PENC_INDEX(j);
                    // copies first: a bit cast applied directly to a vector element reads element 0
                    const float v0 = a0[kFirst + j], v1 = a1[kFirst + j];
                    uint4 e;
                    e.x = slot[kFirst + j] & ((1u << bins.bin_shift) - 1u);
                    e.y = __builtin_bit_cast(uint32_t, v0);
                    e.z = __builtin_bit_cast(uint32_t, v1);
                    e.w = at[j].y + place[j];
                    stage[at[j].x + place[j]] = e;
                });
            }
            wave_lds_fence();
            uint4 e[kCount];  // (past the chunk's last record: what an earlier one left there)
            static_for<kCount>(PENC_BODY(j) {
                PENC_INDEX(j); e[j] = stage[j * 64 + lane]; });
            static_for<kCount>(PENC_BODY(j) {
                PENC_INDEX(j);
                if (j * 64 + lane < total) store_whole_record(bins, e[j]);
            });
        } else {
            room[lane] = taken < bins.segment_capacity ? bins.segment_capacity - taken : 0u;
            wave_lds_fence();
            static_for<kCount>(PENC_BODY(j) {
                PENC_INDEX(j);
                if (active) {
                    const uint32_t b = slot[kFirst + j] >> bins.bin_shift;
                    const float v0 = a0[kFirst + j], v1 = a1[kFirst + j];
                    uint4 e;
                    e.x = slot[kFirst + j];
                    e.y = __builtin_bit_cast(uint32_t, v0);
                    e.z = __builtin_bit_cast(uint32_t, v1);
                    e.w = place[j] < room[b] ? run[b].y + place[j] : kNoRoom;
                    stage[run[b].x + place[j]] = e;
                }
            });
            wave_lds_fence();
            static_for<kCount>(PENC_BODY(j) {
                PENC_INDEX(j);
                const uint32_t i = j * 64 + lane;
                bool spill = false;
                uint4 e = {0u, 0u, 0u, 0u};
                if (i < total) {
                    e = stage[i];
                    spill = e.w == kNoRoom;  // the segment is full: stage 3
                    if (!spill) store_whole_record(bins, make_uint4(e.x & ((1u << bins.bin_shift) - 1u), e.y, e.z, e.w));
                }
                if (__any(spill))
                    global_add_pairs(level_grad, spill, e.x, __builtin_bit_cast(float, e.y), __builtin_bit_cast(float, e.z));
            });
        }
        wave_lds_fence();
    });
}

// Column mode of stage 1, for a level whose points share a few dozen slots.  The cache's values
// are re-laid as 2^id_bits columns of kCacheLines >> id_bits cells; a slot owns a column and a lane adds into the
// cell (lane mod cells) of its slot's column.  With 64 cells a lane meets no other lane of its
// wave, whatever the slots; with 32 or 16 cells two or four lanes share a cell.  The columns are
// summed when the level ends (column_flush).
// A slot finds its column through kColumnEntries entries, eight and more times as many as there are columns, so that nearly every
// look-up ends at its first entry; among as many entries as columns the last lane of a wave took several probes (D = 3, 2^20 points, the six
// coarsest of 24 levels 106 -> 96 us).  Tags, the entries' columns and the columns' slots share the tag array.
constexpr uint32_t kColumnEntriesLog2 = 10, kColumnEntries = 1u << kColumnEntriesLog2;
constexpr uint32_t kColumnPending = 0xFFu, kNoColumn = 0xFEu;  // in place of an entry's column: not known yet, none was left
static_assert(kCacheLines >= static_cast<int>(kColumnEntries + kColumnEntries / 4 + (1u << kColumnMaxIdsLog2)), "they fit the tag array");
static_assert((1u << kColumnMaxIdsLog2) <= kNoColumn, "a column's number is kept in a byte");
template <typename State>
__device__ __forceinline__ uint8_t* column_of_entry(State& c) { return reinterpret_cast<uint8_t*>(c.tag + kColumnEntries); }
template <typename State>
__device__ __forceinline__ int* slot_of_column(State& c) { return c.tag + kColumnEntries + kColumnEntries / 4; }
__device__ __forceinline__ uint32_t column_entry(uint32_t slot) { return (slot * 0x9E3779B1u) >> (32 - kColumnEntriesLog2); }

// Looks on from entry `e` for the slot, and gives it an entry and a column where it has none.  Returns the column, or kNoColumn
// when no entry or column is left (the contribution then takes stage 2 or 3 like any miss).  A lane that finds the slot's entry
// just taken looks again until it says which column, a few times at most: a miss would leave a record, and a level without records
// costs its reducers nothing.
template <typename State>
__device__ __forceinline__ uint32_t column_search(State& c, uint32_t slot, uint32_t e, uint32_t id_bits) {
    const int want = static_cast<int>(slot);
    uint32_t column = kNoColumn;
#pragma unroll 1
    for (int probe = 0; probe < kColumnProbes; ++probe) {
        int owner = c.tag[e];
        if (owner == -1) {
            owner = atomicCAS(&c.tag[e], -1, want);
            if (owner == -1) {
                const uint32_t next = atomicAdd(&c.columns, 1u);
                const bool left = next < (1u << id_bits);
                if (left) slot_of_column(c)[next] = want;
                column_of_entry(c)[e] = static_cast<uint8_t>(left ? next : kNoColumn);
                owner = want;
            }
        }
        // (the lanes of a wave meet here: what one of them has written above, the others read)
        __builtin_amdgcn_wave_barrier();
        if (owner == want) {
#pragma unroll 1
            for (int look = 0; look < 64; ++look) {
                column = __hip_atomic_load(column_of_entry(c) + e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                if (column != kColumnPending) break;
            }
            break;
        }
        e = (e + 1u) & (kColumnEntries - 1u);
    }
    return column != kColumnPending ? column : kNoColumn;
}

template <int D, typename State>
__device__ __forceinline__ void column_tile(State& c, const GradSlice& level_grad, const BinTarget& bins,
                                            uint32_t group, bool active, uint32_t id_bits, uvec<D + 1> slot,
                                            fvec<D + 1> a0, fvec<D + 1> a1) {
    const uint32_t cell_bits = kCacheLinesLog2 - id_bits;
    const uint32_t my_cell = threadIdx.x & ((1u << cell_bits) - 1u);
    static_for<D + 1>(PENC_BODY(r) {
        PENC_INDEX(r);
        bool miss = active;
        if (active) {
            const uint32_t e = column_entry(slot[r]);
            const int owner = c.tag[e];
            uint32_t column = column_of_entry(c)[e];
            if (owner != static_cast<int>(slot[r]) || column == kColumnPending) column = column_search(c, slot[r], e, id_bits);
            if (column != kNoColumn) {
                const uint32_t cell = (column << cell_bits) | my_cell;
                __hip_atomic_fetch_add(&c.val[0][cell], static_cast<double>(a0[r]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                __hip_atomic_fetch_add(&c.val[1][cell], static_cast<double>(a1[r]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                miss = false;
            }
        }
        if (miss && bins.records != nullptr) miss = !append_record(c, bins, group, slot[r], a0[r], a1[r]);
        if (__any(miss)) global_add_pairs(level_grad, miss, slot[r], a0[r], a1[r]);
    });
}

// Sums every column in use and adds the sums to the gradient (stage 3).  By all threads, between barriers.
template <bool kManyBins, typename State>
__device__ __forceinline__ void column_flush(State& c, const GradSlice& level_grad, const BinTarget& bins, uint32_t group, uint32_t id_bits) {
    const uint32_t cell_bits = kCacheLinesLog2 - id_bits, cells = 1u << cell_bits;
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (uint32_t id = wave; id < (1u << id_bits); id += State::kThreads / 64) {
        const int owner = slot_of_column(c)[id];  // the same for all lanes of the wave
        if (owner == -1) continue;
        double s0 = lane < cells ? c.val[0][(id << cell_bits) + lane] : 0.0;
        double s1 = lane < cells ? c.val[1][(id << cell_bits) + lane] : 0.0;
#pragma unroll
        for (int step = 32; step > 0; step >>= 1) {
            s0 += __shfl_xor(s0, step);
            s1 += __shfl_xor(s1, step);
        }
        if (lane == 0) {
            // straight into the gradient: a level in column mode leaves a few dozen sums per workgroup, and
            // as records they would only make every bin's reducer workgroup run for a handful of them.  (Where the reducers write everything they run
            // in any case.)
            if (level_grad.deferred != nullptr) {
                const float v0 = static_cast<float>(s0), v1 = static_cast<float>(s1);
                if (kManyBins || !append_record(c, bins, group, static_cast<uint32_t>(owner), v0, v1)) level_grad.defer(static_cast<uint32_t>(owner), v0, v1);
                continue;
            }
            float* g = level_grad.at(static_cast<uint32_t>(owner));
            level_grad.mark_direct(static_cast<uint32_t>(owner));
            global_add(g, static_cast<float>(s0));
            global_add(g + 1, static_cast<float>(s1));
        }
    }
}

// One tile's D+1 contributions per thread through stages 1-3.  All 64 lanes of every wave must
// call it together; `active` is false for lanes that carry no point (tail of the last tile), which
// only take part in the wave-wide steps.  `use_cache` (wave-uniform) is false once the workgroup
// has seen that the cache does not hit at this level; `mode` and `id_bits` are what
// scatter_mode_decide decided.  The return value is the number of hits of this wave in this tile.
template <int D, bool kManyBins, typename State>
__device__ __forceinline__ uint32_t scatter_tile(State& c, const GradSlice& level_grad, const BinTarget& bins,
                                                 uint32_t group, uint32_t tile, bool active, bool use_cache, int mode, uint32_t id_bits,
                                                 uvec<D + 1> slot, fvec<D + 1> a0, fvec<D + 1> a1, uint32_t& cursor) {
    if (mode == kModeStream) {
        if constexpr (kManyBins) {
            stream_tile_many<D>(c, level_grad, bins, group, active, slot, a0, a1);
        } else if constexpr (D <= kWorkgroupSortMaxDim) {  // measured: the workgroup-wide sort wins up to D = 5, the per-wave one from D = 6 on
            stream_tile<D>(c, level_grad, bins, group, tile, active, slot, a0, a1, cursor);
        } else {
            stream_tile_wave<D>(c, level_grad, bins, group, active, slot, a0, a1);
        }
        return 0u;
    }
    if (mode == kModeColumns) {
        column_tile<D>(c, level_grad, bins, group, active, id_bits, slot, a0, a1);
        return 0u;
    }
    uint32_t hits = 0;
    // (wave-uniform) the points of this tile follow each other in space: neighbouring lanes often add to the same slot
    const bool ordered = use_cache && neighbours_share_slots(slot[0], active);
    static_for<D + 1>(PENC_BODY(r) {
        PENC_INDEX(r);
        float x0 = a0[r], x1 = a1[r];
        bool miss = active;
        if (use_cache) {
            // neighbouring lanes on one slot first (points that follow each other in space), then the slots most of the wave shares
            if (ordered) hits += fold_adjacent_runs(slot[r], miss, x0, x1);
            hits += fold_shared_slots(slot[r], miss, x0, x1);
            bool found = false;
            if (miss) {
                const int e = cache_find<cache_probes(D)>(c, slot[r], found);
                if (e >= 0) {
                    __hip_atomic_fetch_add(&c.val[0][e], static_cast<double>(x0), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    __hip_atomic_fetch_add(&c.val[1][e], static_cast<double>(x1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    miss = false;
                }
            }
            hits += __popcll(__ballot(found));
        }
        // stage 2, then stage 3 for what stage 2 could not take
        if (miss && bins.records != nullptr) miss = !append_record(c, bins, group, slot[r], x0, x1);
        if (__any(miss)) global_add_pairs(level_grad, miss, slot[r], x0, x1);
    });
    return hits;
}

// The workgroup-wide decision whether stage 1 is worth its LDS traffic at this level: keep using the
// cache only while at least one contribution in eight hits.  The evidence before tile `tile` is
// the look at the first tile's slots and the hits of the tiles processed since.  Against appending every miss to its
// bin on its own, one hit in eight pays; against sorting the tile's records by bin (stream_tile),
// which is cheaper than the cache's look-ups, it takes one in four.
template <int D, typename State>
__device__ __forceinline__ bool cache_pays(const State& c, int tile) {
    const uint32_t seen = c.wanted + static_cast<uint32_t>(tile > 1 ? tile - 1 : 0) * State::kThreads * (D + 1);
    return (c.first_hits + c.hits) * 8u >= seen;
}

// Sends every line of the accumulate cache on to stage 2 (or 3).  By all threads, between barriers.
template <typename State>
__device__ __forceinline__ void cache_flush(State& c, const GradSlice& level_grad, const BinTarget& bins,
                                            uint32_t group) {
    for (int e = threadIdx.x; e < kCacheLines; e += State::kThreads) {
        const int owner = c.tag[e];
        if (owner != -1) {
            const float v0 = static_cast<float>(c.val[0][e]), v1 = static_cast<float>(c.val[1][e]);
            const bool binned = bins.records != nullptr && append_record(c, bins, group, static_cast<uint32_t>(owner), v0, v1);
            if (!binned && level_grad.deferred != nullptr) {
                level_grad.defer(static_cast<uint32_t>(owner), v0, v1);
            } else if (!binned) {
                float* g = level_grad.at(static_cast<uint32_t>(owner));
                level_grad.mark_direct(static_cast<uint32_t>(owner));
                global_add(g, v0);
                global_add(g + 1, v1);
            }
        }
    }
}

// Before the first tile is scattered (all threads call it, with the tile's slots): decides for the
// whole workgroup how the level goes, and clears the LDS for it.  Every slot is marked in a bit of its own, nearly, and a bit that was not set
// yet is a slot more: the tile's distinct slots tell what the accumulate cache would be good for.  One
// that would not hit is not used: its LDS becomes staging space (kModeStream, see
// stream_tile; needs bins).  One that would hit on at most 64 lines, and whose group of points is not expected to
// touch more than 96 slots in all, becomes columns (kModeColumns, `id_bits` says how many).  Otherwise the
// cache serves.
// (One LDS operation for a contribution, all of a thread's made together.  Claiming the slots' lines in the cache itself to find out took a workgroup 5700 clocks,
// up to 14000 among others, and all of its LDS had to be cleared before; a tile takes 4000 to 12000.  Scatter, us: D = 3, 2^20 points, 24 levels of 2^18 slots from
// rows 348 -> 337; D = 8, 2^19 points, 16 levels of 2^19 306 -> 267; 2^22 slots, 200001 points, both orders 91.5 -> 86.)
template <int D, typename State, typename NextSlots>
__device__ __forceinline__ int scatter_mode_decide(State& c, const BinTarget& bins, bool active, uint32_t points, uvec<D + 1> slot,
                                                   uint32_t& id_bits, bool next_active, NextSlots&& slots_of_next_tile,
                                                   int tiles_per_group) {
    uint32_t* const seen = seen_bits(c);
    uvec<D + 1> before = 0xFFFFFFFFu;
    if (active) {
        static_for<D + 1>(PENC_BODY(r) {
            PENC_INDEX(r);
            // (LDS atomics of a wave on one word take turns, 5 clocks a lane, and points along a ray bring a coarse level's slot 64 times: where the lane
            // before, which is active too, marks it, a lane leaves a word of its own as it is.  Without a branch: with one, two registers more are spilled
            // at D = 8.  Scatter of 131072 points along rays, 16 levels of 2^14 slots down to 1e-4, us: D = 2 43.6 -> 40.2, D = 4 67.4 -> 63.0.)
            const int key = static_cast<int>(~slot[r]);  // not 0, which the first lane of a row finds before it
            const bool again = __builtin_amdgcn_update_dpp(0, key, 0x111 /* row_shr:1 */, 0xf, 0xf, true) == key;
            const uint32_t bit = seen_bit<State>(slot[r]), mark = again ? 0u : 1u << (bit & 31u);
            const uint32_t old = atomicOr(&seen[again ? threadIdx.x : bit >> 5], mark);
            before[r] = again ? 1u : old & mark;
        });
    }
    uint32_t fresh = 0;  // over the wave
    static_for<D + 1>(PENC_BODY(r) {
        PENC_INDEX(r); fresh += __popcll(__ballot(before[r] == 0u)); });
    if ((threadIdx.x & 63) == 0) atomicAdd(&c.distinct, fresh);
    __syncthreads();
    const uint32_t wanted = points * (D + 1), distinct = c.distinct;
    // Of u slots that each look for one of N lines at two places, N tanh(u/N) find one, and as large a part of the repeats does.
    const float load = static_cast<float>(distinct) * (1.0f / kCacheLines), load2 = load * load;
    const float held = (27.0f + load2) / (27.0f + 9.0f * load2);  // tanh(load) / load, within 2% up to twice as many slots as lines
    const uint32_t first_hits = wanted > distinct ? static_cast<uint32_t>(static_cast<float>(wanted - distinct) * held) : 0u;
    // Columns are for a level whose few slots the whole group shares.  The first tile shows that when the points come in no
    // particular order; where they follow each other in space (every tile another ray, or the next stretch of a space-filling
    // curve) each tile brings slots of its own, the table of columns fills up, and every contribution that then finds no
    // column probes in vain and leaves one record.  The second tile's slots tell the two apart: how many of its contributions
    // go to slots the first tile did not touch?  (Asked only of a level that is a candidate for columns: the look at the
    // second tile costs a simplex search.)
    const bool few_slots = first_hits * 8u >= wanted && distinct <= (1u << (kColumnMaxIdsLog2 - 1));  // the table of columns starts at most half full
    if (few_slots && tiles_per_group > 1) {
        const uvec<D + 1> next_slot = slots_of_next_tile();
        uint32_t strangers = 0;
        static_for<D + 1>(PENC_BODY(r) {
            PENC_INDEX(r);
            const uint32_t bit = seen_bit<State>(next_slot[r]);
            strangers += __popcll(__ballot(next_active && ((seen[bit >> 5] >> (bit & 31u)) & 1u) == 0u));
        });
        if ((threadIdx.x & 63) == 0 && strangers != 0u) atomicAdd(&c.strangers, strangers);
        __syncthreads();
    }
    int mode = kModeCache;
    const bool can_stream = bins.records != nullptr && bins.n_bins <= static_cast<uint32_t>(kMaxBins);
    // The slots the group will have touched in the end: the first tile's, and from every later tile as many new ones as the
    // second tile brought, counted twice (a slot at the rim of what a tile covers gets fewer contributions than one inside).
    const uint32_t expected_slots = distinct + (2u * distinct * c.strangers * static_cast<uint32_t>(tiles_per_group - 1)) / (wanted != 0u ? wanted : 1u);
    if (can_stream && first_hits * 4u < wanted) {
        mode = kModeStream;
        for (int e = threadIdx.x; e < kMaxBins; e += State::kThreads) c.tag[e] = 0;  // stream_tile and stream_tile_many count there
    } else {
        if (few_slots && expected_slots <= (3u << (kColumnMaxIdsLog2 - 2))) {  // the largest table may end up three quarters full
            mode = kModeColumns;
            id_bits = kColumnMinIdsLog2;
            while ((1u << (id_bits - 1)) < expected_slots && id_bits < static_cast<uint32_t>(kColumnMaxIdsLog2)) ++id_bits;
        }
        // lines without a slot, or entries without columns; no sums yet
        const uint32_t kNone = 0xFFFFFFFFu;
        static_assert(kCacheLines % (2 * State::kThreads) == 0, "whole entries to a thread");
#pragma unroll
        for (int e = 0; e < kCacheLines / 2; e += State::kThreads) reinterpret_cast<uint2*>(c.tag)[e + threadIdx.x] = make_uint2(kNone, kNone);
#pragma unroll
        for (int e = 0; e < kCacheLines; e += State::kThreads) reinterpret_cast<uint4*>(c.val)[e + threadIdx.x] = make_uint4(0u, 0u, 0u, 0u);
        if (threadIdx.x == 0) {
            c.wanted = wanted;
            c.first_hits = first_hits;
        }
    }
    __syncthreads();
    if (mode == kModeCache) {
        // The tile's slots claim their lines before any later tile's do: the slots that come often are among them, and every contribution of a slot
        // that finds no line is a record.  (Waves that claimed as they came: reducers of two such levels, D = 8, 22 -> 29 and 34 -> 46 us.)
        static_for<D + 1>(PENC_BODY(r) {
            PENC_INDEX(r);
            bool found = false;
            if (active) cache_find<cache_probes(D)>(c, slot[r], found);
        });
        __syncthreads();
    }
    return mode;
}

// After the last tile: flushes the accumulate cache or the columns (through the bins when there are
// any; a streaming workgroup has neither left) and publishes how many records this workgroup left in each
// bin.  Call once, by all threads.
template <int D, bool kManyBins, typename State>
__device__ __forceinline__ void scatter_end(State& c, const GradSlice& level_grad, const BinTarget& bins,
                                            uint32_t group, int mode, uint32_t id_bits, uint32_t cursor) {
    // (stream_tile keeps count in registers)
    if (D <= kWorkgroupSortMaxDim && !kManyBins && mode == kModeStream && threadIdx.x < 64) c.bin_count[threadIdx.x] = cursor;
    __syncthreads();
    if (mode == kModeCache) cache_flush(c, level_grad, bins, group);
    if (mode == kModeColumns) column_flush<kManyBins>(c, level_grad, bins, group, id_bits);
    if (bins.records == nullptr) return;
    __syncthreads();
    for (uint32_t b = threadIdx.x; b < bins.n_bins; b += State::kThreads) {
        const uint32_t n = c.bin_count[b];
        // (a reducer that takes late adds too looks for them where a segment was to have more records than it has room for)
        const bool as_wanted = !kManyBins && level_grad.deferred != nullptr;
        bins.counts[static_cast<size_t>(b) * bins.n_groups + group] = as_wanted || n < bins.segment_capacity ? n : bins.segment_capacity;
    }
}

}  // namespace penc
