// Tables in cells: copies of a table whose cache lines hold the slots of neighbouring lattice points.
//
// A gather at a level finer than the batch's points is one 128-byte line per vertex, because the hash spreads the D+1 vertices of a
// simplex over the table; the lines the L2s serve (one request per channel and clock) or fetch are what the gathering kernels wait
// for.  For capacities that are powers of two the hash is linear: vertex r+1 is vertex r plus one of D+1 constants (hash_step), and so
// slots modulo a line's B slots tell to which coset of an index-B sublattice a lattice point belongs.  Choose for every residue i one lattice
// vector whose hash T[i] is i modulo B, as short as there is: the B vectors are a compact cell, whose translations by the
// sublattice cover the lattice once, and
//     line(h) = (h - T[h mod B]) / B,   place in the line = h mod B
// gives all points of a cell one line.  It is a permutation of the slots whatever the points, so a gather from the
// permuted copy reads the values it would read from the table.  Lines per simplex, with 16 slots (32) to a line, mean over all
// simplices: D = 2 1.5 of 3 (1.36), D = 3 2.23 of 4 (2.03), D = 4 3.1 of 5 (2.8), D = 5 4.35 of 6 (3.9), D = 6 5.2 of 7 (4.85), D = 7 6.3 of 8
// (5.75), D = 8 7.4 of 9 (7.0); and at levels whose points share vertices, a line holds many that are used.  Forward of 500003 points near a surface, 24 levels of 2^22
// slots in bfloat16, of which the L2s miss every other line: 313 -> 160 us; of 2^20 unordered points, 2^18 slots 276 -> 194, 2^14 194 -> 149.
#pragma once

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>
#include <utility>

#include "penc_lattice.hpp"
#include "penc_scatter.hpp"

namespace penc {

struct bfloat16_bits {
    uint16_t bits;  // the upper half of the fp32 with the same value
};

constexpr int kLineBytes = 128;
constexpr int kMostLineSlots = 32;  // two features in 16 bits
template <int F, typename T>
constexpr int line_slots() { return kLineBytes / (F * static_cast<int>(sizeof(T))); }

// T of the head comment for lines of 32, 16, 8 and 4 slots, one after the other (a line of B from 64 - 2 B): the lattice vectors
// sum_k n_k c_k, c_k the steps from vertex to vertex (c_0 + ... + c_D = 0), hash to sum_k n_k hash_step(k); for every residue the one nearest to a
// centre off the lattice (so that two are hardly ever as near).
struct CellOffsets {
    uint32_t t[64];
};
constexpr int cells_at(int slots) { return 64 - 2 * slots; }
template <int D, int... C>
constexpr uint32_t hash_step_of(int c, std::integer_sequence<int, C...>) {
    return ((C == c ? hash_step<D, C>() : 0u) + ...);
}
template <int D>
constexpr CellOffsets find_cells() {
    constexpr int kReach = D == 2 ? 3 : (D <= 5 ? 2 : 1);  // all residues are found within it
    CellOffsets cells{};
    uint32_t step[D + 1] = {};
    // hash, sum of m_k = 9 n_k - (k < D ? k + 1 : 0) and of its squares, kept up to date while the n_k count through their range; the squared
    // length of sum_k m_k c_k is (D+1) ((D+1) sum m_k^2 - (sum m_k)^2)
    int n[D + 1] = {}, sum = 0, squares = 0, best[64] = {};
    uint32_t hash = 0u;
    for (int k = 0; k <= D; ++k) {
        step[k] = hash_step_of<D>(k, std::make_integer_sequence<int, D + 1>{});
        n[k] = -kReach;
        const int m = 9 * n[k] - (k < D ? k + 1 : 0);
        hash += static_cast<uint32_t>(n[k]) * step[k];
        sum += m;
        squares += m * m;
    }
    for (int i = 0; i < 64; ++i) best[i] = -1;
    for (int k = 0; k <= D;) {
        const int length = (D + 1) * squares - sum * sum;
        for (int slots = 4; slots <= kMostLineSlots; slots *= 2) {
            const int i = cells_at(slots) + static_cast<int>(hash & static_cast<uint32_t>(slots - 1));
            if (best[i] < 0 || length < best[i]) {
                best[i] = length;
                cells.t[i] = hash;
            }
        }
        for (k = 0; k <= D; ++k) {
            const int by = n[k] < kReach ? 1 : -2 * kReach, m = 9 * n[k] - (k < D ? k + 1 : 0);
            n[k] += by;
            hash += static_cast<uint32_t>(by) * step[k];
            sum += 9 * by;
            squares += 18 * m * by + 81 * by * by;
            if (by == 1) break;
        }
    }
    return cells;
}
template <int D>
constexpr CellOffsets kCells = find_cells<D>();
template <int D>
constexpr bool finds_all_cells() {
    for (int slots = 4; slots <= kMostLineSlots; slots *= 2)
        for (int i = 0; i < slots; ++i)
            if (static_cast<int>(kCells<D>.t[cells_at(slots) + i] & static_cast<uint32_t>(slots - 1)) != i) return false;
    return true;
}
static_assert(finds_all_cells<2>() && finds_all_cells<3>() && finds_all_cells<4>() && finds_all_cells<5>() && finds_all_cells<6>() &&
                  finds_all_cells<7>() && finds_all_cells<8>(),
              "every residue has its vector");
template <int D>
static __device__ const CellOffsets cell_offsets = kCells<D>;

// Raw hashes whose low bits are slots of the table in cells.  (A wave's look-ups fall into one line, which the first-level cache holds.)
template <int D, int kSlots>
__device__ __forceinline__ uvec<D + 1> hashes_in_cells(uvec<D + 1> h) {
    uvec<D + 1> moved;
    static_for<D + 1>(PENC_BODY(r) {
        PENC_INDEX(r);
        const uint32_t i = h[r] & (kSlots - 1);
        moved[r] = (h[r] - cell_offsets<D>.t[cells_at(kSlots) + i]) | i;  // (the difference is a multiple of kSlots)
    });
    return moved;
}
// The same for a 16-bit copy that may be in cells.
template <int D, int F, typename T>
__device__ __forceinline__ uvec<D + 1> hashes_in_copy(uint32_t in_cells, uvec<D + 1> h) {
    if constexpr (sizeof(T) == 2) {
        if (in_cells != 0u) h = hashes_in_cells<D, line_slots<F, T>()>(h);
    }
    return h;
}

// ------------------------------------------------------------------------------------------
// making the copy
//
// Place i of line q of the copy is place i of line q + T[i]/B of the table: every column of the table, taken as a matrix of lines, is
// rotated by an amount of its own.  Reading the columns where they are would move a line for every slot, so the table goes
// through a column-major copy (one pass writes the columns, the other reads each from where its rotation starts), a few levels at a time
// so that this copy stays in the memory-side cache.
constexpr int kCellBlock = 256;
constexpr int kCellLines = 128;  // lines a workgroup of either pass takes: runs of 512 bytes and more in a column

__device__ __forceinline__ uint16_t to_bfloat16(float x) {  // to nearest, ties to even
    const uint32_t bits = __builtin_bit_cast(uint32_t, x);
    if ((bits & 0x7FFFFFFFu) > 0x7F800000u) return 0x7FC0u;
    return static_cast<uint16_t>((bits + 0x7FFFu + ((bits >> 16) & 1u)) >> 16);
}

// The offsets of any line as a launch carries them.
struct CellMap {
    uint32_t t[kMostLineSlots];
};

template <int kWords>
struct alignas(kWords * 4 < 16 ? kWords * 4 : 16) CellSlot {
    uint32_t w[kWords];
};

template <int F, typename T>
__device__ __forceinline__ CellSlot<F * sizeof(T) / 4> round_slot(const float* __restrict__ from) {
    float v[F];
    if constexpr (F == 2) {
        const float2 x = *reinterpret_cast<const float2*>(from);
        v[0] = x.x;
        v[1] = x.y;
    } else {
#pragma unroll
        for (int q = 0; q < F / 4; ++q) {
            const float4 x = reinterpret_cast<const float4*>(from)[q];
            v[4 * q + 0] = x.x;
            v[4 * q + 1] = x.y;
            v[4 * q + 2] = x.z;
            v[4 * q + 3] = x.w;
        }
    }
    CellSlot<F * sizeof(T) / 4> slot;
#pragma unroll
    for (int k = 0; k < F; k += 2) {
        uint32_t lo, hi;
        if constexpr (std::is_same<T, bfloat16_bits>::value) {
            lo = to_bfloat16(v[k]);
            hi = to_bfloat16(v[k + 1]);
        } else {
            lo = __half_as_ushort(__float2half_rn(v[k]));
            hi = __half_as_ushort(__float2half_rn(v[k + 1]));
        }
        slot.w[k / 2] = lo | (hi << 16);
    }
    return slot;
}

// A slot of `from`, which is fp32 (kRaw = false) or of the type T itself.
template <int F, typename T, bool kRaw>
__device__ __forceinline__ CellSlot<F * sizeof(T) / 4> convert_slot(const void* __restrict__ table, size_t index) {
    if constexpr (kRaw) return static_cast<const CellSlot<F * sizeof(T) / 4>*>(table)[index];
    else return round_slot<F, T>(static_cast<const float*>(table) + index * F);
}

// columns[level][i][line] = the table's slot i of `line`, converted.
template <int F, typename T, bool kRaw>
__global__ void __launch_bounds__(kCellBlock)
cell_columns_kernel(const void* __restrict__ table, uint32_t lines, void* __restrict__ columns) {
    constexpr int kSlots = line_slots<F, T>();
    using Slot = CellSlot<F * sizeof(T) / 4>;
    constexpr int kPitch = kCellLines + 64 / kSlots;  // the 64 / kSlots lines that a wave writes at a time end up in banks of their own
    __shared__ Slot tile[kSlots * kPitch];
    const uint32_t first = blockIdx.x * kCellLines, count = lines - first < kCellLines ? lines - first : kCellLines;
    const size_t level_first = static_cast<size_t>(blockIdx.y) * lines * kSlots;  // in slots
    const size_t from = level_first + static_cast<size_t>(first) * kSlots;
    constexpr int kEach = kCellLines * kSlots / kCellBlock;
    Slot slot[kEach];
#pragma unroll
    for (int k = 0; k < kEach; ++k) {
        const uint32_t e = k * kCellBlock + threadIdx.x;
        slot[k] = convert_slot<F, T, kRaw>(table, from + (e < count * kSlots ? e : 0u));
    }
#pragma unroll
    for (int k = 0; k < kEach; ++k) {
        const uint32_t e = k * kCellBlock + threadIdx.x;
        tile[(e % kSlots) * kPitch + e / kSlots] = slot[k];
    }
    __syncthreads();
    Slot* const to = static_cast<Slot*>(columns) + level_first + first;
#pragma unroll
    for (int k = 0; k < kEach; ++k) {
        const uint32_t e = k * kCellBlock + threadIdx.x, i = e / kCellLines, line = e % kCellLines;
        if (line < count) to[static_cast<size_t>(i) * lines + line] = tile[i * kPitch + line];
    }
}

// cells[level][line][i] = columns[level][i][line + T[i]/B], lines counted round.
template <int kWords>
__global__ void __launch_bounds__(kCellBlock)
cell_lines_kernel(const void* __restrict__ columns, uint32_t lines, CellMap map, void* __restrict__ cells) {
    constexpr int kSlots = kLineBytes / (kWords * 4);
    using Slot = CellSlot<kWords>;
    constexpr int kPitch = kSlots + 1;
    __shared__ Slot tile[kCellLines * kPitch];
    const uint32_t first = blockIdx.x * kCellLines, count = lines - first < kCellLines ? lines - first : kCellLines;
    const size_t level_first = static_cast<size_t>(blockIdx.y) * lines * kSlots;
    const Slot* const from = static_cast<const Slot*>(columns) + level_first;
    constexpr int kEach = kCellLines * kSlots / kCellBlock;
    Slot slot[kEach];
#pragma unroll
    for (int k = 0; k < kEach; ++k) {
        const uint32_t e = k * kCellBlock + threadIdx.x, line = e % kCellLines;
        const uint32_t i = __builtin_amdgcn_readfirstlane(e / kCellLines);  // (a wave is in one column)
        slot[k] = from[static_cast<size_t>(i) * lines + ((first + line + map.t[i] / kSlots) & (lines - 1u))];
    }
#pragma unroll
    for (int k = 0; k < kEach; ++k) {
        const uint32_t e = k * kCellBlock + threadIdx.x;
        tile[(e % kCellLines) * kPitch + e / kCellLines] = slot[k];
    }
    __syncthreads();
    Slot* const to = static_cast<Slot*>(cells) + level_first + static_cast<size_t>(first) * kSlots;
#pragma unroll
    for (int k = 0; k < kEach; ++k) {
        const uint32_t e = k * kCellBlock + threadIdx.x;
        if (e < count * kSlots) to[e] = tile[(e / kSlots) * kPitch + e % kSlots];
    }
}

// ------------------------------------------------------------------------------------------
// a copy for one forward
//
// The table of a training step is another one in every step, so a copy of an fp32 table serves one forward, and what it costs must be less than
// what that forward gains: for levels that an L2 holds, one die to a level, so that the columns can be read where they are (a request for every
// slot, as in a gather), and of those only the levels where most gathers of a wave are lines of their own.  (Where lanes share lines the
// first-level cache serves them, from either copy alike: the coarse half of 24 levels for unordered points, all but the finest for samples along
// rays.)  Every workgroup of a level looks at the same points, a stretch of 64 from the beginning of each quarter of the batch, and counts a wave's
// lines as bits of a small map; the first says what they found.
// Forward of 2^20 unordered points, 24 levels of 2^18 slots, D = 3: 280 -> 237 us with 16 levels chosen (all of them, or the 16 in two passes through
// columns, 246 and 244; one, two, four times kCellLines lines to a workgroup 241 / 237 / 239), D = 4 377 -> 344.
constexpr int kCellsPerWorkgroup = 2;   // times kCellLines lines
constexpr uint32_t kSampleBits = 4096;  // of a wave's map: up to 8 x 64 lines
template <int D, int F>
__global__ void __launch_bounds__(kCellBlock)
chosen_cells_kernel(const float* __restrict__ table, uint32_t lines, uint32_t n_levels, uint32_t per_level, uint32_t dies, CellMap map, int64_t n_points,
                    const float* __restrict__ positions, const float* __restrict__ scale_factor, const float* __restrict__ random_shift,
                    const float* __restrict__ window, uint32_t* __restrict__ chosen, float* __restrict__ cells) {
    constexpr int kWaves = kCellBlock / 64, kSlots = line_slots<F, float>(), kPitch = kSlots + 1;
    using Slot = CellSlot<F>;
    __shared__ Slot tile[kCellLines * kPitch];
    __shared__ uint32_t seen[kWaves][kSampleBits / 32];
    __shared__ uint32_t distinct;
    const uint32_t j = blockIdx.x / dies, level = j / per_level * dies + blockIdx.x % dies, part = j % per_level;
    if (level >= n_levels) return;
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    bool mine = false;
    if (window[level] != 0.0f) {
        int64_t n = n_points / kWaves * wave + lane;
        n = n < n_points ? n : n_points - 1;
        const float* const p = positions + n * D;
        fvec<D> pos;
        static_for<D>(PENC_BODY(k) {
            PENC_INDEX(k); pos[k] = p[k]; });
        for (uint32_t i = lane; i < kSampleBits / 32; i += 64) seen[wave][i] = 0u;
        if (threadIdx.x == 0) distinct = 0u;
        const Located<D> at = locate<D>(pos, random_shift + level * D, scale_factor + level * D);
        const uvec<D + 1> h = vertex_hashes<D>(at.rank, at.hash0);
        __syncthreads();
        static_for<D + 1>(PENC_BODY(r) {
            PENC_INDEX(r);
            const uint32_t line = (h[r] / kSlots) & (lines - 1u), bit = (line * 0x9E3779B1u) / (0xFFFFFFFFu / kSampleBits + 1u);
            atomicOr(&seen[wave][bit / 32], 1u << (bit % 32));
        });
        wave_lds_fence();
        uint32_t count = 0u;
        for (uint32_t i = lane; i < kSampleBits / 32; i += 64) count += __popc(seen[wave][i]);
        if (count != 0u) atomicAdd(&distinct, count);
        __syncthreads();
        mine = distinct * 8u >= static_cast<uint32_t>(5 * (D + 1) * kCellBlock);
    }
    if (part == 0u && threadIdx.x == 0) chosen[level] = mine ? 1u : 0u;
    if (!mine) return;
    const Slot* const from = reinterpret_cast<const Slot*>(table) + static_cast<size_t>(level) * lines * kSlots;
    Slot* const to = reinterpret_cast<Slot*>(cells) + static_cast<size_t>(level) * lines * kSlots;
    constexpr int kEach = kCellLines * kSlots / kCellBlock;
    for (uint32_t first = part * (kCellsPerWorkgroup * kCellLines), end = first + kCellsPerWorkgroup * kCellLines; first < end && first < lines; first += kCellLines) {
        Slot slot[kEach];
#pragma unroll
        for (int k = 0; k < kEach; ++k) {
            const uint32_t e = k * kCellBlock + threadIdx.x, line = e % kCellLines;
            const uint32_t i = __builtin_amdgcn_readfirstlane(e / kCellLines);  // (a wave is in one column)
            slot[k] = from[((first + line + map.t[i] / kSlots) & (lines - 1u)) * kSlots + i];
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kEach; ++k) {
            const uint32_t e = k * kCellBlock + threadIdx.x;
            tile[(e % kCellLines) * kPitch + e / kCellLines] = slot[k];
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kEach; ++k) {
            const uint32_t e = k * kCellBlock + threadIdx.x;
            if (first + e / kSlots < lines) to[static_cast<size_t>(first) * kSlots + e] = tile[(e / kSlots) * kPitch + e % kSlots];
        }
    }
}

// ------------------------------------------------------------------------------------------
// host side

inline CellMap cell_map(int pos_dim, int slots) {
    const CellOffsets& all = pos_dim == 2 ? kCells<2> : pos_dim == 3 ? kCells<3> : pos_dim == 4 ? kCells<4> : pos_dim == 5 ? kCells<5>
                             : pos_dim == 6 ? kCells<6> : pos_dim == 7 ? kCells<7> : kCells<8>;
    CellMap map{};
    for (int i = 0; i < slots; ++i) map.t[i] = all.t[cells_at(slots) + i];
    return map;
}

}  // namespace penc
