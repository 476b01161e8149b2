// Device-side geometry of the permutohedral lattice for gfx950: everything a kernel derives from
// one (point, level) pair before it touches the hash table.
//
// The arithmetic that decides WHICH simplex and WHICH table slots a point uses is written so that
// it rounds exactly like the CPU checker's: fp32, no implicit contraction (the translation unit is
// compiled with -ffp-contract=off) and one explicit fused multiply-add in the elevation
// (reference: kernels/permutohedral_encoding/EncodingGPU.cuh:130-138, which the reference's
// compiler contracts the same way).
//
// The small per-thread arrays (D+1 residuals, ranks, weights ...) are held in vector VALUES
// (ext_vector_type) indexed only by compile-time constants, and are passed between the helpers
// by value, so that they are registers by construction and never addressable memory.  The reference indexes its barycentric array with a run-time rank
// (EncodingGPU.cuh:195-196), which on a GPU forces the array into scratch memory; here the
// residuals are first put in rank order with compare/select chains, after which every index is
// a compile-time constant:
//
//     sorted[m]  = residual of the coordinate whose rank is m            (m = 0..D)
//     weight[0]  = sorted[D] + (1 - sorted[0])
//     weight[r]  = sorted[D-r] - sorted[D+1-r]                           (r = 1..D)
//
// which is term for term what the reference's "+= delta / -= delta" loop accumulates.
//
// The hash (EncodingGPU.cuh:22-32) is a polynomial in the key coordinates modulo 2^32,
//     h(key) = sum_i key[i] * M^(D-i),  M = 2531011,
// and vertex r of the simplex has key[i] = rem0[i] + r - (D+1)*[rank[i] > D-r]
// (EncodingGPU.cuh:216-220), so consecutive vertices differ by a constant minus one power:
//     h_0     = sum_i rem0[i] * M^(D-i)
//     h_{r+1} = h_r + sum_i M^(D-i) - (D+1) * M^(D-c),   c = the coordinate whose rank is D-r
// (no term when c is the implied last coordinate).  All of it is wrapping uint32 arithmetic, so
// the slots are bit-identical to evaluating the reference's loop per vertex, at D multiplies per
// point instead of D*(D+1).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <utility>

namespace penc {

// Per-thread short arrays as SSA vector values.  They are deliberately not C arrays: a helper
// that receives `const float (&a)[N]` is optimised on its own before it is inlined, and there the
// optimiser turns a compare/select chain over a[0..N-1] into ONE load from a run-time-selected
// address, which after inlining pins the caller's array in scratch memory or LDS.  A vector
// passed by value has no address, so element access stays extractelement/insertelement.
template <int N> using fvec = float __attribute__((ext_vector_type(N)));
template <int N> using ivec = int __attribute__((ext_vector_type(N)));
template <int N> using uvec = uint32_t __attribute__((ext_vector_type(N)));

// Compile-time loop: body(integral_constant<int, 0>) ... body(integral_constant<int, N-1>), so
// that every vector index below is a constant expression.
template <typename F, int... Is>
__device__ __forceinline__ void static_for_impl(F&& body, std::integer_sequence<int, Is...>) {
    (body(std::integral_constant<int, Is>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& body) {
    static_for_impl(static_cast<F&&>(body), std::make_integer_sequence<int, N>{});
}
// Loop body as a lambda: `PENC_BODY(i) { PENC_INDEX(i); ... }` makes `i` a constant expression.
#define PENC_BODY(var) [&](auto var##_constant) __attribute__((always_inline))
#define PENC_INDEX(var) constexpr int var = decltype(var##_constant)::value

constexpr uint32_t kHashMul = 2531011u;

constexpr uint32_t hash_pow(int e) {
    uint32_t r = 1u;
    for (int k = 0; k < e; ++k) r *= kHashMul;
    return r;
}

template <int D>
constexpr uint32_t hash_pow_sum() {
    uint32_t s = 0u;
    for (int i = 0; i < D; ++i) s += hash_pow(D - i);
    return s;
}

// Increment of the raw hash from one simplex vertex to the next when coordinate C is the one
// that starts to wrap (C == D: the implied last coordinate, which is not hashed).
template <int D, int C>
constexpr uint32_t hash_step() {
    return C < D ? hash_pow_sum<D>() - static_cast<uint32_t>(D + 1) * hash_pow(D - C) : hash_pow_sum<D>();
}

// Reduces a raw 32-bit hash to a table slot (EncodingGPU.cuh:34-36).  `cap_mask` is capacity-1
// when the capacity is a power of two and 0 otherwise.
__device__ __forceinline__ uint32_t to_slot(uint32_t h, uint32_t capacity, uint32_t cap_mask) {
    return cap_mask ? (h & cap_mask) : (h % capacity);
}

template <int D>
struct Located {
    ivec<D + 1> rem0;    // remainder-0 lattice point, after the hyperplane wrap
    ivec<D + 1> rank;    // rank of each coordinate's residual, after the wrap (a permutation of 0..D)
    fvec<D + 1> delta;   // (elevated[i] - rem0[i]) / (D+1)
    uint32_t hash0;      // raw hash of vertex 0
};

template <int D>
struct Rounded {
    fvec<D + 1> resid;     // (elevated - rounded) / kUnit: exact in fp32 (the two are within (D+1)/2 of each other)
    ivec<D + 1> multiple;  // rounded / kUnit
    int sum;               // of the rounded coordinates, in units of D+1
    // Where D+1 is a power of two, dividing by it is exact and everything is kept divided (kUnit is what resid and `multiple` count in).
    static constexpr bool kExactInverse = ((D + 1) & D) == 0;
    static constexpr float kUnit = kExactInverse ? static_cast<float>(D + 1) : 1.0f;
};

// Elevate and round (EncodingGPU.cuh:130-158) for one point at one level.
// `shift` and `sf` point at this level's D random shifts and D scale factors.
template <int D, bool kLowerAtTies = true>
__device__ __forceinline__ Rounded<D> elevate_and_round(fvec<D> pos, const float* __restrict__ shift, const float* __restrict__ sf) {
    constexpr int D1 = D + 1;
    constexpr float kInv = 1.0f / D1;
    fvec<D1> elevated;
    float sm = 0.0f;
    static_for<D>(PENC_BODY(k) {
        PENC_INDEX(k);
        constexpr int i = D - k;  // i = D .. 1
        const float cf = (pos[i - 1] + shift[i - 1]) * sf[i - 1];
        elevated[i] = __builtin_fmaf(-static_cast<float>(i), cf, sm);
        sm += cf;
    });
    elevated[0] = sm;

    // Round every coordinate to the nearer multiple of D+1, the lower one at a tie (:149-158).  The
    // upper candidate is formed as down + (D+1) instead of ceil(v)*(D+1): the two differ only when v
    // is an integer, where the reference's candidates coincide and the lower one is chosen here too.
    // Where D+1 is a power of two the nearer integer is one instruction, which takes the even one at a tie, and the lower one has to be put right
    // where that was the upper (unless a caller may do without: see cyclic_simplex).
    Rounded<D> o;
    o.sum = 0;
    static_for<D1>(PENC_BODY(i) {
        PENC_INDEX(i);
        const float e = elevated[i];
        if constexpr (Rounded<D>::kExactInverse) {
            const float v = e * kInv, nearest = __builtin_rintf(v), r = v - nearest;
            const bool lower = kLowerAtTies && r == -0.5f;
            o.multiple[i] = static_cast<int>(nearest) - (lower ? 1 : 0);
            o.resid[i] = lower ? 0.5f : r;
        } else {
            const float down = __builtin_floorf(e * kInv) * static_cast<float>(D1);
            const float up = down + static_cast<float>(D1);
            const float b = (up - e < e - down) ? up : down;
            o.multiple[i] = static_cast<int>(b);
            o.resid[i] = e - b;
        }
        o.sum += o.multiple[i];
    });
    if constexpr (!Rounded<D>::kExactInverse) o.sum /= D1;
    return o;
}

// Elevate, round, rank, wrap (EncodingGPU.cuh:130-186) for one point at one level.
template <int D>
__device__ __forceinline__ Located<D> locate(fvec<D> pos, const float* __restrict__ shift,
                                             const float* __restrict__ sf) {
    constexpr int D1 = D + 1;
    constexpr float kInv = 1.0f / D1;
    constexpr bool kExactInverse = Rounded<D>::kExactInverse;
    constexpr float kUnit = Rounded<D>::kUnit;
    const Rounded<D> rounded = elevate_and_round<D>(pos, shift, sf);
    const fvec<D1> resid = rounded.resid;
    const ivec<D1> multiple = rounded.multiple;
    const int sum = rounded.sum;

    ivec<D1> rank = 0;
    static_for<D>(PENC_BODY(i) {
        PENC_INDEX(i);
        static_for<D - i>(PENC_BODY(jj) {
        PENC_INDEX(jj);
            constexpr int j = i + 1 + jj;
            const int lt = resid[i] < resid[j] ? 1 : 0;
            rank[i] += lt;
            rank[j] += 1 - lt;
        });
    });

    // Wrap back onto the hyperplane (:173-186): a rank pushed outside 0..D by the coordinate sum comes
    // back by D+1 and takes its rem0 along.  `moved` is that multiple of D+1 (0 or +-(D+1)).  The
    // residual after the wrap, elevated - (rounded + moved), is one rounding of an exact difference
    // whichever way it is bracketed, so it is formed from the (exact) residual before the wrap.
    Located<D> o;
    uint32_t h = 0u;
    static_for<D1>(PENC_BODY(i) {
        PENC_INDEX(i);
        const int rk = rank[i] + sum;
        int wrapped_rank;
        if constexpr ((D1 & (D1 - 1)) == 0) {
            wrapped_rank = rk & (D1 - 1);  // rk is within D+1 of 0..D: reduction modulo a power of two
        } else {
            wrapped_rank = rk < 0 ? rk + D1 : (rk > D ? rk - D1 : rk);
        }
        const int moved = wrapped_rank - rk;
        o.rank[i] = wrapped_rank;
        const int r0 = static_cast<int>(static_cast<uint32_t>(multiple[i]) * static_cast<uint32_t>(kUnit)) + moved;
        o.rem0[i] = r0;
        if constexpr (kExactInverse) o.delta[i] = __builtin_fmaf(static_cast<float>(moved), -kInv, resid[i]);  // (the product is exact: one rounding)
        else o.delta[i] = (resid[i] - static_cast<float>(moved)) * kInv;
        if constexpr (i < D) h += static_cast<uint32_t>(r0) * hash_pow(D - i);
    });
    o.hash0 = h;
    return o;
}

// Per-coordinate values put in rank order: out[m] = in[c] where rank[c] == m.
template <int D>
__device__ __forceinline__ fvec<D + 1> by_rank(ivec<D + 1> rank, fvec<D + 1> in) {
    fvec<D + 1> out;
    static_for<D + 1>(PENC_BODY(m) {
        PENC_INDEX(m);
        float acc = in[0];
        static_for<D>(PENC_BODY(cc) {
        PENC_INDEX(cc);
            constexpr int c = cc + 1;
            const float x = in[c];
            acc = (rank[c] == m) ? x : acc;
        });
        out[m] = acc;
    });
    return out;
}

template <int D>
__device__ __forceinline__ fvec<D + 1> barycentric_of_sorted(fvec<D + 1> sorted) {
    fvec<D + 1> w;
    w[0] = sorted[D] + (1.0f + (0.0f - sorted[0]));
    static_for<D>(PENC_BODY(rr) {
        PENC_INDEX(rr);
        constexpr int r = rr + 1;
        w[r] = sorted[D - r] - sorted[D + 1 - r];
    });
    return w;
}

// Barycentric weights of the D+1 vertices (EncodingGPU.cuh:190-199).
template <int D>
__device__ __forceinline__ fvec<D + 1> barycentric(ivec<D + 1> rank, fvec<D + 1> delta) {
    return barycentric_of_sorted<D>(by_rank<D>(rank, delta));
}

// Raw hashes of the D+1 vertices (EncodingGPU.cuh:212-223), by the incremental rule above.
template <int D>
__device__ __forceinline__ uvec<D + 1> vertex_hashes(ivec<D + 1> rank, uint32_t hash0) {
    uvec<D + 1> h;
    h[0] = hash0;
    static_for<D>(PENC_BODY(r) {
        PENC_INDEX(r);
        // the coordinate of rank D-r starts to wrap between vertex r and vertex r+1
        uint32_t step = hash_step<D, 0>();
        static_for<D>(PENC_BODY(cc) {
        PENC_INDEX(cc);
            constexpr int c = cc + 1;
            step = (rank[c] == D - r) ? hash_step<D, c>() : step;
        });
        h[r + 1] = h[r] + step;
    });
    return h;
}

// The same two results (residuals in rank order, raw vertex hashes) through LDS instead of the
// D(D+1) compare-and-select chains above: every thread owns a column of D+1 eight-byte cells
// (`column` points at the thread's cell of row 0, rows are `stride` cells apart, so the lanes of a
// wave hit distinct banks), writes {delta[c], hash step of coordinate c} to row rank[c] and reads
// the rows back in order.  A thread only reads what it wrote itself: no barrier.
template <int D>
__device__ __forceinline__ void sort_by_rank_lds(uint2* column, uint32_t stride, ivec<D + 1> rank, fvec<D + 1> delta,
                                                 uint32_t hash0, fvec<D + 1>& sorted, uvec<D + 1>& hashes) {
    static_for<D + 1>(PENC_BODY(c) {
        PENC_INDEX(c);
        const float d = delta[c];
        uint2 cell;
        cell.x = __builtin_bit_cast(uint32_t, d);
        cell.y = hash_step<D, c>();
        // ranks of finite points are a permutation of 0..D; the clamp keeps a point with NaN or
        // overflowing coordinates inside its own column
        const int row = rank[c] < 0 ? 0 : (rank[c] > D ? D : rank[c]);
        column[static_cast<uint32_t>(row) * stride] = cell;
    });
    uvec<D + 1> step;
    static_for<D + 1>(PENC_BODY(m) {
        PENC_INDEX(m);
        const uint2 cell = column[m * stride];
        sorted[m] = __builtin_bit_cast(float, cell.x);
        step[m] = cell.y;
    });
    hashes[0] = hash0;
    static_for<D>(PENC_BODY(r) {
        PENC_INDEX(r);
        hashes[r + 1] = hashes[r] + step[D - r];  // the coordinate of rank D-r starts to wrap here
    });
}

// The three gradient chains below evaluate their sums in the same order, with the same
// intermediate roundings, as the reference's loops, so that every term a kernel adds is the same
// fp32 number the CPU checker computes; only the order of atomic accumulation can then differ.

// d(loss)/d(barycentric) -> d(loss)/d(position) for one level (EncodingGPU.cuh:698-740), in three
// steps.  dB[r] is the derivative w.r.t. the weight of vertex r.
// Step 1: dE[i] = dB[D-rank[i]]/(D+1) - dB[D+1-rank[i]]/(D+1), with dB[D+1] = dB[0] (the wrap-around
// term, :698), as a function of the rank m: diff[m] = dB[D-m]/(D+1) - dB[D+1-m]/(D+1).
template <int D>
__device__ __forceinline__ fvec<D + 1> bary_grad_by_rank(fvec<D + 1> dB) {
    constexpr int D1 = D + 1;
    constexpr float kInv = 1.0f / D1;
    const fvec<D1> scaled = dB * kInv;
    fvec<D1> diff;
    diff[0] = scaled[D] - scaled[0];
    static_for<D>(PENC_BODY(mm) {
        PENC_INDEX(mm);
        constexpr int m = mm + 1;
        diff[m] = scaled[D - m] - scaled[D1 - m];
    });
    return diff;
}

// Step 2: dE[i] = diff[rank[i]], by compare-and-select chains.
template <int D>
__device__ __forceinline__ fvec<D + 1> pick_by_rank(ivec<D + 1> rank, fvec<D + 1> diff) {
    fvec<D + 1> dE;
    static_for<D + 1>(PENC_BODY(i) {
        PENC_INDEX(i);
        float acc = diff[0];
        static_for<D>(PENC_BODY(mm) {
            PENC_INDEX(mm);
            constexpr int m = mm + 1;
            const float x = diff[m];
            acc = (rank[i] == m) ? x : acc;
        });
        dE[i] = acc;
    });
    return dE;
}

// Step 3: dP[i] = sum_{j<=i} dE[j]*sf[i] - dE[i+1]*sf[i]*(i+1)   (:729-740)
template <int D>
__device__ __forceinline__ fvec<D> elevated_grad_to_pos_grad(fvec<D + 1> dE, const float* __restrict__ sf) {
    fvec<D> dP;
    static_for<D>(PENC_BODY(i) {
        PENC_INDEX(i);
        float acc = dE[0] * sf[i];
        static_for<i>(PENC_BODY(jj) {
            PENC_INDEX(jj);
            acc += dE[jj + 1] * sf[i];
        });
        acc -= dE[i + 1] * sf[i] * static_cast<float>(i + 1);
        dP[i] = acc;
    });
    return dP;
}

template <int D>
__device__ __forceinline__ fvec<D> bary_grad_to_pos_grad(ivec<D + 1> rank, fvec<D + 1> dB,
                                                         const float* __restrict__ sf) {
    return elevated_grad_to_pos_grad<D>(pick_by_rank<D>(rank, bary_grad_by_rank<D>(dB)), sf);
}

// d(loss)/d(position gradient) -> derivative w.r.t. each vertex weight (EncodingGPU.cuh:1187-1218),
// in two steps with the permutation into rank order between them.
// Step 1: the derivative w.r.t. the elevated coordinates, already divided by D+1.
template <int D>
__device__ __forceinline__ fvec<D + 1> pos_grad_grad_to_elevated(fvec<D> q, const float* __restrict__ sf) {
    constexpr int D1 = D + 1;
    constexpr float kInv = 1.0f / D1;
    fvec<D> g;
    static_for<D>(PENC_BODY(i) {
        PENC_INDEX(i);
        g[i] = q[i] * sf[i];
    });
    // dE[j] = g[j] + g[j+1] + ... + g[D-1] (summed in ascending order, :1187-1194), then
    // dE[j] -= g[j-1]*j (:1196-1199)
    fvec<D1> dE;
    dE[D] = 0.0f;
    static_for<D>(PENC_BODY(j) {
        PENC_INDEX(j);
        float acc = g[j];
        static_for<D - 1 - j>(PENC_BODY(k) {
            PENC_INDEX(k);
            acc += g[j + 1 + k];
        });
        dE[j] = acc;
    });
    static_for<D>(PENC_BODY(jj) {
        PENC_INDEX(jj);
        constexpr int j = jj + 1;
        dE[j] -= g[j - 1] * static_cast<float>(j);
    });
    dE *= kInv;
    return dE;
}

// Step 2, from dE in rank order: dB[k] = sorted[D-k] - sorted[D+1-k]; dB[D+1] = -sorted[0] is folded
// into dB[0] (:1218).
template <int D>
__device__ __forceinline__ fvec<D + 1> sorted_elevated_grad_to_bary(fvec<D + 1> sorted) {
    constexpr int D1 = D + 1;
    fvec<D1> dB;
    dB[0] = sorted[D] + (0.0f - sorted[0]);
    static_for<D>(PENC_BODY(rr) {
        PENC_INDEX(rr);
        constexpr int r = rr + 1;
        dB[r] = sorted[D - r] - sorted[D1 - r];
    });
    return dB;
}

template <int D>
__device__ __forceinline__ fvec<D + 1> pos_grad_grad_to_bary(ivec<D + 1> rank, fvec<D> q,
                                                             const float* __restrict__ sf) {
    return sorted_elevated_grad_to_bary<D>(by_rank<D>(rank, pos_grad_grad_to_elevated<D>(q, sf)));
}

// ------------------------------------------------------------------------------------------
// the same simplex, its vertices in cyclic order
//
// A scatter adds every vertex's contribution on its own, so it needs the vertices' weights and slots but not which of them is which.
// Then the residuals can be sorted as they are, before the wrap, and neither ranks nor the selects that bring D+1 values into
// rank order are needed: with m the place in descending order, s[m] the residual and c_m its coordinate, and everything modulo D+1,
//     place m wraps by q_m = floor((m + sum) / (D+1))                    (-1, 0 or 1: the reference's rank + sum beyond 0..D)
//     d[m]   = (s[m] + (D+1) q_m) / (D+1)                                (its delta after the wrap)
//     w_k    = d[D-k] - d[D+1-k], and 1 more where between the two the wrap begins, or does not and k = 0
//     h_0    = sum_i rounded_i M^(D-i) - sum * sum_i M^(D-i),   h_{k+1} = h_k + hash step of c_{D-k}
// are weight and raw hash of remainder vertex r = k - sum, the same fp32 numbers as those of the functions above (the steps of all
// coordinates add up to zero, so the chain closes: it may begin at any vertex).  `turned` is sum modulo D+1: turn_back() brings them into the order of r.
//
// The sort is a network of compare-exchanges, each two instructions (v_max_f64, v_min_f64, at the rate of an fp32 comparison on gfx950): a key is a double
// whose upper word is the residual's fp32 bits, which order doubles as they order floats, and whose lower word, the hash step, comes along.
// Equal residuals have to be taken in the order of their coordinates (the lower first): the upper four bits of the lower word see to that, reversed
// for negative residuals, whose order by magnitude is the reverse; the steps then count modulo 2^28, which capacities that are powers of two up to that
// hide, and for others the upper bits are put back.  Where D+1 is a power of two and only barycentric weights are wanted, the vertex that two equal residuals
// leave open has the weight 0 exactly, and a residual of a half is as good on either side: neither is looked after (kOpenTies).
// Against ranks, selects and trips through the LDS: the scatter of 2^20 points, 24 levels of 2^18 slots, D = 3 issues 94 M vector instructions instead of 120 M
// (2^19 points, 16 levels of 2^19 slots, D = 8: 100 M of 113 M, and 18 KB of LDS less); it is bound by them at the coarse levels only, so a training step with it
// goes 726 -> 722 us (D = 8: 715 -> 701; the gradient of both orders, 2^22 slots, 1239 -> 1230).  The values of the second order ride along, a comparison and two selects an
// exchange: kept in LDS columns and fetched by the coordinate a key names after the sort they took as many registers, and the scatters of both orders, D = 6 to 8, 0.5% less time.
template <int N> using dvec = double __attribute__((ext_vector_type(N)));

// Compare-exchanges (place of the larger, place of the smaller) that sort N keys: networks of the fewest, as B. Dobbelaere's published list of the smallest known ones has them
// (up to eight keys optimal by Knuth, The Art of Computer Programming 3, 5.3.4; the 25 for nine by Floyd), each checked below.
struct SortingNetwork {
    int count;
    int a[25], b[25];
};
template <int N>
constexpr SortingNetwork sorting_network() {
    static_assert(N >= 3 && N <= 9, "networks for 3 to 9 keys");
    if constexpr (N == 3) return {3, {0, 0, 1}, {2, 1, 2}};
    else if constexpr (N == 4) return {5, {0, 1, 0, 2, 1}, {2, 3, 1, 3, 2}};
    else if constexpr (N == 5) return {9, {0, 1, 0, 1, 0, 2, 1, 3, 2}, {3, 4, 2, 3, 1, 4, 2, 4, 3}};
    else if constexpr (N == 6) return {12, {0, 1, 2, 1, 3, 0, 2, 0, 2, 4, 1, 3}, {5, 3, 4, 2, 4, 3, 5, 1, 3, 5, 2, 4}};
    else if constexpr (N == 7) return {16, {0, 2, 4, 0, 1, 3, 0, 2, 3, 1, 4, 2, 4, 1, 3, 5}, {6, 3, 5, 2, 4, 6, 1, 5, 4, 2, 6, 3, 5, 2, 4, 6}};
    else if constexpr (N == 8)
        return {19, {0, 1, 4, 5, 0, 1, 2, 3, 0, 2, 4, 6, 2, 3, 1, 3, 1, 3, 5}, {2, 3, 6, 7, 4, 5, 6, 7, 1, 3, 5, 7, 4, 5, 4, 6, 2, 4, 6}};
    else
        return {25, {0, 1, 2, 4, 0, 2, 3, 5, 0, 1, 4, 7, 1, 3, 5, 0, 2, 3, 6, 2, 4, 6, 1, 3, 5},
                {3, 7, 5, 8, 7, 4, 8, 6, 2, 3, 5, 8, 4, 6, 7, 1, 4, 5, 8, 3, 5, 7, 2, 4, 6}};
}
// (a network that sorts all sequences of zeros and ones sorts everything)
template <int N>
constexpr bool sorts_everything() {
    const SortingNetwork net = sorting_network<N>();
    for (uint32_t keys = 0; keys < (1u << N); ++keys) {
        uint32_t k = keys;
        for (int e = 0; e < net.count; ++e) {
            const uint32_t larger = (k >> net.a[e]) & 1u, smaller = (k >> net.b[e]) & 1u;
            if (larger < smaller) k ^= (1u << net.a[e]) | (1u << net.b[e]);
        }
        if ((k & (k + 1u)) != 0u) return false;  // the ones are the first places
    }
    return true;
}
template <int N>
constexpr SortingNetwork kNetwork = sorting_network<N>();
static_assert(sorts_everything<3>() && sorts_everything<4>() && sorts_everything<5>() && sorts_everything<6>() && sorts_everything<7>() &&
                  sorts_everything<8>() && sorts_everything<9>(),
              "every network sorts");

// v_max_f64 and v_min_f64 as they are: the builtins would first quiet operands that might be signalling NaNs.  A key is a NaN only where its residual is one with
// payload bits of its own (the hardware's has none but the first); such a point's slots are as meaningless as any NaN's, and within the table.
__device__ __forceinline__ double larger_key(double a, double b) {
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ double smaller_key(double a, double b) {
    double r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ double make_key(uint32_t lower, float upper) {
    return __builtin_bit_cast(double, (static_cast<uint64_t>(__builtin_bit_cast(uint32_t, upper)) << 32) | lower);
}

constexpr uint32_t kKeyStepBits = 28;
template <int D, int... C>
constexpr uint64_t upper_step_bits(std::integer_sequence<int, C...>) {  // the upper four bits of coordinate c's hash step at 4 (D - c)
    return ((static_cast<uint64_t>(hash_step<D, C>() >> kKeyStepBits) << (4 * (D - C))) | ...);
}

template <int D>
struct CyclicSimplex {
    fvec<D + 1> w;         // barycentric weights (kFirst)
    fvec<D + 1> dB;        // derivatives of the weights along the direction given (kSecond; see pos_grad_grad_to_bary)
    uvec<D + 1> slot;
    int turned;
};

template <int D, bool kFirst, bool kSecond>
__device__ __forceinline__ CyclicSimplex<D> cyclic_simplex(fvec<D> pos, fvec<D> q, const float* __restrict__ shift, const float* __restrict__ sf,
                                                           uint32_t capacity, uint32_t cap_mask) {
    constexpr int D1 = D + 1;
    constexpr float kInv = 1.0f / D1;
    constexpr bool kExactInverse = Rounded<D>::kExactInverse;
    constexpr bool kOpenTies = kExactInverse && !kSecond;
    constexpr uint32_t kOrderBits = ~((1u << kKeyStepBits) - 1u);
    const Rounded<D> rounded = elevate_and_round<D, !kOpenTies>(pos, shift, sf);
    const int sum = rounded.sum;

    uint32_t h0 = 0u;
    dvec<D1> key;
    static_for<D1>(PENC_BODY(c) {
        PENC_INDEX(c);
        const float r = rounded.resid[c];
        if constexpr (c < D) h0 += static_cast<uint32_t>(rounded.multiple[c]) * (static_cast<uint32_t>(Rounded<D>::kUnit) * hash_pow(D - c));
        if constexpr (kOpenTies) {
            key[c] = make_key(hash_step<D, c>(), r);
        } else {
            constexpr uint32_t kLower = (static_cast<uint32_t>(D - c) << kKeyStepBits) | (hash_step<D, c>() & ~kOrderBits);
            key[c] = make_key(kLower ^ (static_cast<uint32_t>(__builtin_bit_cast(int, r) >> 31) & kOrderBits), r);
        }
    });
    h0 -= static_cast<uint32_t>(sum) * hash_pow_sum<D>();
    fvec<D1> along = 0.0f;  // d(weights)/d(elevated coordinates) along the direction, in the order of the keys
    if constexpr (kSecond) along = pos_grad_grad_to_elevated<D>(q, sf);

    static_for<kNetwork<D1>.count>(PENC_BODY(e) {
        PENC_INDEX(e);
        constexpr int a = kNetwork<D1>.a[e], b = kNetwork<D1>.b[e];
        const double x = key[a], y = key[b];
        if constexpr (kSecond) {
            const float u = along[a], v = along[b];
            const bool swap = x < y;
            along[a] = swap ? v : u;
            along[b] = swap ? u : v;
        }
        key[a] = larger_key(x, y);
        key[b] = smaller_key(x, y);
    });
    if constexpr (kSecond) {  // (moved behind the next branch, the exchanges would keep every stage of the keys in registers)
        static_for<D1>(PENC_BODY(m) {
            PENC_INDEX(m);
            float x = along[m];
            asm volatile("" : "+v"(x));
            along[m] = x;
        });
    }
    fvec<D1> sorted;
    uvec<D1> step;
    static_for<D1>(PENC_BODY(m) {
        PENC_INDEX(m);
        const double k = key[m];
        const uint64_t bits = __builtin_bit_cast(uint64_t, k);
        sorted[m] = __builtin_bit_cast(float, static_cast<uint32_t>(bits >> 32));
        step[m] = static_cast<uint32_t>(bits);
    });
    if constexpr (!kOpenTies) {
        if (cap_mask == 0u || cap_mask >= (1u << kKeyStepBits)) {
            constexpr uint64_t kUpper = upper_step_bits<D>(std::make_integer_sequence<int, D1>{});
            static_for<D1>(PENC_BODY(m) {
                PENC_INDEX(m);
                const float r = sorted[m];
                const uint32_t order = (step[m] ^ static_cast<uint32_t>(__builtin_bit_cast(int, r) >> 31)) >> kKeyStepBits;
                step[m] = (step[m] & ~kOrderBits) | (static_cast<uint32_t>(kUpper >> (4u * order)) << kKeyStepBits);
            });
        }
    }

    CyclicSimplex<D> o;
    uvec<D1> h;
    h[0] = h0;
    static_for<D>(PENC_BODY(k) {
        PENC_INDEX(k); h[k + 1] = h[k] + step[D - k]; });
    if (cap_mask != 0u) {  // (to_slot, asked once)
        o.slot = h & cap_mask;
    } else {
        static_for<D1>(PENC_BODY(k) {
            PENC_INDEX(k); o.slot[k] = h[k] % capacity; });
    }
    o.turned = kExactInverse ? (sum & D) : (sum < 0 ? sum + D1 : sum);
    if constexpr (kFirst) {
        // A residual that is NaN (its point's coordinates are not finite, or overflow) is a key like any other where its bits are an ordinary double's upper word, as 0x7FC00000 is
        // (2.2e307): it ends up first or last, by its sign, and in the two weights beside that end.  With its upper payload bits set (0x7FF00000 and more) it is a NaN as a key
        // too, and vanishes from the network, which then holds another key twice.  So all weights get it from here, each from one of its two deltas.  (Five vector instructions of 240 a point and level at D = 3: training step 713 -> 713 us; 13 at D = 8, 686 -> 691, between cards.)
        float any_nan = rounded.resid[0];
        static_for<D>(PENC_BODY(c) {
            PENC_INDEX(c); any_nan += rounded.resid[c + 1]; });
        static_for<D1>(PENC_BODY(m) {
            PENC_INDEX(m);
            if constexpr ((D - m) % 2 == 0) sorted[m] = __builtin_fmaf(any_nan, 0.0f, sorted[m]); });
        fvec<D1> d, wrap;
        static_for<D1>(PENC_BODY(m) {
            PENC_INDEX(m);
            if constexpr (kExactInverse) {
                constexpr int kLog2 = __builtin_ctz(D1);
                wrap[m] = static_cast<float>((sum + m) >> kLog2);
                d[m] = sorted[m] + wrap[m];
            } else {
                wrap[m] = (sum > D - m ? 1.0f : 0.0f) - (sum < -m ? 1.0f : 0.0f);
                d[m] = __builtin_fmaf(wrap[m], static_cast<float>(D1), sorted[m]) * kInv;
            }
        });
        o.w[0] = d[D] + ((1.0f + wrap[0] - wrap[D]) - d[0]);
        static_for<D>(PENC_BODY(kk) {
            PENC_INDEX(kk);
            constexpr int k = kk + 1;
            o.w[k] = d[D - k] + ((wrap[D1 - k] - wrap[D - k]) - d[D1 - k]);
        });
    }
    if constexpr (kSecond) o.dB = sorted_elevated_grad_to_bary<D>(along);
    return o;
}

// A point's simplex as a scatter takes it.  With two dimensions by ranks, in the order of the remainder vertices: three residuals are ranked as fast as they are sorted,
// and a coarse level, whose few slots a vertex of one remainder meets in turn, is summed faster in that order, in columns and in the accumulate cache, whose
// lines the slots of one remainder claim without getting in each other's way.  (Forward and table gradient, 2^18 points, mean of 12 geometries, network -> ranks, us: 16 levels of 2^16 slots
// down to 1e-2 90.5 -> 88.0, 18 levels 95.6 -> 93.8, of 29429 slots, four features, a window on 0.4 of them, 88.8 -> 87.3;  2^18 slots 90.7 -> 90.1, along rays, 2^16, 101.1 -> 102.8;
// 2^22 slots, 2^19 points 503.0 -> 506.9.)
template <int D, bool kFirst, bool kSecond>
__device__ __forceinline__ CyclicSimplex<D> scatter_simplex(fvec<D> pos, fvec<D> q, const float* __restrict__ shift, const float* __restrict__ sf,
                                                            uint32_t capacity, uint32_t cap_mask) {
    if constexpr (D > 2) {
        return cyclic_simplex<D, kFirst, kSecond>(pos, q, shift, sf, capacity, cap_mask);
    } else {
        CyclicSimplex<D> o;
        const Located<D> s = locate<D>(pos, shift, sf);
        const uvec<D + 1> h = vertex_hashes<D>(s.rank, s.hash0);
        if (cap_mask != 0u) {  // (to_slot, asked once)
            o.slot = h & cap_mask;
        } else {
            static_for<D + 1>(PENC_BODY(k) {
                PENC_INDEX(k); o.slot[k] = h[k] % capacity; });
        }
        if constexpr (kFirst) o.w = barycentric<D>(s.rank, s.delta);
        if constexpr (kSecond) o.dB = pos_grad_grad_to_bary<D>(s.rank, q, sf);
        o.turned = 0;
        return o;
    }
}

// in[k] of a CyclicSimplex in the order of the remainder vertices.
template <int N, typename V>
__device__ __forceinline__ V turn_back(V in, int turned) {
    static_for<4>(PENC_BODY(bit) {
        PENC_INDEX(bit);
        constexpr int kBy = 1 << bit;
        if constexpr (kBy < N) {
            const bool by = (turned & kBy) != 0;
            const V from = in;
            static_for<N>(PENC_BODY(r) {
                PENC_INDEX(r);
                const auto stay = from[r], other = from[(r + kBy) % N];
                in[r] = by ? other : stay;
            });
        }
    });
    return in;
}

}  // namespace penc
