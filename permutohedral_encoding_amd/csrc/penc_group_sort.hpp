// The table gradient of small and ordinary batches, in two kernels whose time is not latency.
//
// The scatter of penc_scatter.hpp is made for batches that keep every workgroup busy for dozens of microseconds: it first finds out
// how its level behaves, caches, bins with room to spare, adds what does not fit straight into the gradient, which must
// therefore be cleared beforehand.  A batch of a few thousand points pays for all of that (2^15 points, 24 levels of 2^18 slots: clear
// 8 us, scatter 26, reduce 20).  Here
//   group_sort_kernel   a workgroup takes 512 points at one level, sorts their contributions by slot range in LDS and writes them
//                       out in one piece, together with where each range starts: nothing can overflow, every level goes
//                       the same way (lanes of a wave that share a slot are summed in registers first, which takes the edge off
//                       the coarse levels), and the search serves all pairs of features;
//   range_sum_kernel    a workgroup takes one slot range of one level, sums its stretches of all groups in LDS (fp64) and
//                       writes the WHOLE range: the gradient needs no clearing.
// Every level leaves (pos_dim + 1) records per point, also the coarse ones the scatter absorbs in LDS: in large batches
// their traffic costs more than the latencies saved (figures at group_sort_serves).
#pragma once

#include "penc_scatter.hpp"
#include "penc_table_backward.hpp"

namespace penc {

constexpr int kGroupPoints = 512;           // points, and threads, of a group_sort_kernel workgroup
constexpr int kGroupMaxRanges = 512;  // slot ranges of a level

}  // namespace penc
