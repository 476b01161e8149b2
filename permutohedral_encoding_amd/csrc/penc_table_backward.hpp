// The launch of the scattering kernel, one translation unit per input dimension (penc_table_backward.hip compiled
// with -DPENC_DIM=2 ... 8): the kernel has a dozen instances per dimension, and the units compile side by side.
#pragma once

#include "penc_scatter.hpp"

namespace penc {

struct TableLaunch {
    dim3 grid;
    hipStream_t stream;
    bool rows;          // the upstream gradient is read as rows
    bool second_order;  // double_pos_grad is given; with second_grad too, both orders
    bool many_bins;     // records go to more than kStageBins bins
    bool most_bins;     // more than kFewerOpenLinesMinBins (many_bins too, where there are records): workgroups of kScatterBlockManyBins threads, else of kScatterBlock
    bool wide_bins;     // (only together with most_bins: the scatter of wide bins has no other instance)
    int n_points, first_level;
    uint32_t n_pass_levels, feat_pairs, dies;
    int tiles_per_group;  // of kScatterBlock points; even
    uint32_t capacity, cap_mask;
    const float *positions, *scale_factor, *random_shift, *window, *grad;
    int64_t grad_row_stride;
    const float *double_pos_grad, *second_grad;
    float *table_grad, *grad_level_major;
    BinTarget bins;
    ClearTarget clear;
};

template <int D>
void launch_table_backward(const TableLaunch& t);

// Where group_sort_kernel leaves the records of a group of points (see penc_group_sort.hpp).
struct GroupSort {
    RecordValues* values;  // [level][pair][group][records]
    uint16_t* slots;       // [level][group][records]: the slot within its range
    uint16_t* starts;      // [level][group][n_ranges + 1]: where each range's records start
    uint32_t n_groups, n_ranges, range_shift;
    uint32_t records;      // room per group: its points times (D + 1)
};

template <int D>
void launch_group_sort(const TableLaunch& t, const GroupSort& sort, uint32_t n_levels);

}  // namespace penc
