// What the forward kernel families (int8, exact fp16 and scaled fp16 matrix operands) share: the launch arguments and the
// mapping from a workgroup to its (column tile, projection, row task).
#pragma once

#include "tgo_device.h"
#include "tgo_launch.h"

namespace tgo {

constexpr int FWD_TN = 128;          // weight rows per workgroup
constexpr int FWD_NT = FWD_TN / 32;  // 32-row weight tiles per workgroup

struct ForwardArgs {
    const uint8_t * packed;
    const uint8_t * packed_second;   // second projection of a pair, or nullptr
    int64_t bytes_per_expert;
    int64_t row_bytes;
    const int8_t * qx;               // int8 tiles, or fp16 tiles (Q8Workspace::layout)
    const float * dx;
    const float * sx;
    const float * power;             // scaled tiles only: 2^(e - E) per row and super-block
    const float * row_power;         // scaled tiles only: 2^E per row
    const uint16_t * block_sums;     // scaled tiles only: fp16 block sums, eight per row and super-block
    uint16_t * y;
    uint16_t * y_second;
    const int32_t * task_count;   // nullptr: dense
    const int32_t * task_early;   // tasks listed before those of few rows (TaskBuild::late_rows)
    int32_t * task_cursor;        // zero at launch; counts the short items that workgroups have taken
    const int32_t * task_expert;
    const int32_t * task_row_start;
    const int32_t * task_row_end;
    int rows;
    int rows_padded;
    int in_features;
    int out_features;
    int out_stride;   // values from one row of y to the next (out_features, or more)
    int n_tiles;
    int projections;   // 1, or 2 for a pair: both share the task's activations, so their tiles run side by side
    int swiglu;        // 1: a workgroup runs gate (-> y) then up and stores swiglu(gate, up) -> y_second
    int task_slots;
    int dense_row_tile;   // dense calls: rows per workgroup (forward_split)
    int wide;             // 2-byte aligned formats: the weights may be fetched as aligned 16-byte units (wide_stage_ok)
    float * partial;      // dense calls too small to fill the chip: fp32 sums of each range of K, [range][row][n_tiles * 128], or nullptr
    int k_splits;         // how many ranges (blockIdx.y picks one); 1 when partial is nullptr
    int early_only;       // grouped calls: 1 = this launch runs the tasks listed before the short ones, another kernel the rest
};

// The (column tile, projection, task) of this workgroup; false when the slot holds no task.
// `linear`: position in the launch order of workgroups (blockIdx.x for kernels that run one task per workgroup).
TGO_DEVICE bool forward_pick_linear(const ForwardArgs & a, int linear, int & n_tile, bool & second, int & expert,
                                    int & row_start, int & row_end) {
    int task;
    int tasks = a.task_count != nullptr ? a.task_count[0] : (a.rows + a.dense_row_tile - 1) / a.dense_row_tile;
    if (a.task_count != nullptr) {
        const int early = min(a.task_early[0], tasks);
        tasks = a.early_only != 0 ? early : tasks;
        xcd_chunk(linear, a.n_tiles * a.projections, tasks, early, n_tile, task);
    } else {
        xcd_tile(linear, a.n_tiles * a.projections, tasks, n_tile, task);
    }
    second = n_tile >= a.n_tiles;
    n_tile -= second ? a.n_tiles : 0;
    expert = 0;
    if (a.task_count != nullptr) {
        if (task >= tasks) {
            return false;
        }
        expert = a.task_expert[task];
        row_start = a.task_row_start[task];
        row_end = a.task_row_end[task];
    } else {
        row_start = task * a.dense_row_tile;
        if (row_start >= a.rows) {
            return false;
        }
        row_end = min(a.rows, row_start + a.dense_row_tile);
    }
    return true;
}

// Super-blocks [begin, end) of K that this workgroup multiplies.  RANGES: the kernel variants for k_splits > 1 (instantiations of
// their own: the branch at the end of the loop alone made the plain ones spill).
template <bool RANGES>
TGO_DEVICE void forward_k_range(const ForwardArgs & a, int & begin, int & end) {
    const int super_blocks = a.in_features / QK_K;
    begin = RANGES ? super_blocks * static_cast<int>(blockIdx.y) / a.k_splits : 0;
    end = RANGES ? super_blocks * (static_cast<int>(blockIdx.y) + 1) / a.k_splits : super_blocks;
}

// A range's sums of a 32 x 32 tile straight from the accumulators.  TRANSPOSED: the lane holds row l32 of the tile and, as
// elements 4 j .. 4 j + 3, columns 8 j + 4 half ..; otherwise column l32 and those rows.
template <bool TRANSPOSED, typename V16>
TGO_DEVICE void store_partial_32x32(const ForwardArgs & a, const V16 & acc, int row0, int row_end, int n0, int lane) {
    const int l32 = lane & 31, half = lane >> 5;
    const int pitch = a.n_tiles * FWD_TN;
    float * const out = a.partial + (static_cast<int64_t>(blockIdx.y) * a.rows + row0) * pitch + n0;
    if constexpr (TRANSPOSED) {
        if (row0 + l32 < row_end) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                *reinterpret_cast<float4 *>(out + static_cast<int64_t>(l32) * pitch + 8 * j + 4 * half) =
                    make_float4(acc[4 * j], acc[4 * j + 1], acc[4 * j + 2], acc[4 * j + 3]);
            }
        }
    } else {
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int row = 8 * (v / 4) + 4 * half + v % 4;
            if (row0 + row < row_end) {
                out[static_cast<int64_t>(row) * pitch + l32] = acc[v];
            }
        }
    }
}

TGO_DEVICE bool forward_pick(const ForwardArgs & a, int & n_tile, bool & second, int & expert, int & row_start,
                             int & row_end) {
    return forward_pick_linear(a, blockIdx.x, n_tile, second, expert, row_start, row_end);
}

// Launch of the fp16-operand kernels for arguments prepared by the common launcher (tgo_forward.hip).
hipError_t launch_forward_half(const ForwardArgs & args, int quant_type, hipStream_t stream);
hipError_t launch_forward_scaled(const ForwardArgs & args, int quant_type, hipStream_t stream);

}  // namespace tgo
