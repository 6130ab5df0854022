// Host-side launchers behind the C ABI.  Each returns the hipError_t of its launch.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <algorithm>

namespace tgo {

// Matrix operands of the MFMA forward kernels, a process-wide setting (tgo_set_forward_operand):
//   OPERAND_INT8    int8 quants on the int8 matrix instruction; every 32-value block result is scaled with two or
//                   three fp32 vector operations (tgo_forward.hip), which bound those kernels.
//   OPERAND_HALF    fp16 numbers holding the same integers exactly; one vector operation per result and block is
//                   left (tgo_forward_half.hip).
//   OPERAND_SCALED  both operands carry their scales: the dequantized q8_1 activation d * q and the dequantized
//                   weight, each normalised by a power of two per row and rounded to fp16 once.  The matrix
//                   instruction then accumulates the whole reduction and no vector instruction touches a result
//                   before the epilogue (tgo_forward_scaled.hip): the only kind whose bound is the matrix pipe.
//   OPERAND_AUTO    (default) scaled operands for calls with enough tasks to fill the chip with its 256-row x
//                   128-column tiles, otherwise exact fp16 for IQ2_S and int8 for the other formats (their smaller
//                   tiles spread a small call over more CUs).
// `quant_type` 0 stands for a workspace that is quantized without knowing the format it will be used with
// (tgo_quantize_q8_1, tgo_mmq_forward_prepared): int8 unless exact fp16 is forced.  The activation workspace is
// written for one kind of operand and records which (Q8Workspace::tag); it must be consumed as that kind.  An entry
// point reads the setting once and hands it to the rules below, so a change by another thread never splits a call.
enum ForwardOperand : int { OPERAND_INT8 = 0, OPERAND_HALF = 1, OPERAND_AUTO = 2, OPERAND_SCALED = 3 };
int forward_operand_setting();
void set_forward_operand_setting(int operand);
// Formats of the scaled-operand kernel (all five).
static constexpr bool scaled_forward_format(int quant_type) {
    return quant_type == 11 || quant_type == 12 || quant_type == 13 || quant_type == 14 || quant_type == 22;
}
// Fewest (256-row x 128-column) tiles for which OPERAND_AUTO picks the scaled kernel: one workgroup per CU runs them,
// so half a chip's worth is where it starts to beat the kernels with smaller tiles (dense 512 x 4096: 64 tiles, a
// tie; 4096 x 2048: 256 tiles, 12 % faster).
constexpr int64_t SCALED_AUTO_MIN_TILES = 128;
// The operand kind a call of this format and size uses under `setting` (never OPERAND_AUTO).  Grouped
// calls pass their total rows: the tiles of a ragged list are at least that many.
static inline int forward_operand_kind(int setting, int quant_type, int64_t rows = 0, int64_t out_features = 0, int projections = 1) {
    const int exact = quant_type == 22 ? OPERAND_HALF : OPERAND_INT8;
    if (setting == OPERAND_SCALED) {
        return scaled_forward_format(quant_type) ? OPERAND_SCALED : exact;
    }
    if (setting == OPERAND_AUTO) {
        const int64_t tiles = ((rows + 255) / 256) * ((out_features + 127) / 128) * projections;
        return scaled_forward_format(quant_type) && tiles >= SCALED_AUTO_MIN_TILES ? OPERAND_SCALED : exact;
    }
    return setting;
}
// Waves per workgroup of the fp16-operand kernels, 32 activation rows each (8: the pipelined variant, measured 5 to
// 11 % faster than the 4-wave one for the formats with 16-value scale groups, and no faster for the others).
static constexpr int half_forward_waves(int quant_type) { return quant_type == 14 || quant_type == 22 ? 8 : 4; }
// Row tile of one forward task; the task list is built for these.  int8 operands: 256 rows for the formats whose
// weights unpack into two int8 planes (Q6_K = 14, IQ2_S = 22), 128 rows for the single-plane ones; exact fp16
// operands: 32 rows per wave of the format's workgroup; scaled operands: 256 (eight multiplying waves of 32 rows).
static constexpr int forward_row_tile(int quant_type, int operand_kind) {
    return operand_kind == OPERAND_SCALED ? 256
           : operand_kind == OPERAND_HALF ? 32 * half_forward_waves(quant_type)
                                          : (quant_type == 14 || quant_type == 22 ? 256 : 128);
}
// Grouped calls with scaled operands: whole groups of at most FORWARD_LATE_ROWS rows are listed behind the other tasks and run by
// groups of four waves that all unpack and multiply (tgo_forward_groups.h), where the role-split workgroups with their 256-row tasks
// wait for four unpacking waves; groups of at most FORWARD_LAST_ROWS rows are listed last.  Uniform groups, 256 experts of 2048 x 512,
// gate and up with quantizing, us role-split -> this: Q4_K 16 rows 136 -> 123, 32 rows 151 -> 135, 64 rows 250 -> 184, 128 rows
// 308 -> 286; IQ2_S 64 rows 260 -> 186, 128 rows 318 -> 288; Q6_K 64 rows 339 -> 246, 128 rows 396 -> 324.  192 rows cut in two:
// a loss (Q4_K 396 -> 405).
// Fewer groups of 33 to 128 rows than larger tasks, and the former stay with the role-split workgroups: they are then too few to
// fill the chip, and four waves alone on a CU take longer over a task than twelve (128 experts of 2048 x 768 Q4_K, 700 tokens with
// power-law 1.1 routing: layer 222 us, 241 with them apart).
constexpr int FORWARD_LATE_ROWS = 128;
constexpr int FORWARD_LAST_ROWS = 32;
constexpr int BACKWARD_ROW_TILE = 256;
// Grad-input tasks of at most this many rows (a group's remainder) are listed behind the others and run by a
// kernel variant whose waves split the K columns of the tile instead of its rows.
constexpr int BACKWARD_SHORT_ROWS = 64;
// Decode regime: tasks of at most this many rows go to the bandwidth-oriented GEMV kernel.
constexpr int GEMV_ROW_TILE = 8;
// Dense calls of up to this many rows take it too, GEMV_ROW_TILE rows at a time: the MFMA kernel's 128-row
// column tiles leave most of the chip idle on a matrix of a few thousand rows, and its latency per tile is long.
constexpr int GEMV_DENSE_ROWS = 32;

// Dense forward calls: rows per workgroup, and, with exact operands, the ranges that K is cut into (each workgroup then leaves
// fp32 sums that a second kernel adds up in a fixed order; needs forward_partial_bytes() of scratch).
// A workgroup takes 2 to 6 us per super-block of K however few rows it has, so a call of a few tiles is as slow as its K is
// long: one row tile of 1024 x 4096 Q6_K 102 us on 8 CUs.  The ranges were chosen from a sweep of tiles x ranges over 1024 x 4096,
// 4096 x 2048, 5003 x 4096 and 4096 x 8192, 64 to 1024 rows:
//  - 128-row tiles (two workgroups per CU): 32-row tiles while those are at most 256, up to 640 workgroups, ranges of four
//    super-blocks, of two where even that leaves CUs idle; short K (fewer than 16) only below 128 tiles.
//    4096 x 8192 Q5_K, 64 rows: 71 -> 37 us, 517 rows 142 -> 99; 1024 x 4096 Q3_K, 64 rows: 50 -> 21.
//  - 256-row int8 tiles (one workgroup per CU; weights of two planes, the longest to unpack): up to 256 workgroups, ranges of two
//    super-blocks.  1024 x 4096 Q6_K, 64 rows: 102 -> 33 us; 5003 x 4096, 517 rows: 124 -> 98.
//  - 256-row fp16 tiles: the narrow variant up to 128 tiles, else the largest tile that yields 128 workgroups; ranges of four
//    super-blocks (a narrow workgroup's start costs as much as one).  4096 x 8192 IQ2_S, 64 rows: 77 -> 44 us.
// Matrices of fewer than four million weights keep one range.  That line is not one of speed: it leaves the sums of small
// dense calls those of the grouped calls on the same rows bit for bit, which the operators' tests hold them to (grouped calls on the
// matrix-core kernels, that is: those of few rows per group that grouped_takes_tiles takes add in another order).  With this rule's
// ranges below it, one range -> ranges: K = 4096, 512 columns, 64 rows Q6_K 102 -> 28 us, Q3_K 50 -> 19, Q4_K 37 -> 17, IQ2_S
// 42 -> 20; K = 2048, 1024 columns, 64 rows 55 -> 24, 29 -> 18, 22 -> 15, 25 -> 20; K = 1024 mostly a tie, from 2048 columns up
// also a loss (Q4_K, 517 rows of 2048: 18 -> 23).  (1024 x 4096, on the line, 64 rows: Q6_K 33, Q3_K 20, Q4_K 18.)
constexpr int SCALED_WORKGROUPS = 256;   // one per CU
struct ForwardSplit {
    int row_tile;
    int k_splits;
};
static inline ForwardSplit forward_split(int64_t rows, int64_t in_features, int64_t out_features, int quant_type, int operand_kind,
                                         bool scratch, int projections = 1) {
    const int64_t n_tiles = (out_features + 127) / 128;
    const int64_t super_blocks = in_features / 256;
    if (operand_kind == OPERAND_SCALED) {
        // One persistent workgroup per CU, items of 256 rows, unless those leave half of the chip without one: then 128 rows (8192 x 4096,
        // 300 rows: Q3_K 0.95 of the time, Q4_K 0.88, Q5_K 0.88, Q6_K 0.96, IQ2_S 0.96; 4096 x 4096, 900 rows: 1.01, 0.93, 0.96, 1.00, 1.00).
        // Fewer rows per item where they make the rounds of items come out even gain nothing that holds: the unpacking that the items repeat
        // costs as much (4096 x 4096, 192 rows per item: 2600 rows 0.97, 0.99, 1.00, 0.97, 0.97; 3000 rows 1.04, 1.06, 1.07, 1.05, 1.04; 11008 x
        // 2048, 600 rows, 224 per item: Q4_K 1.07).
        return {n_tiles * projections * ((rows + 255) / 256) <= SCALED_WORKGROUPS / 2 ? 128 : 256, 1};
    }
    const int full_tile = forward_row_tile(quant_type, operand_kind);
    const auto tiles = [&](int tile) { return n_tiles * ((rows + tile - 1) / tile); };
    if (scratch && out_features * in_features >= (INT64_C(1) << 22)) {
        int tile = full_tile;
        int64_t most;   // ranges
        if (full_tile == 128) {
            tile = tiles(32) <= 256 ? 32 : 128;
            const int64_t wanted = tiles(tile) * (super_blocks / 4) < 256 ? super_blocks / 2 : super_blocks / 4;
            most = tiles(tile) > 128 && super_blocks < 16 ? 1 : std::min(640 / tiles(tile), wanted);
        } else if (operand_kind == OPERAND_INT8) {
            most = std::min(256 / tiles(tile), super_blocks / 2);
        } else {
            most = super_blocks / 4;
            if (tiles(32) <= 128) {
                tile = 32;
            }
            while (tile > 64 && tiles(tile) * most < 128) {
                tile /= 2;
            }
            most = std::min(256 / tiles(tile), most);
        }
        if (most >= 2) {
            return {tile, most >= 8 ? 8 : most >= 4 ? 4 : 2};
        }
    }
    // One range.  Full tiles that would not even give every second CU a workgroup become smaller ones.
    // Single-plane formats: 32 rows, i.e. the kernel's narrow variant, whose four waves split the weight rows
    // (four times the workgroups, each about a third as long).  The two-plane formats have no narrow variant,
    // but their eight waves own 32 rows each: with tiles of 128, 64 or 32 rows only 4, 2 or 1 of them multiply
    // (the others still help to unpack), the vector work of a tile no longer queues two waves deep on every
    // SIMD, and there are 2, 4 or 8 times the workgroups; the largest tile that yields 128 workgroups is taken.
    int row_tile = full_tile;
    if (row_tile == 128) {
        if (tiles(128) <= 128) {
            row_tile = 32;
        }
    } else {
        while (row_tile > 32 && tiles(row_tile) < 128) {
            row_tile /= 2;
        }
    }
    return {row_tile, 1};
}
static inline int64_t forward_partial_bytes(int64_t rows, int64_t in_features, int64_t out_features, int quant_type, int operand_kind) {
    const int splits = forward_split(rows, in_features, out_features, quant_type, operand_kind, true).k_splits;
    return splits > 1 ? splits * rows * ((out_features + 127) / 128 * 128) * 4 : 0;
}

// Dense grad-input: a workgroup owns 256 rows x 128 columns of the result and walks the whole reduction (N weight
// rows, 64 per step) alone, so a call of a few hundred rows keeps K / 128 workgroups busy and takes as long as one
// of them needs for N / 64 dependent steps.  Such calls cut the reduction into this many ranges, one workgroup each,
// which leave fp32 partial results that a second kernel adds up in a fixed order.  1: no split.
// The line lies at half the CUs: 4096 x 2048 Q4_K, 1024 rows (64 items, four ranges) 62 -> 41 us, 2048 rows (128, two) 70 -> 61.
// Short reductions (fewer than 32 steps) gain from it up to an eighth of the CUs only: 1024 x 4096, 512 rows 24 -> 30 us.
constexpr int BACKWARD_WORKGROUPS = 256;   // one per CU
static inline int dense_grad_splits(int64_t rows, int64_t out_features, int64_t in_features) {
    const int64_t items = (rows + BACKWARD_ROW_TILE - 1) / BACKWARD_ROW_TILE * (in_features / 128);
    const int64_t steps = (out_features + 63) / 64;
    if (items > (steps < 32 ? 32 : 128)) {
        return 1;
    }
    int64_t splits = BACKWARD_WORKGROUPS / items;
    splits = splits < steps / 2 ? splits : steps / 2;   // at least two steps each
    splits = splits < 16 ? splits : 16;
    return splits < 2 ? 1 : static_cast<int>(splits);
}
// fp32 scratch of the split reduction for a dense call: the same decision as the launcher's
static inline int64_t dense_grad_partial_bytes(int64_t rows, int64_t out_features, int64_t in_features) {
    const int splits = dense_grad_splits(rows, out_features, in_features);
    return splits > 1 ? splits * rows * in_features * 4 : 0;
}

// Forward kernel family for a shape: dense calls with up to GEMV_DENSE_ROWS rows and grouped calls that
// average at most four rows per group are HBM-bound and take the GEMV kernel, everything else the MFMA one.
static inline bool use_gemv(int64_t rows, int64_t groups) {
    return groups <= 0 ? rows <= GEMV_DENSE_ROWS : rows <= 4 * groups;
}

// Whether the layout of the kernel for tasks of several rows (tgo_gemv_tiles.hip) allows a call: whole tiles of 16 weight rows (with
// them every expert is 16-byte aligned, as the entry points demand of the weights), offsets within a tile of 32 bits, and enough weights that
// are read: four million in grouped calls (fewer: their time is their launches and latencies, and most of them are one launch of the other
// kernel), a hundred thousand in dense ones (of the decode regime; dense_takes_tiles asks for four million).
static inline bool tiles_fit(int64_t rows, int64_t groups, int64_t in_features, int64_t out_features) {
    if (out_features % 16 != 0 || in_features > (INT64_C(1) << 22) || rows > (1 << 24)) {
        return false;
    }
    const int64_t matrices = groups <= 0 ? 1 : rows < groups ? rows : groups;
    return matrices * out_features * in_features >= (groups <= 0 ? INT64_C(1) << 17 : INT64_C(1) << 22);
}
// Decode-regime calls that take the kernel for tasks of several rows (tgo_gemv_tiles.hip), which unpacks every weight once
// per task, instead of those of tgo_gemv.hip, whose dot products cost the same again for every row.  It needs whole tiles of
// 16 weight rows and 16-byte aligned weights.  The lines lie where the two measured equal (2048 x 512 and 4096 x 1024 experts
// and their down projections, 1 to 124 tokens; dense 4096 x 2048 and 28672 x 8192, 1 to 32 rows):
//  - grouped: Q5_K always (1 token 17 -> 12 us), Q4_K too unless K is long enough for the other kernel's own matrix
//    instructions to pay; Q3_K and IQ2_S from 16 and 24 rows.  Q6_K, whose unpacking is the longest: from 16 rows if K is three or
//    four super-blocks, from half as many rows as groups below that (the other kernel folds rows there), from one and a half
//    times as many above.
//  - dense matrices that fill the chip: Q3_K always (28672 x 8192, one row: 54 -> 41 us), Q5_K, Q6_K and IQ2_S from three rows (80 ->
//    65 us for Q6_K), Q4_K from four.  Smaller ones: Q3_K and IQ2_S from five rows, Q6_K from nine, Q4_K and Q5_K beyond 16 (1024 x 2048: 5 rows
//    Q3_K 8.8 -> 7.9 us, 12 rows Q6_K 12.6 -> 11.0, 32 rows Q4_K 10.6 -> 8.8, IQ2_S 20.2 -> 9.8; 512 x 512, 32 rows: Q3_K 24.3 -> 7.3).
constexpr int GEMV_TILES_ROWS = 16;              // rows of its tasks
constexpr int64_t GEMV_TILES_WORKGROUPS = 384;   // workgroups that a launch should have for a wave to take four tiles of 16 weight rows instead of two
static inline bool gemv_takes_tiles(int64_t rows, int64_t groups, int64_t in_features, int64_t out_features, int quant_type) {
    if (!use_gemv(rows, groups) || !tiles_fit(rows, groups, in_features, out_features)) {
        return false;
    }
    const int64_t super_blocks = in_features / 256;
    if (groups <= 0) {
        const bool large = out_features * in_features >= (INT64_C(1) << 25);
        switch (quant_type) {
            case 11: return rows > (large ? 0 : 4);
            case 12: return rows > (large ? 3 : 16);
            case 13: return rows > (large ? 2 : 16);
            case 14: return rows > (large ? 2 : 8);
            default: return rows > (large ? 2 : 4);
        }
    }
    switch (quant_type) {
        case 11: return rows >= 16;
        case 12: return super_blocks <= 8;
        case 13: return true;
        case 14: return super_blocks <= 2 ? 2 * rows >= groups : super_blocks <= 4 ? rows >= 16 : 2 * rows >= 3 * groups;
        default: return rows >= 24;
    }
}
// Dense calls beyond the decode regime that take it all the same: three to eight tasks of 16 rows, each of which unpacks all weights,
// keep the chip busier than the matrix-core kernels' tiles of 128 columns, up to a number of rows that falls with the matrix; of the time
// of the matrix-core kernels (with their ranges of K), weights read from memory:
//  - up to 2^23 weights, 128 rows: 2048 x 2048 Q3_K 0.69, Q4_K 0.73, Q5_K 0.75, Q6_K 0.58, IQ2_S 0.64; 1024 x 8192 Q4_K 0.89, Q5_K 0.92.
//  - up to 2^24: 4096 x 4096, 96 rows Q3_K 0.88, Q4_K 0.94, Q5_K 0.98, Q6_K 1.03 (64 rows 0.79), IQ2_S 0.90; 8192 x 2048, 128 rows Q4_K 1.04.
//  - up to 2^26: 8192 x 4096, 64 rows 0.79, 0.89, 0.94, 0.90, 0.90 in this order, 80 rows 0.77, 0.91, 0.95, 1.15, 1.15.  From 48 million weights on
//    64 rows of a matrix without enough columns for the scaled kernel lose the last round of workgroups (14336 x 4096: 0.89, 1.06, 1.10, 0.98,
//    1.11; 48 rows 0.72, 0.86, 0.91, 0.78, 0.93); with enough of them they do not (16384 x 4096: 0.67, 0.76, 0.77, 0.85, 0.83).
//  - a long K is where ranges gain the most: Q4_K and Q5_K, whose other kernel unpacks the fastest, and beyond 12288 IQ2_S.  8192 x 5120,
//    48 / 64 rows Q4_K 0.96 / 0.95, Q5_K 1.02 / 1.02; 8192 x 8192 Q4_K 1.05 / 1.05, Q5_K 1.09 / 1.09; 4096 x 11008 1.05 / 1.07, 1.09 / 1.11; 1024 x 16384, 64
//    rows 1.09, 1.12, IQ2_S 1.10 (Q3_K 0.90, Q6_K 0.74).
static inline bool dense_takes_tiles(int setting, int64_t rows, int64_t in_features, int64_t out_features, int quant_type) {
    if (use_gemv(rows, 0)) {
        return gemv_takes_tiles(rows, 0, in_features, out_features, quant_type);
    }
    if (setting != OPERAND_AUTO || !tiles_fit(rows, 0, in_features, out_features)) {
        return false;
    }
    const int64_t weights = out_features * in_features;
    const bool quick = quant_type == 12 || quant_type == 13;   // (to unpack, for the other kernels)
    if (in_features > (quick ? 8192 : quant_type == 22 ? 12288 : 1 << 22)) {
        return false;
    }
    if (weights < (INT64_C(1) << 22)) {
        return false;
    }
    if (weights <= (INT64_C(1) << 23)) {
        return rows <= 128;
    }
    if (weights <= (INT64_C(1) << 24)) {
        return rows <= (quant_type == 14 || (quick && in_features > 4096) ? 64 : 96);
    }
    if (weights > (INT64_C(1) << 26) || (quick && in_features > 4096 && weights > (INT64_C(44) << 20))) {
        return false;
    }
    const bool last_round = weights > (INT64_C(48) << 20) && out_features < 16384 && (quick || quant_type == 22);
    return rows <= (last_round || (quant_type == 13 && in_features > 4096) ? 48 : 64);
}

// Grouped calls beyond the decode regime (use_gemv) that take it all the same: its tasks of 16 rows unpack a group's weights once or
// twice, the matrix-core kernels once per 128 or 256 rows and with a fraction of the chip.  The line is a number of rows per group on
// average, by the operand kind that the call has otherwise; the host does not see the sizes of the groups, and the more of the rows are in few
// groups, the more tasks unpack the same weights while the other kernels need fewer.  So the lines lie where a routing with a power law of
// 1.1 over the experts (normal logits on top of it) still gains or ties; of the time of the matrix-core kernels, gate and up of 2048 x 512
// unless said otherwise, mean of three routings with power 0.3 / 1.1 / 1.5:
//  - exact kinds, 256 experts: Q3_K 14 rows 0.59 / 0.96 / 1.06; Q4_K 8 rows 0.72 / 0.92 / 1.05, 10 rows 0.75 / 0.97 / 1.20, 12 rows 0.76 / 1.03 / 1.19;
//    Q5_K 8 rows 0.78 / 0.94 / 1.12, 10 rows 0.78 / 1.07 / 1.09; Q6_K 14 rows 0.41 / 0.70 / 0.99; IQ2_S 10 rows 0.58 / 0.94 / 1.08, 12 rows 0.63 / 1.03 /
//    1.24.  128 experts of 2048 x 768, 16 rows: Q4_K 0.78 / 0.94 / 1.05, Q5_K 0.82 / 0.96 / 1.12.  64 experts, equal groups of 16 rows: Q4_K
//    0.97, Q5_K 0.99.  Q4_K and Q5_K, whose other kernels unpack the fastest, lose to skew by rows in all rather than per group.
//  - scaled operands: 512 columns of K to 2048, 256 experts: Q3_K 12 rows 0.73 / 0.94 / 1.06, Q4_K 10 rows 0.73 / 0.89 / 1.00, Q5_K the same
//    0.73 / 0.83 / 1.02.  Larger experts lose earlier (1024 columns of K to 4096, 256 experts, power 1.1: 6 rows Q4_K 0.98, Q5_K 1.01, 8 rows 1.09 and 1.14; 128
//    experts, 12 rows: 0.94 and 0.97).  Q6_K (0.94 to 1.41 at 8 rows) and IQ2_S (0.99 to 1.53) not at all.
// All rows in one group of 256 is the worst of it: 8 rows on average, Q4_K 1.25 (46 us -> 58), 512 columns of K to 2048 1.73 (24 -> 42), and up to
// twice the time at the lines.
// Not where the operand kind was forced: the caller asked for that kind's kernels.
constexpr int64_t GEMV_TILES_SCALED_WORK = INT64_C(6) << 30;   // rows x columns x K: 1536 rows of 1024 x 4096
static inline bool grouped_takes_tiles(int setting, int64_t rows, int64_t groups, int64_t in_features, int64_t out_features,
                                       int quant_type, int projections) {
    if (use_gemv(rows, groups)) {
        return gemv_takes_tiles(rows, groups, in_features, out_features, quant_type);
    }
    if (setting != OPERAND_AUTO || !tiles_fit(rows, groups, in_features, out_features)) {
        return false;
    }
    const bool scaled = forward_operand_kind(setting, quant_type, rows, out_features, projections) == OPERAND_SCALED;
    switch (quant_type) {
        case 11: return rows <= (scaled ? 12 : 16) * groups && (!scaled || rows <= GEMV_TILES_SCALED_WORK / (out_features * in_features));
        case 12:
        case 13:
            return scaled ? rows <= 10 * groups && rows <= GEMV_TILES_SCALED_WORK / (out_features * in_features)
                          : rows <= 16 * groups && rows <= (quant_type == 12 ? 2560 : 2048);
        case 14: return !scaled && rows <= 32 * groups;
        default: return !scaled && rows <= 12 * groups;
    }
}

// q8_1 workspace: quantized values, then fp32 scales, then fp32 sums, in one of four layouts over the same bytes.
// The MFMA kernels want 32-row tiles in fragment order: int8, fp16 numbers holding the same integers, or (scaled)
// the dequantized values d * q * 2^-e as fp16 with e chosen per row and super-block; the GEMV family reads a few
// rows along K, for which that order would scatter every 16 bytes into a cache line of their own, so calls that
// take the GEMV family (use_gemv) quantize into plain int8 rows instead.
enum WorkspaceLayout : int { LAYOUT_INT8_TILES = 0, LAYOUT_HALF_TILES = 1, LAYOUT_ROWS = 2, LAYOUT_SCALED_TILES = 3 };
constexpr uint32_t WORKSPACE_TAG_MAGIC = 0x71380000u;   // | layout: first word of the workspace's 1 KiB tail

struct Q8Workspace {
    int8_t * q;     // int8 tiles: [rows_padded/32][K/32][2 halves][32 rows][16 bytes]   rows: [rows][K]
                    // half and scaled tiles: [rows_padded/32][K/32][2 k-halves][2 eighths x 32 rows][8 fp16]
    float * d;      // tiles: [K/32][rows_padded]                                         rows: [rows][K/32]
    float * sum;    // same as d
    float * power;  // scaled tiles: 2^(e - E) per row and super-block, [K/256][rows_padded] (2^e until the second pass)
    uint16_t * block_sums;   // scaled tiles: fp16(sum * 2^-e) per block, [rows_padded/32][K/256][32 rows][8 blocks]
    float * row_power;       // scaled tiles: 2^E per row, [rows_padded]
    uint32_t * tag;          // WORKSPACE_TAG_MAGIC | layout, written by the quantizer
    int64_t rows_padded;
    int layout;
    bool by_rows() const { return layout == LAYOUT_ROWS; }
    bool half_tiles() const { return layout == LAYOUT_HALF_TILES; }
    bool scaled_tiles() const { return layout == LAYOUT_SCALED_TILES; }
    int operand_kind() const {
        return layout == LAYOUT_SCALED_TILES ? OPERAND_SCALED : layout == LAYOUT_HALF_TILES ? OPERAND_HALF : OPERAND_INT8;
    }
};

static inline int64_t pad_rows(int64_t rows) { return (rows + 31) / 32 * 32; }

// (sized for the scaled fp16 tiles whichever layout a call ends up using)
static inline int64_t q8_workspace_bytes(int64_t rows, int64_t in_features) {
    const int64_t padded = pad_rows(rows);
    // the 1 KiB tail lets kernels fetch the scales of a whole 32-row tile with 16-byte loads even when the
    // tile starts at the last row; its first word is the layout tag
    return 2 * padded * in_features + 2 * padded * (in_features / 32) * static_cast<int64_t>(sizeof(float)) +
           padded * (in_features / 256) * (static_cast<int64_t>(sizeof(float)) + 16) +
           padded * static_cast<int64_t>(sizeof(float)) + 1024;
}

// `operand_kind`: OPERAND_INT8, OPERAND_HALF or OPERAND_SCALED (forward_operand_kind); ignored for by_rows.
static inline Q8Workspace q8_workspace_view(void * base, int64_t rows, int64_t in_features, bool by_rows, int operand_kind) {
    Q8Workspace view;
    view.layout = by_rows ? LAYOUT_ROWS
                  : operand_kind == OPERAND_SCALED ? LAYOUT_SCALED_TILES
                  : operand_kind == OPERAND_HALF ? LAYOUT_HALF_TILES : LAYOUT_INT8_TILES;
    view.rows_padded = pad_rows(rows);
    view.q = static_cast<int8_t *>(base);
    view.d = reinterpret_cast<float *>(view.q + 2 * view.rows_padded * in_features);
    view.sum = view.d + view.rows_padded * (in_features / 32);
    view.power = view.sum + view.rows_padded * (in_features / 32);
    view.block_sums = reinterpret_cast<uint16_t *>(view.power + view.rows_padded * (in_features / 256));
    view.row_power = reinterpret_cast<float *>(reinterpret_cast<uint8_t *>(view.block_sums) + view.rows_padded * (in_features / 256) * 16);
    view.tag = reinterpret_cast<uint32_t *>(view.row_power + view.rows_padded);
    return view;
}

// Tile tasks of the grouped operators: [count][early][expert x max][row_start x max][row_end x max][cursors].
// `early` is the number of tasks listed before the short ones (TaskBuild::late_rows); count when nothing is short.
// `cursor`: TASK_CURSORS counters, TASK_CURSOR_STRIDE words apart (a cache line each), zero when the list is built: a
// kernel whose workgroups take items of the list in turn counts them there.
constexpr int TASK_CURSORS = 8;
constexpr int TASK_CURSOR_STRIDE = 32;
struct TaskList {
    int32_t * count;
    int32_t * early;
    int32_t * expert;
    int32_t * row_start;
    int32_t * row_end;
    int32_t * cursor;
    int max_tasks;
};

static inline int max_tasks_for(int64_t rows, int64_t groups, int row_tile) {
    return static_cast<int>((rows + row_tile - 1) / row_tile + groups);
}

static inline int64_t task_workspace_bytes(int64_t rows, int64_t groups) {
    // sized for the smallest tile any kernel uses so one buffer fits every path
    return (2 + 3 * static_cast<int64_t>(max_tasks_for(rows, groups, GEMV_ROW_TILE)) + TASK_CURSOR_STRIDE * (TASK_CURSORS + 1)) *
           static_cast<int64_t>(sizeof(int32_t));
}

static inline TaskList task_list_view(void * base, int64_t rows, int64_t groups, int row_tile) {
    TaskList list;
    list.max_tasks = max_tasks_for(rows, groups, row_tile);
    list.count = static_cast<int32_t *>(base);
    list.early = list.count + 1;
    list.expert = list.count + 2;
    list.row_start = list.expert + list.max_tasks;
    list.row_end = list.row_start + list.max_tasks;
    // (the cursors start on a cache line of their own)
    int32_t * const end = list.row_end + list.max_tasks;
    list.cursor = end + (TASK_CURSOR_STRIDE - (end - list.count) % TASK_CURSOR_STRIDE) % TASK_CURSOR_STRIDE;
    return list;
}

// What a kernel needs to build the tile-task list of a grouped call on the side (one of its workgroups does it
// before its own share of the work), so that the list costs neither a launch nor a place in the stream's
// critical path.  tasks.count == nullptr: nothing to build.
struct TaskBuild {
    const int64_t * expert_indices;
    const int32_t * expert_offsets;
    TaskList tasks;
    int num_experts, num_groups, rows, row_tile;
    int late_rows;  // tasks of at most this many rows are listed after all the others; 0: group order throughout
    int last_rows;  // > 0: of these, those of at most this many rows last, the others apart only if they are as many as the ordinary
                    // tasks
    int late_whole_groups;   // 1: only groups of at most late_rows rows are listed late, not the remainders of larger ones
};

static inline TaskBuild no_task_build() {
    TaskBuild build = {};
    build.tasks.count = nullptr;
    return build;
}

// Optional event bracket around a kernel launch (see tgo_profile_enable in the C ABI).
struct ProfileScope {
    ProfileScope(int kernel, hipStream_t stream);
    ~ProfileScope();
    int kernel;
    hipStream_t stream;
    hipEvent_t start;
    bool active;
};

hipError_t launch_dequant_bf16(const uint8_t * packed, uint16_t * out, int64_t rows, int64_t in_features,
                               int quant_type, hipStream_t stream);
// With `gather` set, workspace row r is quantized from input row gather[r] (rows outside [0, input_rows)
// quantize as zeros), i.e. the token -> expert-sorted-row gather of a MoE layer is folded into the read.
// With `build` set, one workgroup of the launch also writes the tile-task list.
hipError_t launch_quantize_q8_1(const uint16_t * input, const Q8Workspace & ws, int64_t rows,
                                int64_t in_features, hipStream_t stream, const int64_t * gather = nullptr,
                                int64_t input_rows = 0, const TaskBuild * build = nullptr);
// up_then_activated[i] = swiglu(gate[i], up_then_activated[i]) over `count` bf16 values (timed with the forward kernels).
hipError_t launch_swiglu_rows(const uint16_t * gate, const uint16_t * up, uint16_t * activated, int64_t count,
                              hipStream_t stream);   // (`activated` may be `up`)
// The (token, choice) slots sorted by expert: one launch up to ROUTE_SINGLE_SLOTS slots, above that two, with room for
// route_blocks(slots) * num_experts counts in `counts` (nullptr otherwise).
constexpr int64_t ROUTE_SINGLE_SLOTS = 4096;
constexpr int ROUTE_MAX_BLOCKS = 64;
constexpr int ROUTE_EXPERT_LIMIT = 4096;
constexpr int64_t ROUTE_SLOT_LIMIT = int64_t{1} << 22;   // (a wave counts its slots of one expert in 16 bits)
int route_blocks(int64_t slots);
hipError_t launch_route(const int64_t * slot_experts, int64_t slots, int top_k, int num_experts, int32_t * counts,
                        int64_t * row_index, int64_t * slot_rows, int64_t * expert_indices, int32_t * expert_offsets,
                        hipStream_t stream);
// row_token[r], row_weight[r]: token and weight of the slot that names row r (-1 and 0 when none does).
hipError_t launch_invert_slots(const int64_t * slot_rows, const float * slot_weights, int64_t slots, int top_k,
                               int64_t num_rows, int64_t * row_token, float * row_weight, hipStream_t stream);
// grad_weights[slot] = dot(rows[slot_rows[slot], :], grad_tokens[slot / top_k, :]); `features` is a multiple of 8.
hipError_t launch_slot_weight_grad(const uint16_t * rows, const uint16_t * grad_tokens, const int64_t * slot_rows,
                                   float * grad_weights, int64_t slots, int top_k, int64_t num_rows, int features,
                                   hipStream_t stream);
// Zeros in the rows that lie in no valid group.
hipError_t launch_clear_uncovered(uint16_t * rows, int64_t num_rows, int features, const int64_t * expert_indices,
                                  const int32_t * expert_offsets, int num_groups, int num_experts, hipStream_t stream);
// out[t, :] = sum of rows[order[i], :] over i in [starts[t], starts[t + 1]), in list order (fp32, one rounding).
hipError_t launch_rows_to_tokens(const uint16_t * rows, const int64_t * order, const int64_t * starts, uint16_t * out,
                                 int tokens, int64_t num_rows, int features, hipStream_t stream);
// d_gate, d_up of silu(gate) * up for the cotangent `grad_activated` (and `grad_gate`, a cotangent of the gate output
// itself, or nullptr), elementwise over `count` bf16 values.
hipError_t launch_swiglu_backward_rows(const uint16_t * gate, const uint16_t * up, const uint16_t * grad_activated,
                                       const uint16_t * grad_gate, uint16_t * d_gate, uint16_t * d_up, int64_t count,
                                       hipStream_t stream);
// Turns `count` bf16 outputs into NaN when the workspace's tag is not the layout of `ws` (runs behind the multiply kernel).
hipError_t launch_workspace_guard(const Q8Workspace & ws, uint16_t * out, int64_t count, hipStream_t stream);
hipError_t launch_q8_unpack(const Q8Workspace & ws, int8_t * q, float * d, float * sum, int64_t rows,
                            int64_t in_features, hipStream_t stream);

// out[t, :] = sum_j slot_weights[t, j] * rows[slot_rows[t, j], :] (bf16 rows, fp32 accumulation in choice order,
// one rounding); a slot whose row is outside [0, num_rows) contributes nothing.  `features` is a multiple of 8;
// `slot_weights` may be null: weights of one.
hipError_t launch_moe_combine(const uint16_t * rows, const int64_t * slot_rows, const float * slot_weights,
                              uint16_t * out, int tokens, int top_k, int64_t num_rows, int features,
                              hipStream_t stream);
// Dense when tasks == nullptr (row tiles follow from `rows`), grouped otherwise.  With `packed_second` and
// `output_second` set, one launch computes both projections of a pair from the same activation workspace.
// `output_stride`: values from one output row to the next, 0 for out_features.
hipError_t launch_mmq_forward(const uint8_t * packed, const uint8_t * packed_second, int64_t bytes_per_expert,
                              const Q8Workspace & ws, uint16_t * output, uint16_t * output_second,
                              const TaskList * tasks, int rows, int in_features, int out_features,
                              int quant_type, hipStream_t stream, int output_stride = 0, float * partial = nullptr);
// Pair only: `output` receives the first projection (gate) and `output_second` silu(gate) * second projection,
// both factors rounded to bf16 first, the product rounded once.
hipError_t launch_mmq_forward_swiglu(const uint8_t * packed, const uint8_t * packed_second, int64_t bytes_per_expert,
                                     const Q8Workspace & ws, uint16_t * output, uint16_t * output_second,
                                     const TaskList * tasks, int rows, int in_features, int out_features,
                                     int quant_type, hipStream_t stream);
hipError_t launch_mmq_gemv(const uint8_t * packed, const uint8_t * packed_second, int64_t bytes_per_expert,
                           const Q8Workspace & ws, uint16_t * output, uint16_t * output_second,
                           const TaskList * tasks, int rows, int in_features, int out_features,
                           int quant_type, hipStream_t stream, int output_stride = 0);
// `ws`: plain rows, or for a dense call without SwiGLU the exact tile layouts as well.
hipError_t launch_mmq_gemv_tiles(const uint8_t * packed, const uint8_t * packed_second, int64_t bytes_per_expert,
                                 const Q8Workspace & ws, uint16_t * output, uint16_t * output_second,
                                 const TaskList * tasks, int rows, int in_features, int out_features,
                                 int quant_type, bool swiglu, hipStream_t stream, int output_stride = 0);
// The same from bf16 activations in one launch: every workgroup quantizes its task's rows itself and, for a grouped
// call (`expert_offsets` set), finds its task in the group list, so neither a quantizer launch nor a task list
// exists.  Formats whose decode-regime routines read their activations one 16-value unit per lane.
// `gather` (or nullptr): row r of the call is row gather[r] of `input`, which has `input_rows` rows.
// The quantization is repeated by every workgroup that shares a task's rows (one per 16 weight rows), which costs a
// workgroup about as much as its dot products once a task has eight rows; it pays while the call is bound by its
// launches and their latencies: dense calls of one task, grouped calls of at most 64 rows (measured on a 256-expert
// layer: 1 token x top-8 32 -> 20 us of kernel time, 8 tokens 52 -> 48 us, 256 rows with 200 in one group 68 -> 101 us).
// Every workgroup of a fused grouped call reads the whole group list to find its task, so a list far longer than any
// expert count in use (GEMV_FUSED_GROUPS) keeps the task list that one workgroup builds for all.
constexpr int GEMV_FUSED_GROUPED_ROWS = 64;
constexpr int GEMV_FUSED_GROUPS = 1024;
static inline bool gemv_fuses(int quant_type, int64_t rows, int64_t groups) {
    const bool format = quant_type == 11 || quant_type == 14 || quant_type == 22;   // Q3_K, Q6_K, IQ2_S
    return format && use_gemv(rows, groups) && groups <= GEMV_FUSED_GROUPS &&
           rows <= (groups <= 0 ? GEMV_ROW_TILE : GEMV_FUSED_GROUPED_ROWS);
}
hipError_t launch_mmq_gemv_fused(const uint8_t * packed, const uint8_t * packed_second, int64_t bytes_per_expert,
                                 const uint16_t * input, const int64_t * gather, int64_t input_rows,
                                 const int64_t * expert_indices, const int32_t * expert_offsets, int num_experts,
                                 int num_groups, uint16_t * output, uint16_t * output_second, int rows, int in_features,
                                 int out_features, int quant_type, hipStream_t stream);
// ---- cross-entropy of a chunk of logits (tgo_loss.hip) ----
constexpr int LOSS_SPAN = 8192;   // columns whose statistics one workgroup forms
static inline int loss_spans(int64_t columns) { return static_cast<int>((columns + LOSS_SPAN - 1) / LOSS_SPAN); }
// count[0] = max(1, targets that are not ignored); loss[0] = sum(row_loss) / count[0].
hipError_t launch_count_targets(const int64_t * targets, int64_t rows, int64_t ignore_index, float * count, hipStream_t stream);
hipError_t launch_loss_total(const float * row_loss, int64_t rows, const float * count, float * loss, hipStream_t stream);
// Loss of each row, and with `cotangent` set (softmax - one_hot) / count as launch_pack_cotangent would pack it.
// `logits`: bf16 rows `pitch` values apart (a multiple of 8, the buffer whole); `stats`: rows * loss_spans(columns).
hipError_t launch_cross_entropy(const uint16_t * logits, int64_t pitch, int rows, int columns, float2 * stats,
                                const int64_t * targets, int64_t ignore_index, const float * count, float * row_loss,
                                uint8_t * cotangent, hipStream_t stream);
// out[i] = bf16(in[i] * factor[0]); `count` is a multiple of 8.
hipError_t launch_scale_bf16(const uint16_t * in, const float * factor, uint16_t * out, int64_t count, hipStream_t stream);

// Cotangent in MFMA fragment order: [rows_padded/32][chunks] slabs of 1 KiB (32 rows x 16 columns), zero
// padded; the column count is rounded up to 64 so that kernels can walk it four chunks at a time.
static inline int cotangent_chunks(int64_t out_features) { return static_cast<int>((out_features + 63) / 64 * 4); }
static inline int64_t cotangent_workspace_bytes(int64_t rows, int64_t out_features) {
    return pad_rows(rows) / 32 * cotangent_chunks(out_features) * 1024;
}
// One launch packs one cotangent or both of a pair (`grad_second`/`packed_second` null or set together) and, with
// `build` set, writes the tile-task list on the side.  With `gather` set (single cotangent), packed row r is
// bf16(scale[r] * grad[gather[r], :]) with `grad` holding `gather_rows` rows; an index outside them gives zeros.
hipError_t launch_pack_cotangent(const uint16_t * grad, const uint16_t * grad_second, uint8_t * packed,
                                 uint8_t * packed_second, int rows, int out_features, hipStream_t stream,
                                 const TaskBuild * build = nullptr, const int64_t * gather = nullptr,
                                 const float * scale = nullptr, int64_t gather_rows = 0);
// `cotangent_*` are buffers written by launch_pack_cotangent.
// `partial` (dense calls): dense_grad_partial_bytes() of scratch for the split reduction, or nullptr.
hipError_t launch_mmq_grad_input(const uint8_t * cotangent_first, const uint8_t * cotangent_second,
                                 const uint8_t * packed_first, const uint8_t * packed_second,
                                 int64_t bytes_per_expert, uint16_t * grad_input, const TaskList * tasks,
                                 int rows, int out_features, int in_features, int quant_type,
                                 hipStream_t stream, float * partial = nullptr);

// ---- dense products whose weights are unpacked once per call (tgo_unpacked.hip) ----
// One projection: its packed weight, and its input (forward) or the cotangent of its output (grad-input).
struct DenseSource {
    const uint8_t * packed;
    const uint16_t * activations;
    int64_t out_features;
    int quant_type;
};
// How a product of slabs is cut into workgroups: `full_rows` rows in tiles of 256 x 256 that fill the chip a whole number of times
// (one workgroup per CU), the rest in tiles of `rest_tile_rows` x `rest_tile_columns`, and what that takes, in microseconds.
struct ProductPlan {
    int64_t full_rows;
    int rest_tile_rows, rest_tile_columns;
    float microseconds;
};
// `tiles` workgroups, 256 to a round: a round is the faster the emptier it is, down to `half` for half a round, below which the CUs at
// work no longer gain from those that are idle.
static inline float rounds_microseconds(int64_t tiles, float half, float whole) {
    const int64_t rounds = (tiles - 1) / 256;
    const float last = static_cast<float>(tiles - 256 * rounds);
    return static_cast<float>(rounds) * whole + (last <= 128.0f ? half : half + (whole - half) * (last - 128.0f) / 128.0f);
}
// Measured (100 to 8192 rows, 2048 to 28672 columns, reduction 512 to 11008), half a round and a whole one, per reduction step of 16 and for
// the stores: 256 x 256 tiles 0.29 us + 5 and 0.42 + 9, 128 x 256 0.18 + 3 and 0.255 + 5, 128 x 128 0.115 + 3 and 0.15 + 4, each of several
// rounds 0.125 + 2.5 (two workgroups share a CU).
static inline ProductPlan product_plan(int64_t rows, int64_t columns, int64_t steps) {
    const auto up = [](int64_t count, int64_t tile) { return (count + tile - 1) / tile; };
    const int64_t across = up(columns, 256);
    const float n = static_cast<float>(steps);
    const auto large = [&](int64_t tiles) { return rounds_microseconds(tiles, 0.29f * n + 5.0f, 0.42f * n + 9.0f); };
    const auto with_rounds = [&](int64_t rounds, int64_t row_tiles) {
        ProductPlan plan = {rounds * row_tiles * 256, 256, 256, static_cast<float>(rounds) * large(row_tiles * across)};
        const int64_t rest = rows - plan.full_rows;
        if (rest > 0) {
            const float a = large(up(rest, 256) * across);
            const float b = rounds_microseconds(up(rest, 128) * across, 0.18f * n + 3.0f, 0.255f * n + 5.0f);
            const int64_t small = up(rest, 128) * up(columns, 128);
            const float c = small <= 256 ? rounds_microseconds(small, 0.115f * n + 3.0f, 0.15f * n + 4.0f)
                                         : static_cast<float>(up(small, 256)) * (0.125f * n + 2.5f) + 3.0f;
            const float least = std::min(a, std::min(b, c));
            plan.rest_tile_rows = least == a ? 256 : 128;
            plan.rest_tile_columns = least == a || least == b ? 256 : 128;
            plan.microseconds += least + (rounds > 0 ? 4.0f : 0.0f);
        }
        return plan;
    };
    const ProductPlan plain = with_rounds(0, 1);
    const int64_t row_tiles = across <= 256 ? 256 / across : 0;
    if (row_tiles * across < 160 || rows < row_tiles * 256) {
        return plain;
    }
    const ProductPlan whole = with_rounds(rows / (row_tiles * 256), row_tiles);
    return whole.microseconds < plain.microseconds ? whole : plain;
}
// Writing both operands: two bytes per weight leave.
static inline float unpack_microseconds(int64_t out_features, int64_t in_features) {
    return 5.0f + static_cast<float>(out_features) * static_cast<float>(in_features) * 0.6e-6f;
}
constexpr int UNPACKED_SOURCES = 4;
// Workspace of a grad-input of `count` projections: slabs of 16 weight rows (`chunks` of all projections together), and those of the cotangents,
// unless all of them have rows of whole stages (32 values), which the product reads as they stand.
struct UnpackedGradWorkspace {
    bool row_major;
    int64_t chunks;
    uint8_t * cotangent;
    uint8_t * weights;
    int64_t bytes;
    // of one projection: row-major it ends with its weight rows, packed with a whole step of 64
    int64_t chunks_of(int64_t out_features) const { return row_major ? out_features / 16 : (out_features + 63) / 64 * 4; }
};
static inline UnpackedGradWorkspace unpacked_grad_workspace(void * base, int64_t rows, int count, const int64_t * out_features, int64_t in_features) {
    UnpackedGradWorkspace view;
    view.row_major = std::all_of(out_features, out_features + count, [](int64_t features) { return features % 32 == 0; });
    view.chunks = 0;
    for (int i = 0; i < count; ++i) {
        view.chunks += view.chunks_of(out_features[i]);
    }
    const int64_t cotangent_bytes = view.row_major ? 0 : pad_rows(rows) / 32 * view.chunks * 1024;
    view.cotangent = static_cast<uint8_t *>(base);
    view.weights = view.cotangent + cotangent_bytes;
    view.bytes = cotangent_bytes + in_features / 32 * view.chunks * 1024;
    return view;
}
// Whether a dense grad-input unpacks its weights once (tgo_unpacked.hip) or leaves it to every workgroup (tgo_backward.hip): by what
// either takes.  The latter packs the cotangent, then runs items of 256 x 128, a round of 256 taking 0.27 us per 16 weight rows and half a
// round 0.18, and cuts the reduction where that leaves half of the chip idle, for fp32 sums to be written and read again.  Projections of one
// input (`out_features`: their weight rows together) would take `calls` calls and an addition for each but the first.
// A product that reads 32 MB of cotangent waits for them at 0.165 us per step, however few tiles it has (rows x weight rows x K: 2048 x 8192 x
// 1536 93 us, 3193 x 15872 x 768 172, 4096 x 28672 x 512 302; the other kernels 85, 129 and 214).
// Of the time of the kernels that unpack as they multiply, where this rule leaves them, inputs from memory, all formats: 246 of 460 calls of 96 to
// 16384 rows, 256 to 28672 weight rows, K 512 to 8192: 0.83 on the mean, 1.17 at most (2 us of an IQ2_S call of 11); 31 of 68 pairs of one shape
// 0.87, 1.11; 46 of 62 calls of three projections 0.67, 1.00.
// 4096 x 2048, 4096 rows Q4_K 85.2 -> 76.2 us, Q6_K 87.4 -> 77.0; 8192 rows 164 -> 125, 168 -> 127.  On the other side of it, always unpacked:
// 28672 x 8192, 300 rows Q4_K 211 -> 439 us; 4096 x 2048, 300 rows 27.6 -> 44.8; and the wrong one: 257 rows of 1260 x 4608 IQ2_S 24.7 -> 27.3.
static inline bool grad_unpacks(int64_t rows, int64_t out_features, int64_t in_features, int calls = 1) {
    // (32-bit lane offsets; a workspace of at most 1 GiB for the weights)
    if (rows < 96 || out_features > (1 << 24) || out_features * in_features > (INT64_C(1) << 29) || rows > (1 << 24)) {
        return false;
    }
    const int64_t steps = (out_features + 15) / 16;
    const int splits = dense_grad_splits(rows, out_features, in_features);
    const int64_t items = (rows + BACKWARD_ROW_TILE - 1) / BACKWARD_ROW_TILE * (in_features / 128) * splits;
    const float together = 9.0f + static_cast<float>(rows) * static_cast<float>(out_features) * 0.8e-6f +
                           static_cast<float>(steps / splits) * rounds_microseconds(items, 0.18f, 0.27f) +
                           (splits > 1 ? 4.0f + static_cast<float>(rows) * static_cast<float>(in_features) * static_cast<float>(splits) * 1.2e-6f : 0.0f) +
                           static_cast<float>(calls - 1) * (9.0f + static_cast<float>(rows) * static_cast<float>(in_features) * 1.5e-6f);
    const float waiting = rows * out_features >= (1 << 24) ? 0.165f * static_cast<float>(steps) : 0.0f;
    return 1.05f * (unpack_microseconds(out_features, in_features) + std::max(product_plan(rows, in_features, steps).microseconds, waiting)) < together;
}
// Of several projections as one reduction: their sums in fp32.  (Below a million weights the terms keep being rounded one by one, for the bits' sake and
// not for speed.)  Two of one width are one call otherwise too (mmq_pair_grad_input, if their formats agree).  More than two count as a call each, also
// where two of them are such a pair, for what the calls cost on the host: 161 rows of 2188 + 547 + 547 x 1280 Q5_K, forward and backward from Python,
// 167 us, and 187 with the pair counted as one call.
static inline bool multi_grad_unpacks(int64_t rows, int count, const int64_t * out_features, int64_t in_features) {
    int64_t total = 0;
    for (int i = 0; i < count; ++i) {
        total += out_features[i];
    }
    const bool pair = count == 2 && out_features[0] == out_features[1];
    return (count == 1 || total * in_features >= (1 << 20)) && grad_unpacks(rows, total, in_features, pair ? 1 : count);
}
// Grad-input of up to four projections of one input: the sum of their Jacobian products, rounded once.  `workspace`:
// unpacked_grad_workspace().bytes.
hipError_t launch_grad_input_unpacked(const DenseSource * sources, int count, void * workspace, uint16_t * grad_input, int64_t rows,
                                      int64_t in_features, hipStream_t stream);

// Reduction steps of 16 of the forward: with Q4_K (12) and Q5_K (13) one more per super-block, for the minima, and an even number.
static inline int64_t unpacked_forward_steps(int quant_type, int64_t in_features) {
    const int64_t super_blocks = in_features / 256;
    return quant_type == 12 || quant_type == 13 ? (17 * super_blocks + 1) / 2 * 2 : 16 * super_blocks;
}
// Scratch: the slabs of `tiles` times 32 weight rows and their powers.  (The activations fit the q8_1 workspace: 2.125 bytes per value and
// 36 per row of the 2.3 and 4 that it holds.)
static inline int64_t unpacked_forward_bytes(int quant_type, int64_t tiles, int64_t in_features) {
    return tiles * (unpacked_forward_steps(quant_type, in_features) * 1024 + 128);
}
// Whether a dense forward call with scaled operands unpacks its weights once (tgo_unpacked.hip) or leaves it to the unpacking waves of
// every workgroup (tgo_forward_scaled.hip): by what either takes.  The latter quantizes in two launches (with their gaps 9 us for 256 rows, 16
// from 1024 on, 12 where tiles of 128 rows follow), then runs items of 256 x 128 on persistent workgroups, half a round and a whole round of 256 in 0.19 and 0.27 us per step of 16 (Q6_K 0.31) and 1.3 for the stores, or of 128
// x 128 (forward_split) in 0.145 and 0.185, the slower formats to unpack 0.22.
// Results of more than 100 million values no longer stay in the last cache, which only the kernel without an overlapped epilogue notices.
// Of the time of the scaled kernel, where this rule leaves it: 277 of 453 calls of 96 to 16384 rows, 512 to 28672 columns, K 512 to 8192 0.84 on the
// mean, 1.12 at most (4 us of 34); with 16 us for any number of rows 296, 0.85 and 1.46 (123 rows of 18688 x 512 Q3_K 18.2 -> 26.6).  Calls of three
// projections (57) 0.73, 1.01.  4096 x 4096, 4096 rows: Q4_K 173 -> 152 us, Q3_K 178 -> 144, Q6_K 196 -> 147; 2048 x 2048, 2000 rows Q4_K 43.7 -> 34.8.
// On the other side of it, always unpacked: 28672 x 8192, 300 rows Q4_K 235 -> 389 us; 16384 x 1024, 8192 rows Q4_K 315 -> 367.
static inline bool forward_unpacks(int quant_type, int64_t rows, int64_t in_features, int64_t out_features) {
    const int64_t tiles = ((rows + 255) / 256) * ((out_features + 127) / 128);
    if (!scaled_forward_format(quant_type) || tiles < SCALED_AUTO_MIN_TILES || out_features > (1 << 24) ||
        out_features * in_features > (INT64_C(1) << 29) || rows > (1 << 24)) {
        return false;
    }
    const float input = static_cast<float>(rows) * static_cast<float>(in_features), results = static_cast<float>(rows) * static_cast<float>(out_features);
    const float steps = static_cast<float>(in_features / 16);
    const bool quick = quant_type == 12 || quant_type == 13;
    const int row_tile = forward_split(rows, in_features, out_features, quant_type, OPERAND_SCALED, false).row_tile;
    const float half = row_tile == 128 ? (quick ? 0.145f : 0.19f) : quant_type == 14 ? 0.22f : 0.19f;
    const float whole = row_tile == 128 ? (quick ? 0.185f : 0.22f) : quant_type == 14 ? 0.311f : 0.273f;
    const int64_t items = ((rows + row_tile - 1) / row_tile) * ((out_features + 127) / 128);
    const float many_rows = std::min(1.0f, std::max(0.0f, (static_cast<float>(rows) - 256.0f) / 768.0f));
    const float together = 9.0f + (row_tile == 128 ? 3.0f : 7.0f) * many_rows + input * 1.0e-6f + rounds_microseconds(items, half * steps + 1.3f, whole * steps + 1.3f);
    const float apart = unpack_microseconds(out_features, in_features) + input * 0.9e-6f + (results > 1.0e8f ? results * 0.3e-6f : 0.0f) +
                        product_plan(rows, out_features, unpacked_forward_steps(quant_type, in_features)).microseconds;
    // (short reductions, but for those of Q6_K, are what the model is least sure of)
    const float margin = quant_type == 14 ? 1.03f : 1.02f + 128.0f / static_cast<float>(in_features);
    return margin * apart < together;
}
// y[i] = x W[i]^T for up to four projections of one format: the bits of the scaled kernel.  `workspace`: q8_workspace_bytes(),
// `scratch`: unpacked_forward_bytes() of all tiles of 32 weight rows.
hipError_t launch_forward_unpacked(const uint16_t * input, void * workspace, const DenseSource * sources, uint16_t * const * outputs, int count,
                                   void * scratch, int64_t rows, int64_t in_features, hipStream_t stream);

// ---- a mixture-of-experts layer of a few tokens (tgo_moe_decode.hip) ----
constexpr int MOE_DECODE_SLOTS = 64;
constexpr int MOE_DECODE_TOP_K = 8;
struct MoeDecodeArgs {
    const uint16_t * hidden;        // [tokens][features]
    const int64_t * slot_experts;   // [tokens][top_k]
    const float * slot_weights;
    const uint8_t * gate, * up, * down;
    uint16_t * activated;           // [slots][intermediate]
    uint16_t * output;              // [tokens][features]
    int tokens, top_k, slots, experts, features, intermediate;
};
// Layers that take it: 64 slots at most (its waves look them over a slot per lane), and as long as the tokens' experts are mostly
// different ones: every token unpacks its experts' down projections again.  Of the time of routing, grouped kernels and combine, eight layers with
// weights of their own in a graph, all formats: a token 0.42 to 0.66 (256 experts of 2048 x 512, IQ2_S and Q6_K: 22.9 -> 12.0 us), six tokens of
// 256 experts with power-law 0.3 routing 0.56 to 0.67 (50.5 -> 32.1), of 128 experts of 2048 x 768 with power-law 1.1 routing 0.66 to 0.90, five
// of 64 of 4096 x 1024 0.83 to 0.94.  Beyond the lines: 8 tokens of 128 of 2048 x 768, 1.1: 0.71 to 1.05; 8 of 64 of 4096 x 1024: 0.98 to 1.29; 16 of
// 256 of 2048 x 512: 0.77 to 0.92 at 0.3, 1.08 to 1.35 at 1.1.  Experts of less than half a million weights keep the operators, and with them
// the operators' bits: those round every expert's row before they add it, and their sums have another order (a line of bits, not of speed: 1024 x 512,
// on it, 17 such layers 0.40 to 0.75 of the time).  The sizes end where the kernels' instances do: a wave of the down projection holds its rows of eight experts in registers
// (up to four super-blocks each), gate and up have instances of 8 and 16 super-blocks; larger layers have not been measured.
static inline bool moe_decodes(int64_t tokens, int64_t top_k, int64_t experts, int64_t features, int64_t intermediate) {
    const int64_t slots = tokens * top_k;
    return top_k <= MOE_DECODE_TOP_K && slots <= MOE_DECODE_SLOTS && features % 256 == 0 && features <= 4096 && intermediate % 256 == 0 &&
           intermediate <= 1024 && experts > 0 && features * intermediate >= (1 << 19) && slots * features * intermediate <= (slots <= 32 ? INT64_C(1) << 27 : INT64_C(96000000));
}
hipError_t launch_moe_decode(const MoeDecodeArgs & args, int gate_up_type, int down_type, hipStream_t stream);

}  // namespace tgo
