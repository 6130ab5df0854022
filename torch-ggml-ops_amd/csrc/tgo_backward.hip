// Grad-input kernels: dX[r, k] = bf16( sum_n dY[r, n] * bf16(W[n, k]) ) on gfx950 bf16 MFMA.
//
// The cotangent is not quantized.  Three kernels:
//
// pack_cotangent_kernel copies dY (row-major bf16) into MFMA fragment order, [rows/32][chunks] slabs of 1 KiB
// laid out [half][row 0..31][8 bf16], zero-padded in both directions (columns to a multiple of 64).  One slab
// is the A operand of one v_mfma_f32_32x32x16_bf16, so the main kernels fetch it with one fully coalesced
// 16-byte-per-lane load (a row-major cotangent would cost 32 cache lines per wave load).
//
// mmq_grad_input_split_kernel: a workgroup owns 256 rows x 128 values of K (half a super-block column) and walks the
// reduction dimension N in steps of 64 weight rows.  Per step the 64 packed blocks are copied to LDS, dequantized once to bf16
// (bit-exact with the scalar reference decoder) into a tile that the multiplying waves read transposed; half of the waves dequantize, half
// multiply.  Dense calls whose tiles do not fill the chip cut N into ranges.
//
// mmq_grad_input_short_kernel: tasks of a few rows of a grouped call; described where it is defined.
//
// mmq_grad_input_kernel: the same tile as the split kernel's by four waves that all dequantize and multiply, for what lies
// beyond the 32-bit offsets of the two others: tasks of more than 64 rows of calls whose packed cotangent has 4 GiB, and every
// task of calls of 22 million weight rows.
//
// The pair variant of both walks a second (dY, W) in the same loop with one fp32 accumulator, so the sum of
// both Jacobian products is rounded to bf16 once.
#include <algorithm>

#include "tgo_cotangent.h"
#include "tgo_device.h"
#include "tgo_launch.h"

namespace tgo {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef u32x4_t u32x4;   // (a native vector type: arrays of the uint4 struct end up in scratch memory)

constexpr int BWD_TR = BACKWARD_ROW_TILE;  // rows per workgroup
constexpr int BWD_TK = 128;                // K columns per workgroup
constexpr int BWD_NS = 64;                 // weight rows per reduction step
constexpr int BWD_PITCH = BWD_NS + 8;      // bf16 per k-row of the tile: +8 keeps 16-byte reads conflict free
constexpr int BWD_THREADS = 256;
static_assert(BWD_TR == 64 * BWD_THREADS / 64, "64 rows per wave");

// ---- cotangent packing (pack_cotangent_tile) -------------------------------------------------------------
__global__ __launch_bounds__(256) void pack_cotangent_kernel(const uint16_t * __restrict__ grad_first,
                                                            const uint16_t * __restrict__ grad_second,
                                                            uint8_t * __restrict__ packed_first,
                                                            uint8_t * __restrict__ packed_second, int rows,
                                                            int out_features, int n_chunks, const TaskBuild build,
                                                            const int64_t * __restrict__ gather,
                                                            const float * __restrict__ scale, int64_t gather_rows) {
    __shared__ __attribute__((aligned(16))) uint8_t tile[PACK_TILE_BYTES];
    if (build.tasks.count != nullptr && blockIdx.x == 0 && blockIdx.y == 0 && blockIdx.z == 0) {
        build_tasks(build, threadIdx.x);
    }
    pack_cotangent_tile(tile, blockIdx.z == 0 ? grad_first : grad_second, blockIdx.z == 0 ? packed_first : packed_second, blockIdx.x,
                        blockIdx.y * 8, rows, out_features, n_chunks, n_chunks, gather, scale, gather_rows, threadIdx.x);
}

hipError_t launch_pack_cotangent(const uint16_t * grad, const uint16_t * grad_second, uint8_t * packed,
                                 uint8_t * packed_second, int rows, int out_features, hipStream_t stream,
                                 const TaskBuild * build, const int64_t * gather, const float * scale,
                                 int64_t gather_rows) {
    if ((grad_second == nullptr) != (packed_second == nullptr)) {
        return hipErrorInvalidValue;
    }
    if (gather != nullptr && (grad_second != nullptr || scale == nullptr || gather_rows <= 0)) {
        return hipErrorInvalidValue;
    }
    const int n_chunks = cotangent_chunks(out_features);
    const dim3 grid(static_cast<unsigned>((rows + 31) / 32), static_cast<unsigned>((n_chunks + 7) / 8),
                    grad_second != nullptr ? 2 : 1);
    const ProfileScope scope(6, stream);
    pack_cotangent_kernel<<<grid, 256, 0, stream>>>(grad, grad_second, packed, packed_second, rows, out_features,
                                                    n_chunks, build != nullptr ? *build : no_task_build(), gather,
                                                    scale, gather_rows);
    return hipGetLastError();
}

// ---- main kernel ----------------------------------------------------------------------------------------
struct BackwardArgs {
    const uint8_t * cotangent[2];   // fragment-ordered dY, see pack_cotangent_kernel
    const uint8_t * packed[2];
    int64_t bytes_per_expert;
    int64_t row_bytes;
    uint16_t * dx;
    const int32_t * task_count;   // nullptr: dense
    const int32_t * task_early;   // tasks listed before the short ones (at most BACKWARD_SHORT_ROWS rows each)
    const int32_t * task_expert;
    const int32_t * task_row_start;
    const int32_t * task_row_end;
    int segment;        // which tasks of the list a launch runs: 0 all, 1 those before the short ones, 2 the short ones
    int rows;
    int rows_padded;    // rows rounded up to 32: extent of the packed cotangent
    int out_features;   // N, the reduction dimension
    int n_chunks;       // 16-column chunks of the packed cotangent (N rounded up to 64, over 16)
    int in_features;    // K
    int k_tiles;        // K / 128
    int task_slots;
    int short_slots;    // upper bound of the short tasks (one per group at most)
    int sources;        // 1, or 2 for the fused pair
    // Dense calls too small to fill the chip: the reduction over the weight rows is cut into n_splits ranges of
    // steps, blockIdx.y picks one, and the workgroup writes its fp32 sums to partial[split][row][K] instead of
    // dx; reduce_partials_kernel adds them in split order.  n_splits == 1: plain operation.
    float * partial;
    int n_splits;
};

// Q4_K / Q5_K: a thread decodes 8 weight rows x 4 consecutive K positions and stores each K position's
// eight bf16 values with one 16-byte write.  `scale_min` holds (d*sc, dmin*m) per row and 32-value group.
template <int TYPE>
TGO_DEVICE void decode_k45_octet(const uint8_t * raw, const float2 * scale_min, uint16_t * wb, int tid,
                                 int half_block, int n0, int n_total) {
    using F = Format<TYPE>;
    constexpr int QS = TYPE == Q4_K ? 16 : 48;
    const int octet = tid & 7;
    const int word = (tid >> 3) & 15;
    const int nibble = tid >> 7;
    const int chunk = word >> 3;                       // 64-value chunk inside this half block
    const int position = (word & 7) * 4;               // first of 4 positions inside the 32-value group
    const int group_local = 2 * chunk + nibble;        // 32-value group inside this half block
    const int group = 4 * half_block + group_local;
    float w[4][8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int n = 8 * octet + i;
        const uint8_t * blk = raw + n * F::RAW_PITCH;
        uint32_t q = (lds_u32(blk + QS + 64 * half_block + 4 * word) >> (4 * nibble)) & 0x0f0f0f0fu;
        if constexpr (TYPE == Q5_K) {
            q |= ((lds_u32(blk + 16 + position) >> group) & 0x01010101u) << 4;
        }
        const float2 sm = scale_min[group_local * (BWD_NS + 8) + n + (n >> 3)];
        const bool valid = n0 + n < n_total;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float value = sm.x * static_cast<float>((q >> (8 * e)) & 0xffu) - sm.y;
            w[e][i] = valid ? value : 0.0f;
        }
    }
    const int k_local = 32 * group_local + position;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const uint4 packed = make_uint4(pack_bf16x2(w[e][0], w[e][1]), pack_bf16x2(w[e][2], w[e][3]),
                                        pack_bf16x2(w[e][4], w[e][5]), pack_bf16x2(w[e][6], w[e][7]));
        *reinterpret_cast<uint4 *>(&wb[(k_local + e) * BWD_PITCH + 8 * octet]) = packed;
    }
}

// fp32 partial sums of range `split` straight from the accumulators (operands swapped): a lane holds row `row` of its tile
// and, as elements 4 j .. 4 j + 3, the four columns from 8 j + 4 half on: 16-byte stores
TGO_DEVICE void store_partial_32x128(const BackwardArgs & a, const v16f (&acc)[4], int split, int row, int row_end, int k_tile, int half) {
    if (row < row_end) {
        float * const out = a.partial + (static_cast<int64_t>(split) * a.rows + row) * a.in_features + k_tile * BWD_TK + 4 * half;
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                *reinterpret_cast<float4 *>(out + kt * 32 + 8 * j) =
                    make_float4(acc[kt][4 * j], acc[kt][4 * j + 1], acc[kt][4 * j + 2], acc[kt][4 * j + 3]);
            }
        }
    }
}

// First task and number of tasks of the list's segment that a launch runs.
// `ordinary`: how many of them come before the short ones (all of them in a segment of one kind).
TGO_DEVICE void task_segment(const BackwardArgs & a, int & first, int & tasks, int & ordinary) {
    const int count = a.task_count[0];
    const int early = min(a.task_early[0], count);
    first = a.segment == 2 ? early : 0;
    tasks = a.segment == 2 ? count - early : a.segment == 1 ? early : count;
    ordinary = a.segment == 0 ? early : tasks;
}
TGO_DEVICE void task_segment(const BackwardArgs & a, int & first, int & tasks) {
    int ordinary;
    task_segment(a, first, tasks, ordinary);
}

// WIDE (formats whose blocks are not multiples of 16 bytes, when wide_stage_ok holds): a step's packed blocks are
// requested as aligned 16-byte units while the previous step multiplies, like those of Q4_K / Q5_K, instead of
// being copied two bytes at a time between the multiplications and the decoding.
template <int TYPE, bool WIDE>
__global__ __launch_bounds__(BWD_THREADS, 2) void mmq_grad_input_kernel(const BackwardArgs a) {
    using F = Format<TYPE>;
    constexpr int KT = 4;   // 32-column tiles per wave
    constexpr bool FAST_K45 = TYPE == Q4_K || TYPE == Q5_K;
    constexpr int RAW_UNITS = F::BLOCK_BYTES / 16;                              // 16-byte units per block (fast types)
    constexpr int RAW_REGS = (BWD_NS * RAW_UNITS + BWD_THREADS - 1) / BWD_THREADS;  // units in flight per thread
    static_assert(!(WIDE && FAST_K45), "the wide copy is for the 2-byte aligned formats");
    using W = WideStage<TYPE>;
    constexpr int WIDE_REGS = WIDE ? W::template regs<BWD_NS, BWD_THREADS>() : 1;
    constexpr int SLOT_PITCH = WIDE ? W::PITCH : F::RAW_PITCH;
    constexpr int SLOT_FRONT = WIDE ? W::FRONT : F::RAW_SHIFT;
    constexpr bool AHEAD = FAST_K45 || WIDE;   // the packed blocks of the next step travel through registers
    __shared__ __attribute__((aligned(16))) uint8_t raw[BWD_NS * SLOT_PITCH];
    __shared__ __attribute__((aligned(16))) uint8_t raw_odd[WIDE ? BWD_NS * SLOT_PITCH : 16];   // second slot of the WIDE pipeline
    __shared__ __attribute__((aligned(16))) uint16_t wb[2][BWD_TK * BWD_PITCH];
    __shared__ float2 scale_min[FAST_K45 ? 4 * (BWD_NS + 8) : 1];
    // (IQ2_S: the selector table of decode16_bf16; the other formats have no codebook)
    using Codebook = std::conditional_t<TYPE == IQ2_S, Iq2sSelectors, uint2>;
    __shared__ Codebook codebook_storage;
    const Codebook * const grid = &codebook_storage;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31;
    const int half = lane >> 5;

    int k_tile, task, first_task = 0, ordinary = 0;
    int tasks = (a.rows + BWD_TR - 1) / BWD_TR;
    if (a.task_count != nullptr) {
        task_segment(a, first_task, tasks, ordinary);
    }
    if (a.task_count != nullptr) {
        xcd_chunk(blockIdx.x, a.k_tiles, tasks, ordinary, k_tile, task);
    } else {
        xcd_tile(blockIdx.x, a.k_tiles, tasks, k_tile, task);
    }
    const int kb = k_tile >> 1;          // super-block column
    const int half_block = k_tile & 1;   // which 128 values of it

    int expert = 0, row_start, row_end;
    if (a.task_count != nullptr) {
        if (task >= tasks) {
            return;
        }
        task += first_task;
        expert = a.task_expert[task];
        row_start = a.task_row_start[task];
        row_end = a.task_row_end[task];
    } else {
        row_start = task * BWD_TR;
        if (row_start >= a.rows) {
            return;
        }
        row_end = min(a.rows, row_start + BWD_TR);
    }
    if constexpr (TYPE == IQ2_S) {
        expand_iq2s_selectors(codebook_storage, tid, BWD_THREADS);
    }

    const int wave_row = row_start + wave * 64;
    const bool wave_active = wave_row < row_end;
    const int n_total = a.out_features;
    const int steps_per_source = (n_total + BWD_NS - 1) / BWD_NS;
    const int steps = steps_per_source * a.sources;
    const int split = blockIdx.y;
    const int step_begin = steps * split / a.n_splits;        // (n_splits <= steps: no range is empty)
    const int step_end = steps * (split + 1) / a.n_splits;

    // byte offset of this lane's fragment piece inside the packed cotangent, per 32-row tile of the wave
    int64_t lane_offset[2];
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
        int r = wave_row + rt * 32 + l32;
        r = r < a.rows_padded ? r : a.rows_padded - 1;
        lane_offset[rt] = static_cast<int64_t>(r >> 5) * a.n_chunks * 1024 + ((r & 31) + 32 * half) * 16;
    }

    v16f acc[2][KT];
#pragma unroll
    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[rt][kt][v] = 0.0f;

    uint4 afrag[2][4] = {};     // cotangent fragments of the step about to be multiplied
    u32x4 raw_regs[FAST_K45 ? RAW_REGS : 1];   // (a native vector type: arrays of the uint4 struct end up in scratch memory)
    WideRegs<WIDE_REGS> wide_regs;

    // requests the cotangent fragments of a step: chunk s covers columns n0 + 16 s .. + 16
    auto load_cotangent = [&](int step) __attribute__((always_inline)) {
        const int source = step / steps_per_source;
        const int n0 = (step - source * steps_per_source) * BWD_NS;
        const uint8_t * base = a.cotangent[source];
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int chunk = (n0 >> 4) + s;
                afrag[rt][s] = chunk < a.n_chunks
                    ? *reinterpret_cast<const uint4 *>(base + lane_offset[rt] + static_cast<int64_t>(chunk) * 1024)
                    : make_uint4(0, 0, 0, 0);
            }
        }
    };
    // requests / stores the packed blocks of a step (16-byte aligned types travel through registers)
    auto load_raw = [&](int step) __attribute__((always_inline)) {
        const int source = step / steps_per_source;
        const int n0 = (step - source * steps_per_source) * BWD_NS;
        const uint8_t * weights = a.packed[source] + static_cast<int64_t>(expert) * a.bytes_per_expert;
        if constexpr (FAST_K45) {
#pragma unroll
            for (int i = 0; i < RAW_REGS; ++i) {
                const int id = tid + BWD_THREADS * i;
                const int row = id / RAW_UNITS;
                const int unit = id - row * RAW_UNITS;
                if (row < BWD_NS) {
                    int src_row = n0 + row;
                    src_row = src_row < n_total ? src_row : n_total - 1;
                    raw_regs[i] = *reinterpret_cast<const u32x4 *>(
                        weights + src_row * a.row_bytes + static_cast<int64_t>(kb) * F::BLOCK_BYTES + unit * 16);
                }
            }
        } else if constexpr (WIDE) {
            wide_fetch<TYPE, BWD_NS, BWD_THREADS, WIDE_REGS>(wide_regs, weights + n0 * a.row_bytes, static_cast<int>(a.row_bytes),
                                                             min(BWD_NS, n_total - n0), kb, tid);
        } else {
            stage_blocks<TYPE>(raw, weights, a.row_bytes, n0, n_total, kb, BWD_NS, tid, BWD_THREADS);
        }
    };
    auto store_raw = [&](int step) __attribute__((always_inline)) {
        if constexpr (WIDE) {
            const int source = step / steps_per_source;
            const int n0 = (step - source * steps_per_source) * BWD_NS;
            const uint8_t * weights = a.packed[source] + static_cast<int64_t>(expert) * a.bytes_per_expert;
            wide_park<TYPE, BWD_NS, BWD_THREADS, WIDE_REGS>(raw, wide_regs, weights + n0 * a.row_bytes, static_cast<int>(a.row_bytes),
                                                            min(BWD_NS, n_total - n0), kb, tid);
        }
        if constexpr (FAST_K45) {
#pragma unroll
            for (int i = 0; i < RAW_REGS; ++i) {
                const int id = tid + BWD_THREADS * i;
                const int row = id / RAW_UNITS;
                const int unit = id - row * RAW_UNITS;
                if (row < BWD_NS) {
                    *reinterpret_cast<u32x4 *>(raw + row * F::RAW_PITCH + unit * 16) = raw_regs[i];
                }
            }
        }
    };
    // dequantizes the staged blocks of a step into one of the two bf16 tiles (ends with the tile visible)
    auto decode = [&](int step, uint16_t * tile) __attribute__((always_inline)) {
        const int source = step / steps_per_source;
        const int n0 = (step - source * steps_per_source) * BWD_NS;
        __syncthreads();   // staged blocks visible
        if constexpr (FAST_K45) {
            const int n = tid & 63;
            const int group_local = tid >> 6;
            const uint8_t * blk = raw + n * F::RAW_PITCH;
            int sc, mn;
            k_scale_min(blk + 4, 4 * half_block + group_local, sc, mn);
            scale_min[group_local * (BWD_NS + 8) + n + (n >> 3)] =
                make_float2(half_bits_to_float(lds_u16(blk)) * static_cast<float>(sc),
                            half_bits_to_float(lds_u16(blk + 2)) * static_cast<float>(mn));
            __syncthreads();
            decode_k45_octet<TYPE>(raw, scale_min, tile, tid, half_block, n0, n_total);
        } else {
            // 64 rows x 8 units of 16 values; a half-wave writes 32 consecutive n of one k
#pragma unroll 1
            for (int pass = 0; pass < 2; ++pass) {
                const int id = tid + BWD_THREADS * pass;
                const int n = id & 63;
                const int unit = id >> 6;
                uint32_t pairs[8];
                decode16_bf16<TYPE>(raw + n * SLOT_PITCH + SLOT_FRONT, 8 * half_block + unit, grid, pairs);
                const bool valid = n0 + n < n_total;
                // Neighbouring lanes hold neighbouring weight rows of the same 16 values of K.  They swap pairs of
                // bf16 values so that the even lane writes both rows of an even k and the odd lane both rows of the
                // odd k, 4 bytes at a time: half the LDS writes of one 2-byte write per value.
                const uint32_t selector = (lane & 1) != 0 ? 0x03020706u : 0x05040100u;
                uint32_t * const pair_row = reinterpret_cast<uint32_t *>(&tile[(unit * 16 + (lane & 1)) * BWD_PITCH + (n & ~1)]);
#pragma unroll
                for (int j = 0; j < 16; j += 2) {
                    const uint32_t own = valid ? pairs[j / 2] : 0u;
                    const uint32_t other = static_cast<uint32_t>(
                        __builtin_amdgcn_mov_dpp(static_cast<int>(own), 0xB1, 0xf, 0xf, true));   // lane ^ 1
                    pair_row[j * (BWD_PITCH / 2)] = __builtin_amdgcn_perm(other, own, selector);
                }
            }
        }
        __syncthreads();   // tile visible
    };

    if constexpr (WIDE) {
        // One barrier per step, and every wave both multiplies and dequantizes between two barriers: while the matrix
        // instructions of step i run on tile i % 2, the same wave's vector instructions decode step i + 1 from its
        // parked blocks into the other tile (the two kinds of instruction issue independently, so inside one block
        // of code they overlap), the blocks of step i + 2 go from registers to the raw slot that step i was decoded
        // from, those of step i + 3 are requested, and each quarter of the cotangent fragments is re-requested for
        // step i + 1 as soon as the matrix instructions of step i that read it have been issued.  Steps past the
        // end repeat the last one where that avoids a branch around a load.
        const int last = step_end - 1;
        auto blocks_of = [&](int step, const uint8_t *& tile_rows, int & rows_valid) __attribute__((always_inline)) {
            step = min(step, last);
            const int source = step / steps_per_source;
            const int n0 = (step - source * steps_per_source) * BWD_NS;
            tile_rows = a.packed[source] + static_cast<int64_t>(expert) * a.bytes_per_expert + n0 * a.row_bytes;
            rows_valid = min(BWD_NS, n_total - n0);
        };
        auto request = [&](int step) __attribute__((always_inline)) {
            const uint8_t * tile_rows;
            int rows_valid;
            blocks_of(step, tile_rows, rows_valid);
            wide_fetch<TYPE, BWD_NS, BWD_THREADS, WIDE_REGS>(wide_regs, tile_rows, static_cast<int>(a.row_bytes), rows_valid, kb, tid);
        };
        auto park = [&](int step, uint8_t * slot) __attribute__((always_inline)) {
            const uint8_t * tile_rows;
            int rows_valid;
            blocks_of(step, tile_rows, rows_valid);
            wide_park<TYPE, BWD_NS, BWD_THREADS, WIDE_REGS>(slot, wide_regs, tile_rows, static_cast<int>(a.row_bytes), rows_valid, kb, tid);
        };
        // half of a step's 64 rows x 8 units of 16 values; a half-wave writes 32 consecutive n of one k
        auto decode_pass = [&](int step, int pass, const uint8_t * slot, uint16_t * tile) __attribute__((always_inline)) {
            const int source = step / steps_per_source;
            const int n0 = (step - source * steps_per_source) * BWD_NS;
            const int n = lane;
            const int unit = wave + 4 * pass;   // (wave-uniform: the unit's shifts and offsets are scalars)
            uint32_t pairs[8];
            decode16_bf16<TYPE>(slot + n * SLOT_PITCH + SLOT_FRONT, 8 * half_block + unit, grid, pairs);
            // rows past the end of the weight matrix become zeros (a mask the compiler cannot see through: a visible
            // condition ends up as a branch around part of the arithmetic, which splits the block of code that the
            // matrix and vector instructions are meant to share)
            uint32_t keep = n0 + n < n_total ? 0xffffffffu : 0u;
            asm volatile("" : "+v"(keep));
            // (pairs of lanes swap halves so that each writes both rows of one k: see the two-barrier loop's decode)
            const uint32_t selector = (lane & 1) != 0 ? 0x03020706u : 0x05040100u;
            uint32_t * const pair_row = reinterpret_cast<uint32_t *>(&tile[(unit * 16 + (lane & 1)) * BWD_PITCH + (n & ~1)]);
#pragma unroll
            for (int j = 0; j < 16; j += 2) {
                const uint32_t own = pairs[j / 2] & keep;
                const uint32_t other = static_cast<uint32_t>(
                    __builtin_amdgcn_mov_dpp(static_cast<int>(own), 0xB1, 0xf, 0xf, true));   // lane ^ 1
                pair_row[j * (BWD_PITCH / 2)] = __builtin_amdgcn_perm(other, own, selector);
            }
        };
        auto request_cotangent = [&](int step, int s) __attribute__((always_inline)) {
            const int source = step / steps_per_source;
            const int n0 = (step - source * steps_per_source) * BWD_NS;
            const uint8_t * base = a.cotangent[source];
#pragma unroll
            for (int rt = 0; rt < 2; ++rt) {
                // (the packed cotangent is zero padded to whole steps of 64 columns)
                afrag[rt][s] = *reinterpret_cast<const uint4 *>(
                    base + lane_offset[rt] + static_cast<int64_t>((n0 >> 4) + s) * 1024);
            }
        };
        // the weight fragments of chunk s of a tile (one per 32-column tile of the wave), and the chunk's multiplications
        uint4 fragment[2][KT];
        auto read_fragments = [&](const uint16_t * tile, int s) __attribute__((always_inline)) {
#pragma unroll
            for (int kt = 0; kt < KT; ++kt) {
                const int k = kt * 32 + l32;
                fragment[s & 1][kt] = *reinterpret_cast<const uint4 *>(&tile[k * BWD_PITCH + 16 * s + 8 * half]);
            }
        };
        auto multiply = [&](int s) __attribute__((always_inline)) {
#pragma unroll
            for (int kt = 0; kt < KT; ++kt) {
                const v8bf bfrag = __builtin_bit_cast(v8bf, fragment[s & 1][kt]);
#pragma unroll
                for (int rt = 0; rt < 2; ++rt) {
                    // (operands swapped: the lane then holds one task row and runs of four neighbouring columns, which
                    // the epilogue stages with 8-byte LDS writes)
                    acc[rt][kt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bfrag, __builtin_bit_cast(v8bf, afrag[rt][s]), acc[rt][kt], 0, 0, 0);
                }
            }
        };
        request(step_begin);
        park(step_begin, raw);
        request(step_begin + 1);
        __syncthreads();
        decode_pass(step_begin, 0, raw, wb[0]);
        decode_pass(step_begin, 1, raw, wb[0]);
        if (wave_active) {
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                request_cotangent(step_begin, s);
            }
        }
        park(step_begin + 1, raw_odd);
        request(step_begin + 2);
        __syncthreads();
        auto run = [&](auto active_tag) __attribute__((always_inline)) {
            constexpr bool ACTIVE = decltype(active_tag)::value;
            // vector instructions scheduled behind each matrix instruction of a step (12: measured best of 0..16)
            constexpr int INTERLEAVED_VALU = 12;
#pragma unroll 1
            for (int step = step_begin; step < last; ++step) {
                const int parity = (step - step_begin) & 1;
                const uint16_t * tile = wb[parity];
                uint16_t * next_tile = wb[parity ^ 1];
                const uint8_t * next_raw = parity != 0 ? raw : raw_odd;
                if constexpr (ACTIVE) {
                    read_fragments(tile, 0);
                }
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    if constexpr (ACTIVE) {
                        if (s + 1 < 4) {
                            read_fragments(tile, s + 1);   // an LDS round trip ahead of the instructions they feed
                        }
                        multiply(s);
                        request_cotangent(step + 1, s);
                    }
                    if (s == 0 || s == 2) {
                        decode_pass(step + 1, s >> 1, next_raw, next_tile);
                    }
                    if (s == 1) {
                        park(step + 2, parity != 0 ? raw_odd : raw);
                    }
                    if (s == 3) {
                        request(step + 3);
                    }
                    if constexpr (ACTIVE) {
                        // one matrix instruction, then a run of the vector instructions that share its chunk
#pragma unroll
                        for (int i = 0; i < 2 * KT; ++i) {
                            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                            __builtin_amdgcn_sched_group_barrier(0x002, INTERLEAVED_VALU, 0);
                        }
                    }
                }
                __syncthreads();
            }
            if constexpr (ACTIVE) {
                const uint16_t * tile = wb[(last - step_begin) & 1];
                read_fragments(tile, 0);
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    if (s + 1 < 4) {
                        read_fragments(tile, s + 1);
                    }
                    multiply(s);
                }
            }
        };
        if (wave_active) {
            run(std::true_type{});
        } else {
            run(std::false_type{});
        }
    } else {
        // prologue: the first step staged and decoded, its cotangent fragments requested
        load_raw(step_begin);
        if (wave_active) {
            load_cotangent(step_begin);
        }
        store_raw(step_begin);
        decode(step_begin, wb[0]);

        for (int step = step_begin; step < step_end; ++step) {
            const bool more = step + 1 < step_end;
            if (more) {
                if constexpr (AHEAD) {
                    load_raw(step + 1);      // in flight during the MFMAs below
                }
            }
            if (wave_active) {
                const uint16_t * tile = wb[(step - step_begin) & 1];
#pragma unroll
                for (int s = 0; s < 4; ++s) {
#pragma unroll
                    for (int kt = 0; kt < KT; ++kt) {
                        const int k = kt * 32 + l32;
                        const uint4 bits = *reinterpret_cast<const uint4 *>(&tile[k * BWD_PITCH + 16 * s + 8 * half]);
                        const v8bf bfrag = __builtin_bit_cast(v8bf, bits);
#pragma unroll
                        for (int rt = 0; rt < 2; ++rt) {
                            acc[rt][kt] =
                                __builtin_amdgcn_mfma_f32_32x32x16_bf16(bfrag, __builtin_bit_cast(v8bf, afrag[rt][s]), acc[rt][kt], 0, 0, 0);
                        }
                    }
                }
            }
            if (more) {
                if (wave_active) {
                    load_cotangent(step + 1);   // in flight while the next tile is decoded
                }
                if constexpr (AHEAD) {
                    store_raw(step + 1);
                } else {
                    load_raw(step + 1);
                }
                decode(step + 1, wb[(step + 1 - step_begin) & 1]);
            }
        }

    }

    __syncthreads();   // the tiles are free: each wave reuses 8.5 KiB of them to transpose its results
    if (!wave_active) {
        return;
    }
    if (a.n_splits > 1) {
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
            store_partial_32x128(a, acc[rt], split, wave_row + rt * 32 + l32, row_end, k_tile, half);
        }
        return;
    }
    uint16_t * stage = &wb[0][0] + wave * (32 * (BWD_TK + 8));
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
        const int r0 = wave_row + rt * 32;
        if (r0 < row_end) {
            store_rows_32x128<BWD_TK + 8, true, true>(stage, acc[rt], a.dx + static_cast<int64_t>(r0) * a.in_features + k_tile * BWD_TK,
                                                a.in_features, row_end - r0, BWD_TK, lane);
        }
    }
}

// A tile of the two kernels below lies as the weights do, [weight row][K column], and is transposed on its way out (the fragments want eight weight rows of a column
// per lane).  The 16-byte granules of a row are exchanged by the row's number, so that the lanes which the LDS serves together, eight that store
// along two rows or 16 that read from four, find theirs on different banks.
constexpr int BWD_ROW_PITCH = BWD_TK * 2;
TGO_DEVICE int tile_granule(int row, int granule) { return granule ^ ((row & 3) * 5); }
// A fragment of 16 weight rows x 32 K columns (column tile kt): lane (column, half) wants eight weight rows of its column.  ds_read_b64_tr_b16 gives
// lane i of 16 the i-th column of the four rows x 16 columns that the 16 lanes address, four lanes side by side in a row; two of them make the
// fragment, the second four rows further on.
TGO_DEVICE uint32_t transposed_offset(int lane, int kt) {
    const int row = (lane >> 2) & 3, half = lane >> 5;
    return (8 * half + row) * BWD_ROW_PITCH + tile_granule(row, 4 * kt + 2 * ((lane >> 4) & 1) + ((lane >> 1) & 1)) * 16 + 8 * (lane & 1);
}
TGO_DEVICE v8bf transposed_fragment(const uint8_t * first, const uint8_t * second) {
    typedef short four_t __attribute__((ext_vector_type(4)));
    typedef short eight_t __attribute__((ext_vector_type(8)));
    const four_t low = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) four_t *)(first));
    const four_t high = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) four_t *)(second));
    return __builtin_bit_cast(v8bf, eight_t{low.x, low.y, low.z, low.w, high.x, high.y, high.z, high.w});
}

// What a column tile, half a super-block, needs of a block, in 16-byte pieces at their own addresses.  Slot of a row in LDS, PITCH bytes:
//   Q4_K   header 0, nibbles 16            Q5_K   header 0, fifth bits 16, nibbles 48
//   Q3_K   high bits 0, low bits 32, the block's last 16 bytes 64: scales from 66, d at 78
//   Q6_K   low bits 0, high bits 64, scales 96, the block's last 16 bytes 112: d at 126
//   IQ2_S  indices 0, signs 16, upper index bits 32, scales 40, the block's first 16 bytes 48: d there
template <int TYPE>
struct HalfBlockPieces {
    static constexpr int UNITS = TYPE == Q5_K ? 7 : TYPE == Q6_K ? 8 : TYPE == IQ2_S ? 4 : 5;
    static constexpr int PITCH = UNITS % 2 == 1 ? 16 * UNITS : 16 * UNITS + 16;   // (4 * odd words: rows spread over the banks)
    static constexpr int REGS = (BWD_NS / 4 * UNITS + 63) / 64;   // of a wave's 16 weight rows, per lane
    __device__ __forceinline__ static int offset(int unit, int half_block) {   // of a piece in the block
        if constexpr (TYPE == Q4_K) {
            return unit == 0 ? 0 : 64 * half_block + 16 * unit;
        } else if constexpr (TYPE == Q5_K) {
            return unit < 3 ? 16 * unit : 64 * half_block + 16 * unit;
        } else if constexpr (TYPE == Q3_K) {
            return unit < 2 ? 16 * unit : unit < 4 ? 32 * half_block + 16 * unit : Format<TYPE>::BLOCK_BYTES - 16;
        } else if constexpr (TYPE == Q6_K) {
            return unit < 4 ? 64 * half_block + 16 * unit : unit < 6 ? 64 + 32 * half_block + 16 * unit : unit == 6 ? 192 : Format<TYPE>::BLOCK_BYTES - 16;
        } else {
            return unit < 2 ? 2 + 32 * unit + 16 * half_block : unit == 2 ? 66 : 0;
        }
    }
};

// ---- role-split variant --------------------------------------------------------------------------------------
// 256 rows x 128 values of K, reduction steps of 64 weight rows, double-buffered bf16
// tile; the eight waves of a workgroup are specialised: waves 0-3 only multiply (64 rows each), waves
// 4-7 only dequantize.  Each SIMD then holds one wave that keeps the matrix pipe busy and one that keeps the
// vector ALU busy, and the two kinds of work overlap instead of alternating; one barrier per step hands the
// finished tile over.
//
// A workgroup is persistent: it owns every gridDim.x-th (task, column tile) item and runs their reduction
// steps as one stream, so the memory latency of an item's first loads and the drain of its last step are
// paid once per workgroup instead of once per item.  Nothing is loaded where it is used.  A decoder wave owns
// 16 of a step's 64 weight rows from global load to tile write (no barrier of its own; LDS traffic inside a
// wave is ordered) and works on several consecutive steps at once: while the multipliers consume step g it
// dequantizes step g+1 from what it read of LDS during the previous round, parks the packed blocks of step g+3 in LDS, reads the inputs of
// step g+2 (IQ2_S: looks up its codebook words, and reads the indices of g+3) and has the blocks of steps g+4..g+7 in flight in registers, so no
// stage waits for the one before it.  A
// multiplier wave keeps the cotangent fragments of the next step in flight (two steps were measured: no faster, and
// the registers serve the weight-fragment look-ahead better).
//
// Measured, 256 rows of a 248320 x 2048 head (16 ranges): Q4_K 955 -> 316 us, Q6_K 655 -> 356, IQ2_S 527 -> 333 (820 TFLOP/s)
// against the general kernel, whose waves dequantize and multiply in turn.  Then a lane decoded four values of eight weight rows, for a tile that
// was stored transposed, after a stage for the block scales; with 32 values of a row per lane and the transposition in the reads (tile_granule) a
// step has neither that stage nor its two waits: 4096 tokens of eight choices among 256 experts with power-law 0.3 routing, 2 x
// 512 x 2048 IQ2_S 276 -> 254 us, 512 x 2048 Q5_K 150 -> 138; dense calls of 33 to 900 rows 0.97 on the mean.  (The LDS moves
// data for 0.31 of the time instead of 0.46, a pair of 8192 tokens Q5_K; its instructions take 0.40 to 0.58 of it over the formats and 0.43 to 0.61 before.)  With the pieces of the column tile's
// half block in place of the whole block (5 to 8 of 9 to 14) the head Q6_K 344 -> 317, IQ2_S 313 -> 305, Q5_K 319 -> 315; a pair of 8192 tokens
// Q6_K 497 -> 478, IQ2_S 448 -> 439, Q5_K 458 -> 454.  What is left: the matrix pipe is busy
// for 0.24 (tasks that half fill 256 rows, Q5_K) to 0.47 of the time (256 rows of the Q6_K head) at the clock that the card's power leaves (1.9 GHz with 256 rows of the head).
constexpr int BSP_THREADS = 512;
constexpr int BSP_ROWS_PER_DECODER = BWD_NS / 4;   // weight rows a decoder wave owns per step
constexpr int BSP_RAW_DEPTH = 4;                   // steps of packed blocks in flight per decoder wave
constexpr int BSP_COT_DEPTH = 2;                   // cotangent fragment sets per multiplier wave (1 in use)
constexpr int BSP_MAX_ITEMS = 64;                  // items per workgroup (one wave builds the table)
constexpr int BSP_GRID = 256;                      // one workgroup per CU

// The compiler's wait-count bookkeeping gives up on loads that stay in flight across the back edge of the
// persistent loop (it drains the queue once per round, which exposes a full memory latency every few steps),
// so the prefetches of the role-split kernel are issued and awaited by hand.  Global loads return in order:
// waiting until at most N of them are outstanding completes everything but the N youngest.  The wait names
// the awaited registers as read-write operands so that no use of them can be scheduled ahead of it.  What that cannot forbid
// -- a copy, a spill or a reuse of a register between its load and its wait -- check_loads_in_flight.py looks for on every
// path of the assembly, and the build fails if there is one.

// `base` must be wave-uniform (it travels in scalar registers); `offset` is this lane's byte offset.
template <int IMMEDIATE = 0>
TGO_DEVICE void async_load16(u32x4 & destination, const void * base, uint32_t offset) {
    asm volatile("global_load_dwordx4 %0, %1, %2 offset:%3" : "=v"(destination) : "v"(offset), "s"(base), "n"(IMMEDIATE));
}
template <int YOUNGER>
TGO_DEVICE void await_loads(u32x4 (&r)[1]) {
    asm volatile("s_waitcnt vmcnt(%1)" : "+v"(r[0]) : "n"(YOUNGER));
}
template <int YOUNGER>
TGO_DEVICE void await_loads(u32x4 (&r)[2]) {
    asm volatile("s_waitcnt vmcnt(%2)" : "+v"(r[0]), "+v"(r[1]) : "n"(YOUNGER));
}
template <int YOUNGER>
TGO_DEVICE void await_loads(u32x4 (&r)[4]) {
    asm volatile("s_waitcnt vmcnt(%4)" : "+v"(r[0]), "+v"(r[1]), "+v"(r[2]), "+v"(r[3]) : "n"(YOUNGER));
}
template <int YOUNGER>
TGO_DEVICE void await_loads(u32x4 (&r)[3]) {
    asm volatile("s_waitcnt vmcnt(%3)" : "+v"(r[0]), "+v"(r[1]), "+v"(r[2]) : "n"(YOUNGER));
}
template <int YOUNGER>
TGO_DEVICE void await_loads(u32x4 (&r)[2][4]) {
    asm volatile("s_waitcnt vmcnt(%8)"
                 : "+v"(r[0][0]), "+v"(r[0][1]), "+v"(r[0][2]), "+v"(r[0][3]), "+v"(r[1][0]), "+v"(r[1][1]),
                   "+v"(r[1][2]), "+v"(r[1][3])
                 : "n"(YOUNGER));
}

struct SplitItem {
    int expert;
    int row_start;
    int row_end;
    int k_tile;
    int step_begin;   // its range of reduction steps
    int step_end;
    int split;        // which range that is
};

// How the decoder waves hold a format's packed blocks.
template <int TYPE>
struct SplitBlock : HalfBlockPieces<TYPE> {
    static constexpr int SLOT_BYTES = BSP_ROWS_PER_DECODER * HalfBlockPieces<TYPE>::PITCH;
    static constexpr int BIAS = TYPE == Q3_K ? 4 : TYPE == Q6_K ? 32 : TYPE == IQ2_S ? 128 : 0;   // of the quants as unsigned bytes
};

// Position in a workgroup's stream of reduction steps, with the item's description cached in scalars.
struct SplitCursor {
    int item;
    int source;
    int n_step;
    int expert;
    int row_start;
    int row_end;
    int k_tile;
    int step_begin;
    int step_end;
    const uint8_t * base;   // where this step's loads start (meaning depends on the stage that owns the cursor)
};

template <int TYPE>
__global__ __launch_bounds__(BSP_THREADS, 2) void mmq_grad_input_split_kernel(const BackwardArgs a,
                                                                              const int total_items) {
    using B = SplitBlock<TYPE>;
    constexpr bool K45 = TYPE == Q4_K || TYPE == Q5_K;
    constexpr int RAW_UNITS = B::UNITS;
    constexpr int BSP_RAW_PITCH = B::PITCH;
    constexpr int RAW_REGS = B::REGS;
    __shared__ __attribute__((aligned(16))) uint8_t wb[2][BWD_NS * BWD_ROW_PITCH];   // [weight row][K column], bf16 (tile_granule)
    __shared__ __attribute__((aligned(16))) uint8_t raw_all[4][3][B::SLOT_BYTES];
    __shared__ uint2 grid[TYPE == IQ2_S ? TGO_IQ2S_GRID_ENTRIES : 1];   // codebook
    __shared__ __attribute__((aligned(16))) uint16_t stage_all[4][32 * (BWD_TK + 8)];
    __shared__ SplitItem items[BSP_MAX_ITEMS];
    __shared__ int item_count, step_count;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31;
    const int half = lane >> 5;

    // item table: slot i of this workgroup is linear item blockIdx.x + i * gridDim.x; empty slots (padding of
    // the task list) are squeezed out
    const int n_total = a.out_features;
    const int steps_per_source = (n_total + BWD_NS - 1) / BWD_NS;
    if constexpr (TYPE == IQ2_S) {
        expand_iq2s_grid(grid, tid, BSP_THREADS);
    }
    if (wave == 0) {
        SplitItem item = {0, 0, 0, -1, 0, steps_per_source, 0};
        const int64_t linear = blockIdx.x + static_cast<int64_t>(lane) * gridDim.x;
        if (linear < total_items) {
            int k_tile, task, first_task = 0, ordinary = 0;
            int tasks = (a.rows + BWD_TR - 1) / BWD_TR;
            if (a.n_splits > 1) {
                if (tasks == 1) {
                    // Every XCD takes an eighth of the items range by range: its L2 serves a range's cotangent to all column tiles (250 rows of a
                    // 248320 x 2048 Q6_K head 361 -> 344 us, 250 of 151936 x 4096 Q4_K 352 -> 344, 256 of 14336 x 4096 Q5_K 49.9 -> 48.9).
                    const int index = static_cast<int>(linear) % XCDS * (total_items / XCDS) + static_cast<int>(linear) / XCDS;
                    item.split = index / a.k_tiles;
                    k_tile = index - item.split * a.k_tiles;
                    task = 0;
                } else {
                    // several row tiles: the two column tiles of a super-block, which read the same packed blocks, side by side on an XCD,
                    // neighbouring super-blocks on neighbouring ones (300 rows of 4096 x 4096 Q3_K 32.2 us, 34.5 range by range; 900 of 4096 x
                    // 768 Q6_K 29.7 and 30.5)
                    const int pairs = a.k_tiles / 2;
                    const int pair = static_cast<int>(linear) / (2 * XCDS) * XCDS + static_cast<int>(linear) % XCDS;
                    const int rest = pair / pairs;
                    k_tile = 2 * (pair - rest * pairs) + (static_cast<int>(linear) / XCDS) % 2;
                    task = rest % tasks;
                    item.split = rest / tasks;
                }
                item.step_begin = static_cast<int>(static_cast<int64_t>(steps_per_source) * item.split / a.n_splits);
                item.step_end = static_cast<int>(static_cast<int64_t>(steps_per_source) * (item.split + 1) / a.n_splits);
                task = item.split < a.n_splits ? task : tasks;
            } else if (a.task_count != nullptr) {
                task_segment(a, first_task, tasks, ordinary);   // (never the short segment: first_task is 0)
                xcd_chunk(static_cast<int>(linear), a.k_tiles, tasks, ordinary, k_tile, task);
            } else {
                xcd_tile(static_cast<int>(linear), a.k_tiles, tasks, k_tile, task);
            }
            if (a.task_count != nullptr) {
                if (task < tasks) {
                    item.expert = a.task_expert[task];
                    item.row_start = a.task_row_start[task];
                    item.row_end = a.task_row_end[task];
                    item.k_tile = k_tile;
                }
            } else if (task * BWD_TR < a.rows) {
                item.row_start = task * BWD_TR;
                item.row_end = min(a.rows, item.row_start + BWD_TR);
                item.k_tile = k_tile;
            }
        }
        const bool valid = item.k_tile >= 0;
        const unsigned long long mask = __ballot(valid);
        if (valid) {
            items[__popcll(mask & ((1ull << lane) - 1ull))] = item;
        }
        int steps = valid ? (item.step_end - item.step_begin) * a.sources : 0;
#pragma unroll
        for (int offset = 32; offset > 0; offset >>= 1) {
            steps += __shfl_xor(steps, offset);
        }
        if (lane == 0) {
            item_count = __popcll(mask);
            step_count = steps;
        }
    }
    __syncthreads();
    const int n_items = item_count;
    if (n_items == 0) {
        return;
    }
    const int total_steps = step_count;
    // Both roles walk whole rounds of the decoders' ring.  Steps behind the last one repeat its loads and are not multiplied (at
    // most three, none where the matrix has a multiple of 256 rows): so no branch leads around a load or its wait, and every
    // path through the loops is one that can be taken, which is what the build's proof (check_loads_in_flight.py) follows.
    const int walked_steps = (total_steps + BSP_RAW_DEPTH - 1) / BSP_RAW_DEPTH * BSP_RAW_DEPTH;
    static_assert(BSP_RAW_DEPTH % BSP_COT_DEPTH == 0, "the multipliers' rounds fill the decoders'");

    auto item_field = [&](int item, int field) {
        return __builtin_amdgcn_readfirstlane(reinterpret_cast<const int *>(&items[item])[field]);
    };
    auto open_item = [&](SplitCursor & c, int item) {
        c.item = item;
        c.expert = item_field(item, 0);
        c.row_start = item_field(item, 1);
        c.row_end = item_field(item, 2);
        c.k_tile = item_field(item, 3);
        c.step_begin = item_field(item, 4);
        c.step_end = item_field(item, 5);
        c.n_step = c.step_begin;
        c.source = 0;
    };
    // `rebase(cursor)` sets cursor.base for the first step of the cursor's (item, source); within a source the base
    // moves by `step_bytes` per step.
    auto first_step = [&](auto && rebase) {
        SplitCursor c;
        open_item(c, 0);
        rebase(c);
        return c;
    };
    // A cursor at the last step stays there: stages that look past the end repeat it (harmless re-reads
    // instead of branches).  Returns true when the cursor moved to another item.
    auto advance = [&](SplitCursor & c, auto && rebase, int64_t step_bytes) {
        if (c.n_step + 1 < c.step_end) {
            ++c.n_step;
            c.base += step_bytes;
            return false;
        }
        if (c.source + 1 < a.sources) {
            c.n_step = c.step_begin;
            ++c.source;
            rebase(c);
            return false;
        }
        if (c.item + 1 < n_items) {
            open_item(c, c.item + 1);
            rebase(c);
            return true;
        }
        return false;
    };
    const uint8_t * const packed_of[2] = {a.packed[0], a.packed[1]};
    const uint8_t * const cotangent_of[2] = {a.cotangent[0], a.cotangent[1]};

    // Both roles run the same number of barriers: one after the first tile, then one per step.
    if (wave >= 4) {
        // ---------------- decoder wave ----------------
        const int dw = wave - 4;
        u32x4 ring[BSP_RAW_DEPTH][RAW_REGS];
        // loads of the other BSP_RAW_DEPTH - 1 register sets are younger than the set about to be parked
        constexpr int RAW_YOUNGER = (BSP_RAW_DEPTH - 1) * RAW_REGS;

        // Lane offsets of the 16-byte units this lane fetches per step, relative to the step's first weight
        // row; the last step of a source clamps rows past the end of the matrix to its last row.
        const int tail_rows = n_total - (steps_per_source - 1) * BWD_NS;
        uint32_t unit_offset[RAW_REGS], unit_offset_tail[RAW_REGS], second_half[RAW_REGS];   // (second_half: from a piece of the first half block to the other's)
        const auto lane_row = [&](int i) { return min(lane + 64 * i, BSP_ROWS_PER_DECODER * RAW_UNITS - 1) / RAW_UNITS; };
        const auto lane_unit = [&](int i) { return min(lane + 64 * i, BSP_ROWS_PER_DECODER * RAW_UNITS - 1) % RAW_UNITS; };
#pragma unroll
        for (int i = 0; i < RAW_REGS; ++i) {
            const int row = dw * BSP_ROWS_PER_DECODER + lane_row(i);
            const int piece = B::offset(lane_unit(i), 0);
            unit_offset[i] = static_cast<uint32_t>(row * a.row_bytes + piece);
            unit_offset_tail[i] = static_cast<uint32_t>(min(row, tail_rows - 1) * a.row_bytes + piece);
            second_half[i] = static_cast<uint32_t>(B::offset(lane_unit(i), 1) - piece);
        }
        const int64_t step_bytes = BWD_NS * a.row_bytes;
        auto rebase = [&](SplitCursor & c) {
            c.base = (c.source == 0 ? packed_of[0] : packed_of[1]) + static_cast<int64_t>(c.expert) * a.bytes_per_expert +
                     static_cast<int64_t>(c.k_tile >> 1) * Format<TYPE>::BLOCK_BYTES + c.step_begin * step_bytes;
        };
        auto load_raw = [&](const SplitCursor & c, u32x4 (&regs)[RAW_REGS]) {
            const bool tail = c.n_step == steps_per_source - 1;
#pragma unroll
            for (int i = 0; i < RAW_REGS; ++i) {
                async_load16(regs[i], c.base, (tail ? unit_offset_tail[i] : unit_offset[i]) + ((c.k_tile & 1) != 0 ? second_half[i] : 0u));
            }
        };
        // stage 1: packed blocks from registers to an LDS slot
        auto park = [&](u32x4 (&regs)[RAW_REGS], uint8_t * raw) {
            await_loads<RAW_YOUNGER>(regs);
#pragma unroll
            for (int i = 0; i < RAW_REGS; ++i) {
                *reinterpret_cast<u32x4 *>(raw + lane_row(i) * BSP_RAW_PITCH + 16 * lane_unit(i)) = regs[i];
            }
        };
        // stage 2: a lane decodes 32 values of one weight row (lane / 4) in two runs of 16 along K.  The LDS reads and the arithmetic on
        // what was read are apart, so that the reads can be issued well before their results are needed (a lone wave has nothing else to
        // cover an LDS round trip with).
        struct DecodeInputs {
            uint32_t low[4], high[4];   // K45: nibbles and fifth bits; Q3_K, Q6_K: low and high bits; IQ2_S: codebook words of the runs
            uint32_t header[4];         // scales
        };
        const int n = lane >> 2, quarter = lane & 3;
        const auto unpack4 = [](const uint4 v, uint32_t (&to)[4]) {
            to[0] = v.x; to[1] = v.y; to[2] = v.z; to[3] = v.w;
        };
        auto decode_fetch = [&](int info, const uint8_t * raw) {
            const int half_block = info & 1;
            const uint8_t * const blk = raw + n * BSP_RAW_PITCH;
            DecodeInputs in = {};
            const auto bytes16 = [&](int at) { return *reinterpret_cast<const uint4 *>(blk + at); };
            if constexpr (K45) {
                unpack4(bytes16(0), in.header);
                unpack4(bytes16((TYPE == Q4_K ? 16 : 48) + 16 * quarter), in.low);
                if constexpr (TYPE == Q5_K) {
                    unpack4(bytes16(16 + 16 * (quarter & 1)), in.high);
                }
            } else if constexpr (TYPE == Q3_K) {
                unpack4(bytes16(32 + 16 * (quarter & 1)), in.low);
                unpack4(bytes16(16 * (quarter & 1)), in.high);
                const int unit = 4 * (quarter >> 1) + (quarter & 1);   // of the half block, and the one two behind it
                in.header[0] = lds_u16(blk + 78);
                in.header[1] = (static_cast<uint32_t>(blk[66 + unit]) >> (4 * half_block)) | (static_cast<uint32_t>(blk[68 + unit]) >> (4 * half_block) << 16);
                in.header[2] = blk[74 + (quarter & 1)] | (static_cast<uint32_t>(blk[76 + (quarter & 1)]) << 16);
            } else if constexpr (TYPE == Q6_K) {
                unpack4(bytes16(16 * quarter), in.low);
                unpack4(bytes16(64 + 16 * (quarter & 1)), in.high);
                in.header[0] = lds_u16(blk + 126);
                in.header[1] = blk[96 + 8 * half_block + quarter];
                in.header[2] = blk[100 + 8 * half_block + quarter];
            } else {
                in.low[0] = lds_u32(blk + 4 * quarter);        // codebook indices of four octets, eight bits each
                in.low[1] = lds_u32(blk + 16 + 4 * quarter);   // their signs
                in.low[2] = blk[32 + 4 * half_block + quarter];   // the indices' upper two bits
                in.header[0] = lds_u16(blk + 48);
                in.header[1] = blk[40 + 4 * half_block + quarter];
            }
            return in;
        };
        // IQ2_S: the codebook words that a step's indices name, a round before they are needed
        auto codebook_fetch = [&](const DecodeInputs & in) {
            DecodeInputs out = in;
            if constexpr (TYPE == IQ2_S) {
                uint32_t words[8];
#pragma unroll
                for (int o = 0; o < 4; ++o) {
                    const uint2 entry = grid[((in.low[0] >> (8 * o)) & 0xffu) | (((in.low[2] >> (2 * o)) & 3u) << 8)];
                    words[2 * o] = entry.x;
                    words[2 * o + 1] = entry.y;
                }
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    out.low[w] = words[w];
                    out.high[w] = words[4 + w];
                }
                out.header[2] = in.low[1];
            }
            return out;
        };
        auto decode_finish = [&](int info, const DecodeInputs & in, uint8_t * tile) {
            const int half_block = info & 1;
            uint32_t keep = (info >> 1) * BWD_NS + dw * BSP_ROWS_PER_DECODER + n < n_total ? 0xffffffffu : 0u;
            asm volatile("" : "+v"(keep));   // (a mask, not a branch around part of the arithmetic; rows past the end become exact zeros)
            const uint32_t header = in.header[0] & keep;
            const float d = half_bits_to_float(header & 0xffffu);
            uint8_t * const row = tile + (dw * BSP_ROWS_PER_DECODER + n) * BWD_ROW_PITCH;
            uint32_t k45_scales = 0, k45_minima = 0;
            if constexpr (K45) {
                const int shift = 16 * (quarter >> 1);
                const uint32_t first = in.header[1] >> shift, second = in.header[2] >> shift, third = in.header[3] >> shift;
                // groups 0 .. 3 of the super-block: plain 6-bit fields; 4 .. 7: nibbles of the third word, their top bits above the first four's
                k45_scales = half_block == 0 ? first & 0x3f3fu : (third & 0x0f0fu) | ((first >> 2) & 0x3030u);
                k45_minima = half_block == 0 ? second & 0x3f3fu : ((third >> 4) & 0x0f0fu) | ((second >> 2) & 0x3030u);
            }
#pragma unroll
            for (int run = 0; run < 2; ++run) {
                float scale, offset;
                int column;
                if constexpr (K45) {
                    scale = d * static_cast<float>((k45_scales >> (8 * run)) & 0xffu);
                    offset = half_bits_to_float(header >> 16) * static_cast<float>((k45_minima >> (8 * run)) & 0xffu);
                    column = 64 * (quarter >> 1) + 32 * run + 16 * (quarter & 1);
                } else {
                    if constexpr (TYPE == Q3_K) {
                        const uint32_t low = (in.header[1] >> (16 * run)) & 15u;
                        const uint32_t high = (in.header[2] >> (16 * run + 4 * half_block + 2 * (quarter >> 1))) & 3u;
                        scale = d * static_cast<float>(static_cast<int>(low | (high << 4)) - 32);
                        column = 64 * (quarter >> 1) + 32 * run + 16 * (quarter & 1);
                    } else if constexpr (TYPE == Q6_K) {
                        scale = d * static_cast<float>(static_cast<int>(in.header[1 + run] << 24) >> 24);
                        column = 64 * run + 16 * quarter;
                    } else {
                        scale = d * 0.125f * static_cast<float>(((in.header[1] >> (4 * run)) & 15u) * 2 + 1);
                        column = 32 * quarter + 16 * run;
                    }
                    // (products of an 11-bit and an at most 8-bit number: exact, and so is the bias, a power of two)
                    offset = scale * B::BIAS;
                }
                uint32_t pairs[8];
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    uint32_t q;   // four quants as unsigned bytes, above their true values by the bias
                    if constexpr (K45) {
                        q = (in.low[w] >> (4 * run)) & 0x0f0f0f0fu;
                        if constexpr (TYPE == Q5_K) {
                            q |= ((in.high[w] >> (4 * half_block + 2 * (quarter >> 1) + run)) & 0x01010101u) << 4;
                        }
                    } else if constexpr (TYPE == Q3_K) {
                        const int group = 2 * (quarter >> 1) + run;   // 32-value group of the half block
                        q = ((in.low[w] >> (2 * group)) & 0x03030303u) | (((in.high[w] >> (4 * half_block + group)) & 0x01010101u) << 2);
                    } else if constexpr (TYPE == Q6_K) {
                        q = ((in.low[w] >> (4 * run)) & 0x0f0f0f0fu) | (((in.high[w] >> (2 * (quarter >> 1) + 4 * run)) & 0x03030303u) << 4);
                    } else {
                        // the four signs spread to a bit per byte; a negative magnitude is its complement plus one
                        const uint32_t negative = (((in.header[2] >> (16 * run + 4 * w)) & 15u) * 0x00204081u) & 0x01010101u;
                        q = (((run == 0 ? in.low[w] : in.high[w]) ^ (negative * 0xffu)) + negative) ^ 0x80808080u;
                    }
                    float value[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        value[e] = scale * static_cast<float>((q >> (8 * e)) & 0xffu) - offset;
                    }
                    pairs[2 * w] = pack_bf16x2(value[0], value[1]);
                    pairs[2 * w + 1] = pack_bf16x2(value[2], value[3]);
                }
                *reinterpret_cast<uint4 *>(row + tile_granule(n, column / 8) * 16) = make_uint4(pairs[0], pairs[1], pairs[2], pairs[3]);
                *reinterpret_cast<uint4 *>(row + tile_granule(n, column / 8 + 1) * 16) = make_uint4(pairs[4], pairs[5], pairs[6], pairs[7]);
            }
        };
        auto wave_sync = [&]() {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        };
        auto raw_slot = [&](int slot) { return raw_all[dw][slot]; };

        // Step t uses raw slot t % 3, tile t & 1 and register set t % 4.  Only the load
        // stage walks the item list; what the later stages need to know about a step (which half of the
        // super-block, which 64 weight rows) follows it through a seven-deep queue of scalars.
        SplitCursor c_load = first_step(rebase);
        int info[7];   // info[i]: step g + 6 - i while the multipliers consume step g
        auto request = [&](u32x4 (&regs)[RAW_REGS]) {
            load_raw(c_load, regs);
#pragma unroll
            for (int i = 6; i > 0; --i) {
                info[i] = info[i - 1];
            }
            info[0] = (c_load.n_step << 1) | (c_load.k_tile & 1);
            advance(c_load, rebase, step_bytes);
        };
#pragma unroll
        for (int p = 0; p < BSP_RAW_DEPTH; ++p) {
            request(ring[p]);
        }
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            park(ring[t], raw_slot(t));
            request(ring[t]);
        }
        wave_sync();
        decode_finish(info[6], codebook_fetch(decode_fetch(info[6], raw_slot(0))), wb[0]);
        // IQ2_S has its codebook words looked up in the round before they are decoded, and the indices read in the round before that
        constexpr bool LOOKS_UP = TYPE == IQ2_S;
        DecodeInputs pending = codebook_fetch(decode_fetch(info[5], raw_slot(1)));   // step 1
        DecodeInputs indices = {};
        if constexpr (LOOKS_UP) {
            indices = decode_fetch(info[4], raw_slot(2));   // step 2
        }
        __syncthreads();
        // While the multipliers consume step g: finish decoding g + 1 (its inputs were read from LDS during
        // the previous round), park g + 3, request g + 7, and read the decode inputs of g + 2 so that they arrive during the barrier (IQ2_S: look
        // up what g + 2 needs first thing, and read the indices of g + 3).  LDS
        // executes a wave's accesses in order, so a stage may read what an earlier stage of the same round
        // wrote without waiting; the fences only keep the compiler from reordering them.
        int g3 = 0;   // g % 3
#pragma unroll 1
        for (int base = 0; base < walked_steps; base += BSP_RAW_DEPTH) {
#pragma unroll
            for (int u = 0; u < BSP_RAW_DEPTH; ++u) {
                const int g = base + u;
                const int g3_plus1 = g3 == 2 ? 0 : g3 + 1;
                const int g3_plus2 = g3_plus1 == 2 ? 0 : g3_plus1 + 1;
                DecodeInputs next;
                if constexpr (LOOKS_UP) {
                    next = codebook_fetch(indices);
                    __builtin_amdgcn_sched_barrier(0);
                }
                decode_finish(info[5], pending, wb[(g + 1) & 1]);
                park(ring[(u + 3) % BSP_RAW_DEPTH], raw_slot(g3));
                wave_sync();
                if constexpr (LOOKS_UP) {
                    indices = decode_fetch(info[3], raw_slot(g3));
                    pending = next;
                } else {
                    pending = decode_fetch(info[4], raw_slot(g3_plus2));
                }
                request(ring[(u + 3) % BSP_RAW_DEPTH]);
                __builtin_amdgcn_sched_barrier(0);
                g3 = g3_plus1;
                __syncthreads();
            }
        }
        return;
    }

    // ---------------- multiplier wave ----------------
    // byte offsets of this lane's fragment pieces inside the packed cotangent for an item, per 32-row tile of
    // the wave; a wave without rows in the item points every lane at one line (the loads stay, the cost goes)
    auto lane_offsets = [&](const SplitCursor & c, uint32_t (&offset)[2]) {
        const int wave_row = c.row_start + wave * 64;
        const bool active = wave_row < c.row_end;
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
            int r = wave_row + rt * 32 + l32;
            r = r < a.rows_padded ? r : a.rows_padded - 1;
            offset[rt] = active ? static_cast<uint32_t>(r >> 5) * a.n_chunks * 1024 + ((r & 31) + 32 * half) * 16 : 0;
        }
    };
    // A step covers four 16-column chunks (the packed cotangent is zero padded to whole steps); a fragment
    // set is 2 row tiles x 4 chunks.
    u32x4 cot[BSP_COT_DEPTH][2][4];
    constexpr int COT_YOUNGER = (BSP_COT_DEPTH - 1) * 8;
    uint32_t fetch_offset[2];
    auto load_cotangent = [&](const SplitCursor & c, u32x4 (&regs)[2][4]) {
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
            async_load16<0>(regs[rt][0], c.base, fetch_offset[rt]);
            async_load16<1024>(regs[rt][1], c.base, fetch_offset[rt]);
            async_load16<2048>(regs[rt][2], c.base, fetch_offset[rt]);
            async_load16<3072>(regs[rt][3], c.base, fetch_offset[rt]);
        }
    };
    auto rebase_fetch = [&](SplitCursor & c) {
        c.base = (c.source == 0 ? cotangent_of[0] : cotangent_of[1]) + static_cast<int64_t>(c.step_begin) * ((BWD_NS / 16) * 1024);
    };
    auto rebase_none = [&](SplitCursor &) {};

    // where the lane's share of a fragment of column tile kt lies (ds_read_b64_tr_b16, see transposed_fragment)
    uint32_t fragment_offset[4];
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) {
        fragment_offset[kt] = transposed_offset(lane, kt);
    }
    v16f acc[2][4];
#pragma unroll
    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[rt][kt][v] = 0.0f;

    SplitCursor c_fetch = first_step(rebase_fetch), c_now = c_fetch;
    lane_offsets(c_fetch, fetch_offset);
    auto fetch_next = [&]() {
        if (advance(c_fetch, rebase_fetch, (BWD_NS / 16) * 1024)) {
            lane_offsets(c_fetch, fetch_offset);
        }
    };
#pragma unroll
    for (int d = 0; d + 1 < BSP_COT_DEPTH; ++d) {
        load_cotangent(c_fetch, cot[d]);
        fetch_next();
    }
    __syncthreads();
#pragma unroll 1
    for (int base = 0; base < walked_steps; base += BSP_COT_DEPTH) {
#pragma unroll
        for (int u = 0; u < BSP_COT_DEPTH; ++u) {
            const int g = base + u;
            load_cotangent(c_fetch, cot[(u + BSP_COT_DEPTH - 1) % BSP_COT_DEPTH]);
            fetch_next();
            await_loads<COT_YOUNGER>(cot[u]);
            const int wave_row = c_now.row_start + wave * 64;
            const int row_end = c_now.row_end;
            if (wave_row < row_end && g < total_steps) {
                // 16 weight fragments (4 chunks x 4 column tiles), two MFMAs each.  An LDS read takes
                // longer than the two MFMAs it feeds, so fragment j + AHEAD is requested before fragment j
                // is used; the scheduling groups below pin that interleaving.
                const uint8_t * const tile = wb[g & 1];
                auto read_fragment = [&](int j) {
                    const uint8_t * const from = tile + fragment_offset[j & 3] + 16 * (j >> 2) * BWD_ROW_PITCH;
                    return transposed_fragment(from, from + 4 * BWD_ROW_PITCH);
                };
                constexpr int AHEAD = 6;
                v8bf fragment[16];
#pragma unroll
                for (int j = 0; j < AHEAD; ++j) {
                    fragment[j] = read_fragment(j);
                }
#pragma unroll
                for (int j = 0; j < 16; ++j) {
                    if (j + AHEAD < 16) {
                        fragment[j + AHEAD] = read_fragment(j + AHEAD);
                    }
#pragma unroll
                    for (int rt = 0; rt < 2; ++rt) {
                        // (operands swapped: the lane ends up with one task row and runs of four neighbouring
                        // columns, which the epilogue stages with 8-byte LDS writes instead of 2-byte ones)
                        acc[rt][j & 3] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                            fragment[j], __builtin_bit_cast(v8bf, cot[u][rt][j >> 2]),
                            acc[rt][j & 3], 0, 0, 0);
                    }
                }
                __builtin_amdgcn_sched_group_barrier(0x100, 2 * AHEAD, 0);   // LDS reads
#pragma unroll
                for (int j = 0; j < 16; ++j) {
                    if (j + AHEAD < 16) {
                        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
                    }
                    __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);   // MFMAs
                }
                if (c_now.source == a.sources - 1 && c_now.n_step == c_now.step_end - 1) {
                    // last step of the item: transpose the results through this wave's staging area
                    // and write whole rows, then start the next item from zero
                    const int k_tile = c_now.k_tile;
                    // recomputing the per-lane store offsets here is cheaper than keeping them alive
                    // (spilled) through the loop, which is what happens if they can be hoisted
                    int lane_here = lane;
                    asm volatile("" : "+v"(lane_here));
#pragma unroll
                    for (int rt = 0; rt < 2; ++rt) {
                        const int r0 = wave_row + rt * 32;
                        if (a.n_splits > 1) {
                            store_partial_32x128(a, acc[rt], item_field(c_now.item, 6), r0 + (lane_here & 31), row_end, k_tile,
                                                 lane_here >> 5);
                        } else if (r0 < row_end) {
                            store_rows_32x128<BWD_TK + 8, true, true>(
                                stage_all[wave], acc[rt],
                                a.dx + static_cast<int64_t>(r0) * a.in_features + k_tile * BWD_TK, a.in_features,
                                row_end - r0, BWD_TK, lane_here);
                        }
#pragma unroll
                        for (int kt = 0; kt < 4; ++kt)
#pragma unroll
                            for (int v = 0; v < 16; ++v) acc[rt][kt][v] = 0.0f;
                    }
                }
            }
            advance(c_now, rebase_none, 0);
            __syncthreads();
        }
    }
}

// ---- short tasks ----------------------------------------------------------------------------------------------
// Tasks of at most BACKWARD_SHORT_ROWS rows.  Dequantizing a step's 64 x 128 weights costs the same however few
// rows multiply them, so here it is nearly all of the work and every wave does it: a wave owns 16 of the step's 64
// weight rows from the global load to the bf16 tile (packed blocks DEPTH steps ahead in registers, parked in the
// wave's own LDS slot, decoded; LDS executes a wave's accesses in order, so these stages need no
// workgroup barrier), one barrier per step publishes the tile, and then every wave multiplies the task's rows with
// one 32-column slice of it (4 or 8 matrix instructions).  Small footprint: three workgroups share a CU, so one's
// barrier and memory waits are covered by the others' decoding.  One workgroup per (task, column tile).
// Blocks are fetched as 16-byte pieces at their own addresses, those that the column tile needs (HalfBlockPieces).  A lane decodes 32 values of one weight row and stores them along K; the transposition to the fragments'
// order happens in the reads (ds_read_b64_tr_b16).  Against a lane that decodes four values of eight rows and stores a transposed tile
// (24 four- and eight-byte reads of LDS per lane and step instead of three of 16 bytes): groups of 8192 tokens with power-law 1.1 routing over 256
// experts of 2 x 512 x 2048 Q5_K 133 -> 115 us, 4096 tokens with 0.3, 512 x 2048 Q5_K 57 -> 48, 2 x 512 x 2048 IQ2_S 93 -> 86.  The formats with a
// scale per 16 values unpack four quants per operation as the role-split kernel does, instead of one by one: the whole gradient of 1024 tokens of
// eight choices, 256 experts of 2 x 512 x 2048, IQ2_S 215 -> 175 us, Q3_K 205 -> 188, Q6_K 240 -> 227, and with pieces instead of the aligned units
// that cover a block, and of those only what the tile needs, 155, 177 and 193 (Q5_K 187 -> 179, Q4_K 176 -> 162; 600 tokens of 128 experts of 2048 x
// 768: IQ2_S 118 -> 90, Q3_K 104 -> 89, Q6_K 115 -> 91).  Four workgroups per CU, which Q3_K to Q5_K then have room for, are no faster.  No unit
// is full: the groups of 8192 tokens above have the LDS busy for 0.52 of the time (Q5_K), the vector unit for 0.45, the matrix cores for 0.10, and their
// waves wait for a counter 0.30 of theirs.
constexpr int BSH_THREADS = 256;
constexpr int BSH_ROWS_PER_WAVE = BWD_NS / 4;
constexpr int BSH_DEPTH = 2;

template <int TYPE>
__global__ __launch_bounds__(BSH_THREADS, 3) void mmq_grad_input_short_kernel(const BackwardArgs a) {
    using B = HalfBlockPieces<TYPE>;
    constexpr bool K45 = TYPE == Q4_K || TYPE == Q5_K;
    constexpr int RAW_UNITS = B::UNITS;
    constexpr int RAW_PITCH = B::PITCH;
    constexpr int RAW_REGS = B::REGS;
    __shared__ __attribute__((aligned(16))) uint8_t wb[2][BWD_NS * BWD_ROW_PITCH];   // [weight row][K column], bf16 (tile_granule)
    __shared__ __attribute__((aligned(16))) uint8_t raw_all[4][BSH_ROWS_PER_WAVE * RAW_PITCH];
    // (the magnitude grid: with the 16 KiB selector table of decode16_bf16 only two of these workgroups fit a CU instead of three)
    __shared__ uint2 grid[TYPE == IQ2_S ? TGO_IQ2S_GRID_ENTRIES : 1];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31;
    const int half = lane >> 5;

    int k_tile, task, first_task, tasks;
    task_segment(a, first_task, tasks);
    xcd_tile(blockIdx.x, a.k_tiles, tasks, k_tile, task);
    if (task >= tasks) {
        return;
    }
    task += first_task;
    const int expert = a.task_expert[task];
    const int row_start = a.task_row_start[task];
    const int row_end = a.task_row_end[task];
    const int kb = k_tile >> 1;
    const int half_block = k_tile & 1;
    const int row_tiles = (row_end - row_start + 31) / 32;   // 1 or 2
    const int n_total = a.out_features;
    const int steps_per_source = (n_total + BWD_NS - 1) / BWD_NS;
    const int steps = steps_per_source * a.sources;
    const int last = steps - 1;

    uint8_t * const raw = raw_all[wave];
    if constexpr (TYPE == IQ2_S) {
        expand_iq2s_grid(grid, tid, BSH_THREADS);   // (visible after the barrier that follows the first decode's inputs)
        __syncthreads();
    }

    // lane offsets of the 16-byte units this lane fetches per step, relative to the step's first weight row
    // (the last step of a source clamps rows past the end of the matrix to its last row)
    const int tail_rows = n_total - (steps_per_source - 1) * BWD_NS;
    uint32_t unit_offset[RAW_REGS], unit_offset_tail[RAW_REGS];
#pragma unroll
    for (int i = 0; i < RAW_REGS; ++i) {
        const int id = min(lane + 64 * i, BSH_ROWS_PER_WAVE * RAW_UNITS - 1);
        const int row = wave * BSH_ROWS_PER_WAVE + id / RAW_UNITS;
        const int piece = B::offset(id % RAW_UNITS, half_block);
        unit_offset[i] = static_cast<uint32_t>(row * a.row_bytes + piece);
        unit_offset_tail[i] = static_cast<uint32_t>(min(row, tail_rows - 1) * a.row_bytes + piece);
    }
    const int64_t expert_offset = static_cast<int64_t>(expert) * a.bytes_per_expert + static_cast<int64_t>(kb) * Format<TYPE>::BLOCK_BYTES;
    // A step's packed blocks in flight.  (Pieces of the 2-byte aligned formats start on any even address.)
    typedef uint32_t even_t __attribute__((ext_vector_type(4), aligned(2)));
    struct InFlight {
        u32x4 unit[RAW_REGS];
    };
    auto request = [&](int step, InFlight & regs) __attribute__((always_inline)) {
        step = min(step, last);
        const int source = step >= steps_per_source ? 1 : 0;
        const int n_step = step - source * steps_per_source;
        const uint8_t * base = (source == 0 ? a.packed[0] : a.packed[1]) + expert_offset +
                               static_cast<int64_t>(n_step) * BWD_NS * a.row_bytes;
        const bool tail = n_step == steps_per_source - 1;
#pragma unroll
        for (int i = 0; i < RAW_REGS; ++i) {
            const uint8_t * const from = base + (tail ? unit_offset_tail[i] : unit_offset[i]);
            if constexpr (K45) {
                regs.unit[i] = *reinterpret_cast<const u32x4 *>(from);
            } else {
                regs.unit[i] = *reinterpret_cast<const even_t *>(from);
            }
        }
    };
    auto park = [&](const InFlight & regs) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < RAW_REGS; ++i) {
            const int id = min(lane + 64 * i, BSH_ROWS_PER_WAVE * RAW_UNITS - 1);
            const int row = id / RAW_UNITS;
            const int unit = id - row * RAW_UNITS;
            *reinterpret_cast<u32x4 *>(raw + row * RAW_PITCH + unit * 16) = regs.unit[i];
        }
    };
    auto wave_sync = [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    // A lane decodes 32 values of one weight row (its own, lane / 4): whole 16-byte pieces of the block, the scales from its header, and
    // four 16-byte stores along K.  Rows past the end of the weight matrix decode to exact zeros.
    const int n = lane >> 2;
    uint8_t * const tile_row = &wb[0][(wave * BSH_ROWS_PER_WAVE + n) * BWD_ROW_PITCH];
    auto store_sixteen = [&](int buffer, int column, const uint32_t (&pairs)[8]) __attribute__((always_inline)) {
        uint8_t * const row = tile_row + buffer * sizeof(wb[0]);
        *reinterpret_cast<uint4 *>(row + tile_granule(n, column / 8) * 16) = make_uint4(pairs[0], pairs[1], pairs[2], pairs[3]);
        *reinterpret_cast<uint4 *>(row + tile_granule(n, column / 8 + 1) * 16) = make_uint4(pairs[4], pairs[5], pairs[6], pairs[7]);
    };
    auto decode = [&](int step, int buffer) __attribute__((always_inline)) {
        const int n0 = (step >= steps_per_source ? step - steps_per_source : step) * BWD_NS;
        uint32_t keep = n0 + wave * BSH_ROWS_PER_WAVE + n < n_total ? 0xffffffffu : 0u;
        asm volatile("" : "+v"(keep));   // (a mask, not a branch around part of the arithmetic)
        const uint8_t * const blk = raw + n * RAW_PITCH;
        if constexpr (K45) {
            // 16 bytes of nibbles: 16 values of group 2 chunk of the half block and 16 of the next one
            const int chunk = (lane >> 1) & 1, part = lane & 1;
            const uint4 header = *reinterpret_cast<const uint4 *>(blk);
            const uint4 nibbles = *reinterpret_cast<const uint4 *>(blk + (TYPE == Q4_K ? 16 : 48) + 32 * chunk + 16 * part);
            const uint4 planes = TYPE == Q5_K ? *reinterpret_cast<const uint4 *>(blk + 16 + 16 * part) : uint4{0, 0, 0, 0};
            const uint32_t word[4] = {nibbles.x, nibbles.y, nibbles.z, nibbles.w}, plane[4] = {planes.x, planes.y, planes.z, planes.w};
            const uint32_t first = header.y >> (16 * chunk), second = header.z >> (16 * chunk), third = header.w >> (16 * chunk);
            // groups 0 .. 3 of the super-block: plain 6-bit fields; 4 .. 7: nibbles of the third word, their top bits above the first four's
            const uint32_t scales = half_block == 0 ? first & 0x3f3fu : (third & 0x0f0fu) | ((first >> 2) & 0x3030u);
            const uint32_t minima = half_block == 0 ? second & 0x3f3fu : ((third >> 4) & 0x0f0fu) | ((second >> 2) & 0x3030u);
            const uint32_t d_dmin = header.x & keep;
            const float d = half_bits_to_float(d_dmin & 0xffffu), dmin = half_bits_to_float(d_dmin >> 16);
#pragma unroll
            for (int high = 0; high < 2; ++high) {
                const float scale = d * static_cast<float>((scales >> (8 * high)) & 0xffu);
                const float minimum = dmin * static_cast<float>((minima >> (8 * high)) & 0xffu);
                uint32_t pairs[8];
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    uint32_t q = (word[w] >> (4 * high)) & 0x0f0f0f0fu;
                    if constexpr (TYPE == Q5_K) {
                        q |= ((plane[w] >> (4 * half_block + 2 * chunk + high)) & 0x01010101u) << 4;
                    }
                    float value[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        value[e] = scale * static_cast<float>((q >> (8 * e)) & 0xffu) - minimum;
                    }
                    pairs[2 * w] = pack_bf16x2(value[0], value[1]);
                    pairs[2 * w + 1] = pack_bf16x2(value[2], value[3]);
                }
                store_sixteen(buffer, 64 * chunk + 32 * high + 16 * part, pairs);
            }
        } else if constexpr (TYPE == IQ2_S) {
            // a block of 32 values: codebook magnitudes with their signs applied, four bytes at a time, above their true values by 128 (as in the
            // role-split kernel; exact before its rounding)
            const int quarter = lane & 3, block = 4 * half_block + quarter;
            const uint32_t indices = lds_u32(blk + 4 * quarter), signs = lds_u32(blk + 16 + 4 * quarter);
            const uint32_t upper = blk[32 + block], scales = blk[40 + block];
            const float d = half_bits_to_float(lds_u16(blk + 48) & keep);
#pragma unroll
            for (int run = 0; run < 2; ++run) {
                const float scale = d * 0.125f * static_cast<float>(((scales >> (4 * run)) & 15u) * 2 + 1);
                const float offset = scale * 128.0f;
                uint32_t pairs[8];
#pragma unroll
                for (int o = 0; o < 2; ++o) {
                    const int octet = 2 * run + o;
                    const uint2 entry = grid[((indices >> (8 * octet)) & 0xffu) | (((upper >> (2 * octet)) & 3u) << 8)];
#pragma unroll
                    for (int w = 0; w < 2; ++w) {
                        // the four signs spread to a bit per byte; a negative magnitude is its complement plus one
                        const uint32_t negative = (((signs >> (8 * octet + 4 * w)) & 15u) * 0x00204081u) & 0x01010101u;
                        const uint32_t q = (((w == 0 ? entry.x : entry.y) ^ (negative * 0xffu)) + negative) ^ 0x80808080u;
                        float value[4];
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            value[e] = scale * static_cast<float>((q >> (8 * e)) & 0xffu) - offset;
                        }
                        pairs[4 * o + 2 * w] = pack_bf16x2(value[0], value[1]);
                        pairs[4 * o + 2 * w + 1] = pack_bf16x2(value[2], value[3]);
                    }
                }
                store_sixteen(buffer, 32 * quarter + 16 * run, pairs);
            }
        } else {
            // two runs of 16 values that share their bytes, four quants at a time, above their true values by the bias
            const int quarter = lane & 3, part = quarter & 1, upper = quarter >> 1;
            const uint4 low_bits = *reinterpret_cast<const uint4 *>(TYPE == Q6_K ? blk + 16 * quarter : blk + 32 + 16 * part);
            const uint4 high_bits = *reinterpret_cast<const uint4 *>(TYPE == Q6_K ? blk + 64 + 16 * part : blk + 16 * part);
            const uint32_t low[4] = {low_bits.x, low_bits.y, low_bits.z, low_bits.w}, high[4] = {high_bits.x, high_bits.y, high_bits.z, high_bits.w};
            const float d = half_bits_to_float(lds_u16(blk + (TYPE == Q6_K ? 126 : 78)) & keep);
#pragma unroll
            for (int run = 0; run < 2; ++run) {
                int sub, column;
                if constexpr (TYPE == Q6_K) {
                    sub = static_cast<int8_t>(blk[96 + 8 * half_block + quarter + 4 * run]);
                    column = 64 * run + 16 * quarter;
                } else {
                    const uint32_t nibble = blk[66 + 4 * upper + 2 * run + part] >> (4 * half_block);
                    const uint32_t top = blk[74 + 2 * run + part] >> (4 * half_block + 2 * upper);
                    sub = static_cast<int>((nibble & 15u) | ((top & 3u) << 4)) - 32;
                    column = 64 * upper + 32 * run + 16 * part;
                }
                const float scale = d * static_cast<float>(sub);
                const float offset = scale * (TYPE == Q6_K ? 32.0f : 4.0f);
                uint32_t pairs[8];
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    uint32_t q;
                    if constexpr (TYPE == Q6_K) {
                        q = ((low[w] >> (4 * run)) & 0x0f0f0f0fu) | (((high[w] >> (2 * upper + 4 * run)) & 0x03030303u) << 4);
                    } else {
                        const int group = 2 * upper + run;   // 32-value group of the half block
                        q = ((low[w] >> (2 * group)) & 0x03030303u) | (((high[w] >> (4 * half_block + group)) & 0x01010101u) << 2);
                    }
                    float value[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        value[e] = scale * static_cast<float>((q >> (8 * e)) & 0xffu) - offset;
                    }
                    pairs[2 * w] = pack_bf16x2(value[0], value[1]);
                    pairs[2 * w + 1] = pack_bf16x2(value[2], value[3]);
                }
                store_sixteen(buffer, column, pairs);
            }
        }
    };

    // cotangent fragments of the task's (up to) two 32-row tiles; one set, requested right after the
    // multiplications that used the previous one and awaited a whole decode later
    // (offsets from the 32-row tile that the task starts in: it reaches into two more at most)
    const int first_tile = row_start >> 5;
    const int64_t task_offset = static_cast<int64_t>(first_tile) * a.n_chunks * 1024;
    uint32_t lane_offset[2];
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
        int r = row_start + rt * 32 + l32;
        r = r < a.rows_padded ? r : a.rows_padded - 1;
        lane_offset[rt] = static_cast<uint32_t>((r >> 5) - first_tile) * a.n_chunks * 1024 + ((r & 31) + 32 * half) * 16;
    }
    u32x4 cot[2][4] = {};
    auto request_cotangent = [&](int step) __attribute__((always_inline)) {
        step = min(step, last);
        const int source = step >= steps_per_source ? 1 : 0;
        const int n0 = (step - source * steps_per_source) * BWD_NS;
        // (the packed cotangent is zero padded to whole steps of 64 columns)
        const uint8_t * base = (source == 0 ? a.cotangent[0] : a.cotangent[1]) + task_offset + static_cast<int64_t>(n0 >> 4) * 1024;
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
            if (rt < row_tiles) {
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    cot[rt][c] = *reinterpret_cast<const u32x4 *>(base + lane_offset[rt] + c * 1024);
                }
            }
        }
    };
    v16f acc[2];
#pragma unroll
    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[rt][v] = 0.0f;
    const uint8_t * const tr_from = &wb[0][transposed_offset(lane, wave)];   // the wave's 32 columns
    auto multiply = [&](int buffer) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const uint8_t * const from = tr_from + buffer * sizeof(wb[0]) + 16 * c * BWD_ROW_PITCH;
            const v8bf bfrag = transposed_fragment(from, from + 4 * BWD_ROW_PITCH);
#pragma unroll
            for (int rt = 0; rt < 2; ++rt) {
                if (rt < row_tiles) {
                    acc[rt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, cot[rt][c]), bfrag, acc[rt], 0, 0, 0);
                }
            }
        }
    };

    InFlight ring[BSH_DEPTH];
#pragma unroll
    for (int d = 0; d < BSH_DEPTH; ++d) {
        request(d, ring[d]);
    }
    request_cotangent(0);
    park(ring[0]);
    request(BSH_DEPTH, ring[0]);
    wave_sync();
    decode(0, 0);
    __syncthreads();
    // A step that has a successor: multiply its tile and prepare the next one.  The loop below holds no branch, so
    // the compiler's wait-count bookkeeping sees every request on every path; with the last step's exceptions inside
    // it, the paths that skip a wait made it wait for the newest requests before the matrix instructions (a whole
    // memory round trip per step).
    static_assert(BSH_DEPTH == 2, "tile and ring parity follow the position in the unrolled round");
    auto advance = [&](int step, auto parity_tag) __attribute__((always_inline)) {
        constexpr int u = decltype(parity_tag)::value;
        // (this wave's decode of the current step, the last reader of its slot, is behind it in program order)
        // the chain of dependent waits goes first, the arithmetic of the decode fills in (measured: 1 %)
        __builtin_amdgcn_s_setprio(3);
        park(ring[u ^ 1]);
        multiply(u);
        // both requests go out behind the matrix instructions, which wait for the previous step's cotangent only
        request_cotangent(step + 1);
        request(step + 1 + BSH_DEPTH, ring[u ^ 1]);
        wave_sync();
        __builtin_amdgcn_s_setprio(0);
        decode(step + 1, u ^ 1);
        __syncthreads();
    };
    int step = 0;
#pragma unroll 1
    for (; step + 2 <= last; step += 2) {
        advance(step, std::integral_constant<int, 0>{});
        advance(step + 1, std::integral_constant<int, 1>{});
    }
    if (step < last) {   // uniform
        advance(step, std::integral_constant<int, 0>{});
        multiply(1);
    } else {
        multiply(0);
    }
    __syncthreads();
    // the tiles are free (every wave is past its last multiplication): the four 32-column slices of a 32-row tile
    // meet in LDS and leave as whole 256-byte rows
    constexpr int STAGE_PITCH = BWD_TK + 8;
    static_assert(2 * 32 * STAGE_PITCH * 2 <= sizeof(wb), "both row tiles fit the weight tiles");
    static_assert(BSH_DEPTH % 2 == 0, "tile parity follows the position in the unrolled round");
    uint16_t * stage = reinterpret_cast<uint16_t *>(&wb[0][0]);
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
        if (rt < row_tiles) {
            stage_tile_32x32<STAGE_PITCH>(stage + rt * 32 * STAGE_PITCH, acc[rt], wave * 32, lane);
        }
    }
    __syncthreads();
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
        const int r0 = row_start + rt * 32;
        if (rt < row_tiles) {
            store_staged_rows<STAGE_PITCH>(stage + rt * 32 * STAGE_PITCH,
                                           a.dx + static_cast<int64_t>(r0) * a.in_features + k_tile * BWD_TK,
                                           a.in_features, row_end - r0, BWD_TK, tid, BSH_THREADS);
        }
    }
}

// dx[i] = bf16(partial[0][i] + partial[1][i] + ...), eight values per thread; `count` is a multiple of 8.
__global__ __launch_bounds__(256) void reduce_partials_kernel(const float * __restrict__ partial,
                                                              uint16_t * __restrict__ dx, int64_t count, int n_splits) {
    const int64_t first = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * 8;
    if (first >= count) {
        return;
    }
    float sum[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) sum[e] = 0.0f;
    for (int s = 0; s < n_splits; ++s) {
        const float4 lo = *reinterpret_cast<const float4 *>(partial + s * count + first);
        const float4 hi = *reinterpret_cast<const float4 *>(partial + s * count + first + 4);
        sum[0] += lo.x; sum[1] += lo.y; sum[2] += lo.z; sum[3] += lo.w;
        sum[4] += hi.x; sum[5] += hi.y; sum[6] += hi.z; sum[7] += hi.w;
    }
    *reinterpret_cast<uint4 *>(dx + first) = make_uint4(pack_bf16x2(sum[0], sum[1]), pack_bf16x2(sum[2], sum[3]),
                                                        pack_bf16x2(sum[4], sum[5]), pack_bf16x2(sum[6], sum[7]));
}

template <int TYPE>
static hipError_t launch_backward_typed(const BackwardArgs & args, hipStream_t stream) {
    const int64_t total = xcd_slots(static_cast<int64_t>(args.k_tiles) * (args.task_count != nullptr ? xcd_chunk_slots(args.task_slots) : args.task_slots));
    const int64_t total_short = xcd_slots(static_cast<int64_t>(args.k_tiles) * args.short_slots);
    if (total <= 0 || total > 0x7fffffffLL || total_short > 0x7fffffffLL) {
        return hipErrorInvalidValue;
    }
    const ProfileScope scope(3, stream);
    // the general kernel, with the packed blocks fetched as wide units where the format needs that and the weights allow it
    const auto general = [&](dim3 grid, const BackwardArgs & launch_args) {
        if constexpr (Format<TYPE>::BLOCK_BYTES % 16 != 0) {
            const int64_t weight_bytes = static_cast<int64_t>(args.out_features) * args.row_bytes;
            // (and the rows short enough for the 24-bit multiplies of the unit offsets)
            if (args.row_bytes < (1 << 24) && wide_stage_ok(args.packed[0], weight_bytes) &&
                (args.packed[1] == nullptr || wide_stage_ok(args.packed[1], weight_bytes))) {
                mmq_grad_input_kernel<TYPE, true><<<grid, BWD_THREADS, 0, stream>>>(launch_args);
                return;
            }
        }
        mmq_grad_input_kernel<TYPE, false><<<grid, BWD_THREADS, 0, stream>>>(launch_args);
    };
    // (32-bit lane offsets into a step's weight rows, in both kernels below; in_features ends far below)
    if (args.row_bytes * 2 * BWD_NS >= (int64_t{1} << 32)) {
        return hipErrorInvalidValue;
    }
    if (args.segment == 1) {
        // (32-bit lane offsets into the three row tiles that a task may touch)
        if (int64_t{3} * args.n_chunks * 1024 >= (int64_t{1} << 32)) {
            // twenty million weight rows and more: all tasks in one launch of the general kernel
            BackwardArgs all_args = args;
            all_args.segment = 0;
            general(dim3(static_cast<unsigned>(total)), all_args);
            return hipGetLastError();
        }
        // grouped call: the short tasks (a separate segment of the task list) run in a launch of their own
        BackwardArgs short_args = args;
        short_args.segment = 2;
        mmq_grad_input_short_kernel<TYPE><<<static_cast<unsigned>(total_short), BSH_THREADS, 0, stream>>>(short_args);
        const hipError_t status = hipGetLastError();
        if (status != hipSuccess) {
            return status;
        }
    }
    // the role-split kernel addresses the packed cotangent with 32-bit lane offsets
    const bool role_split = cotangent_workspace_bytes(args.rows, args.out_features) < (int64_t{1} << 32);
    const bool splits = args.n_splits > 1;
    if (role_split) {
        // one persistent workgroup per CU, more only when a workgroup's item table would overflow
        const int tasks = (args.rows + BWD_TR - 1) / BWD_TR;
        const int64_t items = splits ? (static_cast<int64_t>(args.k_tiles / 2) * tasks * args.n_splits + XCDS - 1) / XCDS * XCDS * 2 : total;
        const int64_t needed = (items + BSP_MAX_ITEMS - 1) / BSP_MAX_ITEMS;
        const int64_t grid = (std::max<int64_t>(std::min<int64_t>(items, BSP_GRID), needed) + XCDS - 1) / XCDS * XCDS;
        mmq_grad_input_split_kernel<TYPE><<<static_cast<unsigned>(grid), BSP_THREADS, 0, stream>>>(args, static_cast<int>(items));
    } else {
        general(dim3(static_cast<unsigned>(total), static_cast<unsigned>(args.n_splits)), args);
    }
    if (splits) {
        const int64_t count = static_cast<int64_t>(args.rows) * args.in_features;
        reduce_partials_kernel<<<static_cast<unsigned>((count / 8 + 255) / 256), 256, 0, stream>>>(
            args.partial, args.dx, count, args.n_splits);
    }
    return hipGetLastError();
}

hipError_t launch_mmq_grad_input(const uint8_t * cotangent_first, const uint8_t * cotangent_second,
                                 const uint8_t * packed_first, const uint8_t * packed_second,
                                 int64_t bytes_per_expert, uint16_t * grad_input, const TaskList * tasks,
                                 int rows, int out_features, int in_features, int quant_type,
                                 hipStream_t stream, float * partial) {
    BackwardArgs args;
    // `partial` (dense calls only): room for dense_grad_splits() fp32 copies of the result, or nullptr
    args.partial = partial;
    args.n_splits = tasks == nullptr && partial != nullptr
        ? dense_grad_splits(rows, out_features, in_features) : 1;
    args.cotangent[0] = cotangent_first;
    args.cotangent[1] = cotangent_second;
    args.packed[0] = packed_first;
    args.packed[1] = packed_second;
    args.sources = packed_second != nullptr ? 2 : 1;
    args.bytes_per_expert = bytes_per_expert;
    args.row_bytes = static_cast<int64_t>(in_features / QK_K) * block_bytes(quant_type);
    args.dx = grad_input;
    args.rows = rows;
    args.rows_padded = static_cast<int>(pad_rows(rows));
    args.out_features = out_features;
    args.n_chunks = cotangent_chunks(out_features);
    args.in_features = in_features;
    args.k_tiles = in_features / BWD_TK;
    if (tasks != nullptr) {
        args.task_count = tasks->count;
        args.task_early = tasks->early;
        args.task_expert = tasks->expert;
        args.task_row_start = tasks->row_start;
        args.task_row_end = tasks->row_end;
        args.task_slots = tasks->max_tasks;
        // max_tasks = full row tiles + one remainder per group: the remainders are all that can be short
        args.short_slots = tasks->max_tasks - (rows + BWD_TR - 1) / BWD_TR;
        args.segment = 1;
    } else {
        args.task_count = nullptr;
        args.task_early = nullptr;
        args.short_slots = 0;
        args.segment = 0;
        args.task_expert = nullptr;
        args.task_row_start = nullptr;
        args.task_row_end = nullptr;
        args.task_slots = (rows + BWD_TR - 1) / BWD_TR;
    }
    switch (quant_type) {
        case Q3_K: return launch_backward_typed<Q3_K>(args, stream);
        case Q4_K: return launch_backward_typed<Q4_K>(args, stream);
        case Q5_K: return launch_backward_typed<Q5_K>(args, stream);
        case Q6_K: return launch_backward_typed<Q6_K>(args, stream);
        case IQ2_S: return launch_backward_typed<IQ2_S>(args, stream);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace tgo
