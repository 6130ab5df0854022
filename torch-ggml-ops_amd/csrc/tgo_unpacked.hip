// Dense products whose weights are unpacked once per call.
//
// The other matrix-core kernels unpack a column tile's weights again for every tile of 128 or 256 rows, in the workgroup that multiplies
// with them: they are bound by that unpacking where a call has few tiles (a workgroup takes microseconds per super-block, however few rows
// it has) and share issue slots and LDS with it where it has many.  Here one launch writes both operands to memory in the order in which
// the matrix instructions want them (slabs of 1 KiB: 32 rows x 16 values of the reduction, [half][row 0..31][8 values]), and a second
// one is a plain matrix product of slabs.  The unpacked weights cost 2 bytes each, written once and read from the caches.
//
// The operands are those of the other kernels, value for value, and they meet in the same order.
#include <algorithm>
#include <type_traits>

#include "tgo_cotangent.h"
#include "tgo_device.h"
#include "tgo_launch.h"
#include "tgo_scaled_operand.h"

namespace tgo {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

constexpr int UNP_SOURCES = UNPACKED_SOURCES;   // projections of one product

// ---- operands of the grad-input ---------------------------------------------------------------------------------
// Workgroups 0 .. unpack_blocks - 1 turn 32 weight rows x SPAN super-blocks each into slabs of 32 K columns x 16 weight rows (the
// reduction runs over the weight rows): decoded once to bf16 into LDS, read back two K columns by eight weight rows per thread.  The
// others pack the cotangent.  Bound by memory: 4096 x 2048 Q4_K with a cotangent of 4096 rows to pack 16 us (88 MB, 5.5 TB/s), 28672 x 8192
// alone 130 us (602 MB, 4.6 TB/s).
struct GradOperandSource {
    const uint8_t * packed;
    uint8_t * weights;      // slabs [K / 32][row_chunks], this source's first chunk
    const uint16_t * grad;  // nullptr: nothing to pack
    uint8_t * cotangent;    // slabs [rows / 32][row_chunks], this source's first chunk
    int out_features;
    int n_chunks;           // of this source: 16 weight rows each, whole steps of 64 rows if the cotangent is packed, else of 32
    int unpack_blocks;      // n_chunks / 2 x span_blocks
    int pack_columns;       // workgroups side by side along N that pack
    int first_block;        // of the launch
};
struct GradOperandArgs {
    GradOperandSource source[UNP_SOURCES];   // of one format
    int count;
    int64_t row_bytes;
    int in_features, rows;
    int row_chunks;         // of all sources of the product together
    int span_blocks;        // workgroups side by side along K
};
constexpr int UNT_ROWS = 32;
constexpr int UNT_PITCH = QK_K * 2 + 16;   // bytes of a weight row's bf16 in LDS

template <int TYPE, bool WIDE>
__global__ __launch_bounds__(256) void grad_operands_kernel(const GradOperandArgs args) {
    using F = Format<TYPE>;
    using W = WideStage<TYPE>;
    constexpr int SPAN = TYPE == IQ2_S ? 4 : 1;   // (a workgroup of IQ2_S expands its codebook first)
    constexpr int SLOT_PITCH = WIDE ? W::PITCH : F::RAW_PITCH;
    constexpr int SLOT_FRONT = WIDE ? W::FRONT : F::RAW_SHIFT;
    constexpr int RAW_BYTES = (UNT_ROWS * SLOT_PITCH + 15) / 16 * 16;
    constexpr int REGS = WIDE ? W::template regs<UNT_ROWS, 256>() : 1;
    __shared__ __attribute__((aligned(16))) uint8_t shared[RAW_BYTES + UNT_ROWS * UNT_PITCH];
    __shared__ std::conditional_t<TYPE == IQ2_S, Iq2sSelectors, uint2> codebook;
    static_assert(sizeof(shared) >= PACK_TILE_BYTES, "the packing workgroups' tile fits");
    const int tid = threadIdx.x;
    int index = 0;
#pragma unroll
    for (int i = 1; i < UNP_SOURCES; ++i) {
        index = i < args.count && static_cast<int>(blockIdx.x) >= args.source[i].first_block ? i : index;
    }
    const GradOperandSource a = args.source[index];
    int block = static_cast<int>(blockIdx.x) - a.first_block;
    if (block >= a.unpack_blocks) {
        block -= a.unpack_blocks;
        const int row_tile = block / a.pack_columns;
        pack_cotangent_tile(shared, a.grad, a.cotangent, row_tile, (block - row_tile * a.pack_columns) * 8, args.rows, a.out_features,
                            a.n_chunks, args.row_chunks, nullptr, nullptr, 0, tid);
        return;
    }
    if constexpr (TYPE == IQ2_S) {
        expand_iq2s_selectors(codebook, tid, 256);
    }
    uint8_t * const raw = shared;
    uint8_t * const tile = shared + RAW_BYTES;
    const int row_block = block / args.span_blocks;
    const int kb0 = (block - row_block * args.span_blocks) * SPAN;
    const int kb_end = min(kb0 + SPAN, args.in_features / QK_K);
    const int n0 = row_block * UNT_ROWS;
    // (the weight rows that fill up the last step of 64 are zeros; their workgroups read the last row)
    const int first_row = min(n0, a.out_features - 1);
    const int rows_valid = min(UNT_ROWS, a.out_features - first_row);
    const uint8_t * const rows = a.packed + static_cast<int64_t>(first_row) * args.row_bytes;
    WideRegs<REGS> regs;
    if constexpr (WIDE) {
        wide_fetch<TYPE, UNT_ROWS, 256, REGS>(regs, rows, static_cast<int>(args.row_bytes), rows_valid, kb0, tid);
    }
    for (int kb = kb0; kb < kb_end; ++kb) {
        if constexpr (WIDE) {
            wide_park<TYPE, UNT_ROWS, 256, REGS>(raw, regs, rows, static_cast<int>(args.row_bytes), rows_valid, kb, tid);
            if (kb + 1 < kb_end) {
                wide_fetch<TYPE, UNT_ROWS, 256, REGS>(regs, rows, static_cast<int>(args.row_bytes), rows_valid, kb + 1, tid);
            }
        } else {
            stage_blocks<TYPE>(raw, a.packed, args.row_bytes, first_row, a.out_features, kb, UNT_ROWS, tid, 256);
        }
        __syncthreads();
#pragma unroll
        for (int pass = 0; pass < 2; ++pass) {
            const int row = (tid >> 4) + 16 * pass, unit = tid & 15;
            uint32_t pairs[8];
            decode16_bf16<TYPE>(raw + row * SLOT_PITCH + SLOT_FRONT, unit, &codebook, pairs);
            const bool inside = n0 + row < a.out_features;
            uint4 * const dst = reinterpret_cast<uint4 *>(tile + row * UNT_PITCH + unit * 32);
            dst[0] = inside ? make_uint4(pairs[0], pairs[1], pairs[2], pairs[3]) : make_uint4(0, 0, 0, 0);
            dst[1] = inside ? make_uint4(pairs[4], pairs[5], pairs[6], pairs[7]) : make_uint4(0, 0, 0, 0);
        }
        __syncthreads();
        const int column = 2 * (tid & 127);   // of the super-block; this thread: it and the next
#pragma unroll
        for (int pass = 0; pass < 2; ++pass) {
            const int octet = 2 * pass + (tid >> 7);   // eight weight rows of the 32
            uint32_t word[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                word[i] = lds_u32(tile + (8 * octet + i) * UNT_PITCH + column * 2);
            }
            uint32_t even[4], odd[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                even[i] = __builtin_amdgcn_perm(word[2 * i + 1], word[2 * i], 0x05040100u);
                odd[i] = __builtin_amdgcn_perm(word[2 * i + 1], word[2 * i], 0x07060302u);
            }
            const int64_t slab = static_cast<int64_t>(kb * 8 + (column >> 5)) * args.row_chunks + row_block * 2 + (octet >> 1);
            uint4 * const dst = reinterpret_cast<uint4 *>(a.weights + slab * 1024 + (octet & 1) * 512 + (column & 31) * 16);
            dst[0] = make_uint4(even[0], even[1], even[2], even[3]);
            dst[1] = make_uint4(odd[0], odd[1], odd[2], odd[3]);
        }
    }
}

// ---- the product -----------------------------------------------------------------------------------------------
// y[r, c] = sum over the steps of w[c] . x[r], both in slabs [tile of 32][step].
// Slabs go from memory to LDS directly (global_load_lds: a slab is one instruction of a wave and lands in the order in which the matrix
// instructions read it), UNP_RING - 1 stages of two steps ahead; every wave requests its share of a stage, waits for its own requests of the
// next one and meets the others at a barrier, once per stage.  Fragments are read from LDS a step ahead.
// Bound: LDS.  A step of a 64 x 64 wave tile is 4 fragment reads to 4 matrix instructions, and with the stage's arrival the LDS is busy
// 1.5 times as long as the matrix pipe; 64 x 128 tiles of eight waves 0.9 times.  Of operands in slabs, 4096 x 4096 x 2048: 256 x 256 tiles 68 us
// (1009 TFLOP/s), 128 x 128 72; 4096 x 2048 x 4096: 128 x 256 66 us, 256 x 256 (half of the CUs) 98; 1000 x 4096 x 4096: 128 x 128 38 us, 128 x 256 42.
constexpr int UNP_RING = 4;
struct ProductArgs {
    const uint8_t * w;       // slabs [w_tiles][steps]
    const uint8_t * x;       // slabs [x_tiles][steps], or row-major sources side by side along the reduction (ROW_MAJOR)
    int steps;               // even
    int sources;
    const uint8_t * x_source[UNP_SOURCES];
    int x_first_stage[UNP_SOURCES];   // of two steps, 32 values
    int x_stride[UNP_SOURCES];        // bytes from row to row
    int w_tiles, x_tiles;    // of 32
    int w_blocks, x_blocks;  // workgroups along either
    int rows;
    int outputs;
    uint16_t * y[UNP_SOURCES];
    int first_tile[UNP_SOURCES];   // tile of w at which an output's columns start
    int columns[UNP_SOURCES];      // and how many there are: the stride of its rows
};

// 32-bit address of an LDS object
TGO_DEVICE uint32_t lds_address(const void * p) {
    return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) uint8_t *)p));
}

// A wave's tile is MT x 32 rows by NT x 32 columns, the workgroup's WM x WN of those.
// ROW_MAJOR: x are rows as they stand (bf16, whole stages of 32 values, 16-byte aligned).  The lanes of a request then take 64 bytes
// from each of 16 rows, which land row by row; the 16-byte pieces of a row are exchanged by (row / 2) % 4 on the way, so that the eight
// lanes that the LDS serves together (eight rows, the same piece) find theirs on different banks.  That spares the pass that would
// write the rows as slabs (4096 rows x 4096: 67 MB moved, 12 us).
template <bool BF16, bool ROW_MAJOR, int MT, int NT, int WM, int WN>
__global__ __launch_bounds__(64 * WM * WN, 2) void fragment_product_kernel(const ProductArgs a) {
    constexpr int SS = 2;                              // steps per stage
    constexpr int W_TILES = NT * WN, X_TILES = MT * WM;
    constexpr int SLABS = (W_TILES + X_TILES) * SS;    // of a stage: [tile][step], the weights' tiles first
    constexpr int WAVES = WM * WN;
    constexpr int PER = SLABS / WAVES;                 // requested by each wave
    constexpr int STAGE = SLABS * 1024;
    static_assert(SLABS % WAVES == 0, "every wave requests as many slabs");
    __shared__ __attribute__((aligned(1024))) uint8_t ring[UNP_RING * STAGE];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // Every XCD takes a contiguous share of the tiles, in bands of eight row tiles: its L2 then serves a near-square piece of the result.
    const int total = a.w_blocks * a.x_blocks;
    const int per_xcd = (total + XCDS - 1) / XCDS;
    const int id = static_cast<int>(blockIdx.x % XCDS) * per_xcd + static_cast<int>(blockIdx.x / XCDS);
    if (static_cast<int>(blockIdx.x / XCDS) >= per_xcd || id >= total) {
        return;
    }
    constexpr int BAND = 8;
    const int band = id / (BAND * a.w_blocks);
    const int band_rows = min(BAND, a.x_blocks - band * BAND);
    const int in_band = id - band * BAND * a.w_blocks;
    const int x_block = band * BAND + in_band % band_rows;
    const int w_block = in_band / band_rows;
    const int stages = a.steps / SS;

    // (tiles past the last one repeat it; nothing of what they give is stored)
    // W_PER of a wave's requests are slabs of the weights, the others the rows' share.
    constexpr int W_PER = W_TILES * SS / WAVES, X_PER = PER - W_PER;
    static_assert(W_TILES * SS % WAVES == 0, "every wave requests as many slabs of either kind");
    const uint8_t * w_source[W_PER];
    const uint8_t * x_source[X_PER];
    uint32_t x_lane[X_PER];
#pragma unroll
    for (int i = 0; i < W_PER; ++i) {
        const int slab = wave * W_PER + i;
        const int t = min(w_block * W_TILES + slab / SS, a.w_tiles - 1);
        w_source[i] = a.w + (static_cast<int64_t>(t) * a.steps + slab % SS) * 1024;
    }
    const uint32_t ring_address = lds_address(ring);
    const uint32_t lane16 = lane * 16;
    int x_left = 0;   // ROW_MAJOR: stages until the next source begins
    int x_next = 0;   // and which one that is
    auto open_source = [&](int index, int stage) __attribute__((always_inline)) {
        const int stride = a.x_stride[index];
#pragma unroll
        for (int i = 0; i < X_PER; ++i) {
            const int slab = wave * X_PER + i;
            const int row0 = (x_block * X_TILES + slab / SS) * 32 + 16 * (slab % SS);
            const int row = lane >> 2;
            const int piece = (lane & 3) ^ ((row >> 1) & 3);
            const int first = min(row0, a.rows - 1);   // (rows past the last one repeat it)
            x_source[i] = a.x_source[index] + static_cast<int64_t>(first) * stride + static_cast<int64_t>(stage - a.x_first_stage[index]) * (SS * 32);
            x_lane[i] = static_cast<uint32_t>(min(row, a.rows - 1 - first)) * static_cast<uint32_t>(stride) + piece * 16;
        }
        x_next = index + 1;
        x_left = (x_next < a.sources ? a.x_first_stage[x_next] : stages) - stage;
    };
    if constexpr (ROW_MAJOR) {
        open_source(0, 0);
    } else {
#pragma unroll
        for (int i = 0; i < X_PER; ++i) {
            const int slab = wave * X_PER + i;
            const int t = min(x_block * X_TILES + slab / SS, a.x_tiles - 1);
            x_source[i] = a.x + (static_cast<int64_t>(t) * a.steps + slab % SS) * 1024;
            x_lane[i] = lane16;
        }
    }
    // Requests the next stage; past the last one, that one again, into a buffer that nobody reads any more.
    int requested = 0;
    auto request = [&](int buffer) __attribute__((always_inline)) {
        const uint32_t to = ring_address + buffer * STAGE;
#pragma unroll
        for (int i = 0; i < W_PER; ++i) {
            asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(to + (wave * W_PER + i) * 1024), "v"(lane16), "s"(w_source[i])
                         : "memory");
        }
#pragma unroll
        for (int i = 0; i < X_PER; ++i) {
            asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(to + (W_TILES * SS + wave * X_PER + i) * 1024), "v"(x_lane[i]),
                         "s"(x_source[i])
                         : "memory");
        }
        if (++requested < stages) {
#pragma unroll
            for (int i = 0; i < W_PER; ++i) w_source[i] += SS * 1024;
#pragma unroll
            for (int i = 0; i < X_PER; ++i) x_source[i] += ROW_MAJOR ? SS * 32 : SS * 1024;
            if constexpr (ROW_MAJOR) {
                if (--x_left == 0 && x_next < a.sources) {
                    open_source(x_next, requested);
                }
            }
        }
    };
    // The wave's requests are complete but for those of the two youngest stages, its reads are done, and so are the others'.
    auto meet = [&]() __attribute__((always_inline)) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((UNP_RING - 2) * PER) : "memory");
    };
    const int wm = wave % WM, wn = wave / WM;
    // ROW_MAJOR: where the lane's piece of step 0 lies in a row tile
    const int x_piece = (lane & 31) * 64 + (((lane >> 5) ^ ((lane >> 1) & 3)) * 16);
    v16f acc[NT][MT];
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[n][m] = v16f{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    uint4 w[2][NT], x[2][MT];
    auto read_step = [&](int buffer, int step, int slot) __attribute__((always_inline)) {
        const uint8_t * const base = ring + buffer * STAGE + lane16;
#pragma unroll
        for (int n = 0; n < NT; ++n) w[slot][n] = *reinterpret_cast<const uint4 *>(base + ((wn * NT + n) * SS + step) * 1024);
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const uint8_t * const tile = ring + buffer * STAGE + (W_TILES + wm * MT + m) * (SS * 1024);
            x[slot][m] = *reinterpret_cast<const uint4 *>(ROW_MAJOR ? tile + (x_piece ^ (32 * step)) : tile + step * 1024 + lane16);
        }
    };
    auto multiply = [&](int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < NT; ++n) {
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                if constexpr (BF16) {
                    acc[n][m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, w[slot][n]), __builtin_bit_cast(v8bf, x[slot][m]),
                                                                        acc[n][m], 0, 0, 0);
                } else {
                    acc[n][m] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, w[slot][n]), __builtin_bit_cast(half8_t, x[slot][m]),
                                                                       acc[n][m], 0, 0, 0);
                }
            }
        }
    };
#pragma unroll
    for (int s = 0; s < UNP_RING - 1; ++s) request(s);
    meet();
    read_step(0, 0, 0);
    int buffer = 0, free_buffer = UNP_RING - 1;
#pragma unroll 1
    for (int s = 0; s < stages; ++s) {
        // the buffer of stage s - 1: all waves have read it before they last met
        request(free_buffer);
        read_step(buffer, 1, 1);
        multiply(0);
        __builtin_amdgcn_sched_barrier(0);
        const int next = buffer + 1 == UNP_RING ? 0 : buffer + 1;
        meet();
        read_step(next, 0, 0);
        multiply(1);
        __builtin_amdgcn_sched_barrier(0);
        free_buffer = buffer;
        buffer = next;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (nothing may arrive in the LDS of a workgroup that has ended)

    const int l32 = lane & 31, half = lane >> 5;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        const int tile = w_block * W_TILES + wn * NT + n;
        int output = 0;
#pragma unroll
        for (int i = 1; i < UNP_SOURCES; ++i) {
            output = i < a.outputs && tile >= a.first_tile[i] ? i : output;
        }
        const int c0 = (tile - a.first_tile[output]) * 32;
        const int columns = a.columns[output];
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const int r0 = (x_block * X_TILES + wm * MT + m) * 32;
            if (r0 >= a.rows || c0 >= columns) {   // uniform
                continue;
            }
            store_rows_32xn<1>(&acc[n][m], a.y[output] + static_cast<int64_t>(r0) * columns + c0, columns, a.rows - r0, columns - c0, lane);
        }
    }
}

template <bool BF16, bool ROW_MAJOR, int MT, int NT, int WM, int WN>
static hipError_t launch_product_tiled(ProductArgs args, hipStream_t stream) {
    args.w_blocks = (args.w_tiles + NT * WN - 1) / (NT * WN);
    args.x_blocks = (args.x_tiles + MT * WM - 1) / (MT * WM);
    const int64_t total = xcd_slots(static_cast<int64_t>(args.w_blocks) * args.x_blocks);
    if (total <= 0 || total > 0x7fffffffLL) {
        return hipErrorInvalidValue;
    }
    fragment_product_kernel<BF16, ROW_MAJOR, MT, NT, WM, WN><<<static_cast<unsigned>(total), 64 * WM * WN, 0, stream>>>(args);
    return hipGetLastError();
}

template <bool BF16, bool ROW_MAJOR>
static hipError_t launch_product(const ProductArgs & call, int64_t rows, int64_t columns, hipStream_t stream) {
    const ProductPlan plan = product_plan(rows, columns, call.steps);
    ProductArgs args = call;
    if (plan.full_rows > 0) {
        args.rows = static_cast<int>(plan.full_rows);
        args.x_tiles = args.rows / 32;
        const hipError_t status = launch_product_tiled<BF16, ROW_MAJOR, 2, 4, 4, 2>(args, stream);
        if (status != hipSuccess || plan.full_rows == rows) {
            return status;
        }
    }
    // the rows behind those of whole rounds
    args.rows = static_cast<int>(rows - plan.full_rows);
    args.x_tiles = (args.rows + 31) / 32;
    args.x += plan.full_rows / 32 * call.steps * 1024;
    for (int i = 0; i < args.sources; ++i) {
        args.x_source[i] += plan.full_rows * args.x_stride[i];
    }
    for (int i = 0; i < args.outputs; ++i) {
        args.y[i] += plan.full_rows * args.columns[i];
    }
    if (plan.rest_tile_columns == 256) {
        return plan.rest_tile_rows == 256 ? launch_product_tiled<BF16, ROW_MAJOR, 2, 4, 4, 2>(args, stream)
                                          : launch_product_tiled<BF16, ROW_MAJOR, 2, 2, 2, 4>(args, stream);
    }
    return launch_product_tiled<BF16, ROW_MAJOR, 2, 2, 2, 2>(args, stream);
}

template <int TYPE>
static hipError_t launch_grad_operands(GradOperandArgs args, hipStream_t stream) {
    constexpr int SPAN = TYPE == IQ2_S ? 4 : 1;
    args.row_bytes = static_cast<int64_t>(args.in_features / QK_K) * Format<TYPE>::BLOCK_BYTES;
    args.span_blocks = (args.in_features / QK_K + SPAN - 1) / SPAN;
    // (rows short enough for the 24-bit multiplies of the unit offsets: see wide_fetch)
    bool wide = Format<TYPE>::BLOCK_BYTES % 16 != 0 && args.row_bytes < (1 << 24);
    int64_t blocks = 0;
    for (int i = 0; i < args.count; ++i) {
        GradOperandSource & source = args.source[i];
        source.first_block = static_cast<int>(blocks);
        source.unpack_blocks = source.n_chunks / 2 * args.span_blocks;
        source.pack_columns = (source.n_chunks + 7) / 8;
        blocks += source.unpack_blocks + (source.grad != nullptr ? static_cast<int64_t>(source.pack_columns) * ((args.rows + 31) / 32) : 0);
        if (blocks > 0x7fffffffLL) {
            return hipErrorInvalidValue;
        }
        wide = wide && wide_stage_ok(source.packed, source.out_features * args.row_bytes);
    }
    if constexpr (Format<TYPE>::BLOCK_BYTES % 16 != 0) {
        if (wide) {
            grad_operands_kernel<TYPE, true><<<static_cast<unsigned>(blocks), 256, 0, stream>>>(args);
            return hipGetLastError();
        }
    }
    grad_operands_kernel<TYPE, false><<<static_cast<unsigned>(blocks), 256, 0, stream>>>(args);
    return hipGetLastError();
}

hipError_t launch_grad_input_unpacked(const DenseSource * sources, int count, void * workspace, uint16_t * grad_input, int64_t rows,
                                      int64_t in_features, hipStream_t stream) {
    if (count < 1 || count > UNP_SOURCES) {
        return hipErrorInvalidValue;
    }
    int64_t chunks = 0;
    // cotangents whose rows are whole stages are multiplied as they stand
    bool row_major = true;
    for (int i = 0; i < count; ++i) {
        chunks += cotangent_chunks(sources[i].out_features);
        row_major = row_major && sources[i].out_features % 32 == 0;
    }
    const UnpackedGradWorkspace view = unpacked_grad_workspace(workspace, rows, chunks, in_features);
    // (row-major: a source ends with its weight rows, a multiple of 32, and not with a whole step of 64)
    const auto chunks_of = [&](int i) { return row_major ? static_cast<int>(sources[i].out_features / 16) : cotangent_chunks(sources[i].out_features); };
    ProductArgs args = {};
    for (int i = 0; i < count; ++i) {
        args.x_source[i] = reinterpret_cast<const uint8_t *>(sources[i].activations);
        args.x_first_stage[i] = args.steps / 2;
        args.x_stride[i] = static_cast<int>(sources[i].out_features * 2);
        args.steps += chunks_of(i);
    }
    {
        const ProfileScope scope(6, stream);
        GradOperandArgs operands = {};
        operands.in_features = static_cast<int>(in_features);
        operands.rows = static_cast<int>(rows);
        operands.row_chunks = args.steps;
        for (int i = 0; i < count; ++i) {
            const int64_t first = static_cast<int64_t>(args.x_first_stage[i]) * 2 * 1024;
            operands.source[operands.count++] = {sources[i].packed, view.weights + first, row_major ? nullptr : sources[i].activations,
                                                 view.cotangent + first, static_cast<int>(sources[i].out_features), chunks_of(i)};
            if (i + 1 < count && sources[i + 1].quant_type == sources[i].quant_type) {
                continue;   // neighbours of one format share a launch
            }
            hipError_t status = hipErrorInvalidValue;
            switch (sources[i].quant_type) {
                case Q3_K: status = launch_grad_operands<Q3_K>(operands, stream); break;
                case Q4_K: status = launch_grad_operands<Q4_K>(operands, stream); break;
                case Q5_K: status = launch_grad_operands<Q5_K>(operands, stream); break;
                case Q6_K: status = launch_grad_operands<Q6_K>(operands, stream); break;
                case IQ2_S: status = launch_grad_operands<IQ2_S>(operands, stream); break;
                default: break;
            }
            if (status != hipSuccess) {
                return status;
            }
            operands.count = 0;
        }
    }
    const ProfileScope scope(3, stream);
    args.w = view.weights;
    args.x = view.cotangent;
    args.sources = count;
    args.w_tiles = static_cast<int>(in_features / 32);
    args.outputs = 1;
    args.y[0] = grad_input;
    args.columns[0] = static_cast<int>(in_features);
    return row_major ? launch_product<true, true>(args, rows, in_features, stream) : launch_product<true, false>(args, rows, in_features, stream);
}

}  // namespace tgo
