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

// ---- operands of the forward -------------------------------------------------------------------------------------
// The scaled operands of tgo_forward_scaled.hip.  A super-block is 16 steps, with Q4_K / Q5_K 17: the ninth holds the block minima
// and the fp16 block sums (eight each, the rest zero); an odd number of steps is filled up with a step of zeros.
TGO_DEVICE int unpacked_step(bool k45, int kb, int step) { return k45 ? 17 * kb + step + (step >= 8 ? 1 : 0) : 16 * kb + step; }

struct ForwardOperandSource {
    const uint8_t * packed;
    uint8_t * weights;      // slabs [out_features / 32][steps]
    float * column_power;   // 2^S of every weight row
    int out_features;
    int unpack_blocks;
    int first_block;        // of the launch
};
struct ForwardOperandArgs {
    ForwardOperandSource source[UNP_SOURCES];   // of one format
    int count;
    int64_t row_bytes;
    int in_features, rows, steps;
    int spans;              // workgroups that share 16 weight rows, each with its share of the super-blocks
    int quantize_first;     // block of the launch from which on the activations are quantized
    const uint16_t * input;
    uint8_t * x;            // slabs [rows / 32][steps]
    float * row_power;      // 2^E of every activation row
    uint32_t * tag;         // of the workspace, which holds no q8_1 layout afterwards
};
constexpr int UNF_ROWS = 16;   // weight rows of a workgroup
constexpr int UNF_X_ROWS = 8;  // activation rows of a workgroup

// One row of a Q4_K / Q5_K super-block, 64 values from group 2 `pair` on, as scaled fp16 (see tgo_forward_scaled.hip: the same operations
// in the same order): low[2w], low[2w + 1] are the group's values 4w .. 4w + 3, high[] the next group's; `part` selects 16 of the 32.
template <int TYPE>
TGO_DEVICE void decode_k45_scaled(const u32x4_t header, const u32x4_t nibbles, const u32x4_t planes, int pair, float shrink, uint32_t (&low)[8],
                                  uint32_t (&high)[8]) {
    const float d = half_bits_to_float(header.x & 0xffffu) * shrink;
    const auto scale_of = [&](int g) {
        const int j = g & 3;
        const uint32_t first = (header.y >> (8 * j)) & 63u;
        const uint32_t last = ((header.w >> (8 * j)) & 15u) | (((header.y >> (8 * j + 6)) & 3u) << 4);
        return half_scale_of(d * static_cast<float>(static_cast<int>(g < 4 ? first : last)));
    };
    const HalfScale scale_low = scale_of(2 * pair), scale_high = scale_of(2 * pair + 1);
    const uint32_t word[4] = {nibbles.x, nibbles.y, nibbles.z, nibbles.w};
    const uint32_t plane[4] = {planes.x, planes.y, planes.z, planes.w};
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        uint32_t bytes_low = word[w] & 0x0f0f0f0fu;
        uint32_t bytes_high = (word[w] >> 4) & 0x0f0f0f0fu;
        if constexpr (TYPE == Q5_K) {
            bytes_low |= ((plane[w] >> (2 * pair)) & 0x01010101u) << 4;
            bytes_high |= ((plane[w] >> (2 * pair + 1)) & 0x01010101u) << 4;
        }
        scaled_halves(bytes_low, scale_low, low[2 * w], low[2 * w + 1]);
        scaled_halves(bytes_high, scale_high, high[2 * w], high[2 * w + 1]);
    }
}

// 16 weight rows: S by a scan of the rows' scales, then a super-block per wave in turn.
template <int TYPE, bool WIDE>
TGO_DEVICE void unpack_forward_rows(const ForwardOperandArgs & args, const ForwardOperandSource & a, int block, uint8_t * shared,
                                    float * reach_lds, const void * codebook, int tid) {
    using F = Format<TYPE>;
    using W = WideStage<TYPE>;
    constexpr bool K45 = TYPE == Q4_K || TYPE == Q5_K;
    constexpr int SLOT_PITCH = WIDE ? W::PITCH : F::RAW_PITCH;
    constexpr int SLOT_FRONT = WIDE ? W::FRONT : F::RAW_SHIFT;
    constexpr int REGS = WIDE ? W::template regs<UNF_ROWS, 64>() : 1;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int row_block = block / args.spans;
    const int span = block - row_block * args.spans;
    const int super_blocks = args.in_features / QK_K;
    const int n0 = row_block * UNF_ROWS;
    const int first_row = min(n0, a.out_features - 1);   // (rows past the last one repeat it; their results are never stored)
    const int rows_valid = min(UNF_ROWS, a.out_features - first_row);
    const uint8_t * const rows = a.packed + static_cast<int64_t>(first_row) * args.row_bytes;
    const int row = lane & 15;
    const uint8_t * const my_row = rows + static_cast<int64_t>(min(row, rows_valid - 1)) * args.row_bytes;
    // S: the row's largest weight magnitude goes to [2^8, 2^9)
    float reach = 0.0f;
    for (int kb = tid >> 4; kb < super_blocks; kb += 16) {
        const uint8_t * const blk = my_row + static_cast<int64_t>(kb) * F::BLOCK_BYTES;
        if constexpr (K45) {
            const uint32_t word = *reinterpret_cast<const uint32_t *>(blk);
            reach = fmaxf(reach, fmaxf(fabsf(half_bits_to_float(word & 0xffffu)) * weight_reach<TYPE>(), fabsf(half_bits_to_float(word >> 16)) * 63.0f));
        } else {
            reach = fmaxf(reach, fabsf(half_bits_to_float(*reinterpret_cast<const uint16_t *>(blk + scale_offset<TYPE>()))) * weight_reach<TYPE>());
        }
    }
    reach = fmaxf(reach, __shfl_xor(reach, 16));
    reach = fmaxf(reach, __shfl_xor(reach, 32));
    if (lane < 16) {
        reach_lds[wave * 16 + lane] = reach;
    }
    __syncthreads();   // (and the codebook)
    reach = fmaxf(fmaxf(reach_lds[row], reach_lds[16 + row]), fmaxf(reach_lds[32 + row], reach_lds[48 + row]));
    int exponent = static_cast<int>(__float_as_uint(reach) >> 23);   // biased
    exponent = min(max(exponent, 9), 254);
    const float shrink = __uint_as_float(static_cast<uint32_t>(262 - exponent) << 23);   // 2^-S
    if (span == 0 && tid < 16) {
        a.column_power[n0 + tid] = __uint_as_float(static_cast<uint32_t>(exponent - 8) << 23);   // 2^S
    }
    const int kb0 = static_cast<int>(static_cast<int64_t>(span) * super_blocks / args.spans);
    const int kb_end = static_cast<int>(static_cast<int64_t>(span + 1) * super_blocks / args.spans);
    // slab 0 of the row tile, at this lane's row
    uint8_t * const out = a.weights + static_cast<int64_t>(row_block >> 1) * args.steps * 1024 + ((row_block & 1) * 16 + row) * 16;
    const int quarter = lane >> 4;   // 64 values of the super-block
    if constexpr (K45) {
        constexpr int QS = TYPE == Q4_K ? 16 : 48;
        for (int kb = kb0 + wave; kb < kb_end; kb += 4) {
            const uint8_t * const blk = my_row + static_cast<int64_t>(kb) * F::BLOCK_BYTES;
            const u32x4_t header = *reinterpret_cast<const u32x4_t *>(blk);
            u32x4_t nibbles[2], planes[2] = {};
#pragma unroll
            for (int part = 0; part < 2; ++part) {
                nibbles[part] = *reinterpret_cast<const u32x4_t *>(blk + QS + quarter * 32 + part * 16);
                if constexpr (TYPE == Q5_K) {
                    planes[part] = *reinterpret_cast<const u32x4_t *>(blk + 16 + part * 16);
                }
            }
#pragma unroll
            for (int part = 0; part < 2; ++part) {
                uint32_t low[8], high[8];
                decode_k45_scaled<TYPE>(header, nibbles[part], planes[part], quarter, shrink, low, high);
                uint8_t * const at_low = out + static_cast<int64_t>(unpacked_step(true, kb, 4 * quarter + part)) * 1024;
                uint8_t * const at_high = out + static_cast<int64_t>(unpacked_step(true, kb, 4 * quarter + 2 + part)) * 1024;
                *reinterpret_cast<uint4 *>(at_low) = make_uint4(low[0], low[1], low[2], low[3]);
                *reinterpret_cast<uint4 *>(at_low + 512) = make_uint4(low[4], low[5], low[6], low[7]);
                *reinterpret_cast<uint4 *>(at_high) = make_uint4(high[0], high[1], high[2], high[3]);
                *reinterpret_cast<uint4 *>(at_high + 512) = make_uint4(high[4], high[5], high[6], high[7]);
            }
            uint8_t * const minima = out + static_cast<int64_t>(17 * kb + 8) * 1024;
            if (quarter == 0) {
                const float minus = -half_bits_to_float(header.x >> 16) * shrink;
                uint32_t packed[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float product[2];
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        const int g = 2 * i + e, j = g & 3;
                        const uint32_t mn = g < 4 ? (header.z >> (8 * j)) & 63u
                                                  : ((header.w >> (8 * j + 4)) & 15u) | (((header.z >> (8 * j + 6)) & 3u) << 4);
                        product[e] = minus * static_cast<float>(static_cast<int>(mn));
                    }
                    packed[i] = __builtin_bit_cast(uint32_t, half2_t{static_cast<_Float16>(product[0]), static_cast<_Float16>(product[1])});
                }
                *reinterpret_cast<uint4 *>(minima) = make_uint4(packed[0], packed[1], packed[2], packed[3]);
            } else if (quarter == 1) {
                *reinterpret_cast<uint4 *>(minima + 512) = make_uint4(0, 0, 0, 0);
            } else if (kb + 1 == super_blocks && (super_blocks & 1) != 0) {
                *reinterpret_cast<uint4 *>(out + static_cast<int64_t>(args.steps - 1) * 1024 + (quarter - 2) * 512) = make_uint4(0, 0, 0, 0);
            }
        }
    } else {
        uint8_t * const raw = shared + wave * (UNF_ROWS * SLOT_PITCH);
        WideRegs<REGS> regs;
        if constexpr (WIDE) {
            wide_fetch<TYPE, UNF_ROWS, 64, REGS>(regs, rows, static_cast<int>(args.row_bytes), rows_valid, min(kb0 + wave, super_blocks - 1), lane);
        }
        for (int kb = kb0 + wave; kb < kb_end; kb += 4) {
            if constexpr (WIDE) {
                wide_park<TYPE, UNF_ROWS, 64, REGS>(raw, regs, rows, static_cast<int>(args.row_bytes), rows_valid, kb, lane);
                wide_fetch<TYPE, UNF_ROWS, 64, REGS>(regs, rows, static_cast<int>(args.row_bytes), rows_valid, min(kb + 4, super_blocks - 1), lane);
            } else {
                stage_blocks<TYPE>(raw, a.packed, args.row_bytes, first_row, a.out_features, kb, UNF_ROWS, lane, 64);
            }
            // (LDS executes a wave's accesses in order; the compiler keeps them so)
            __builtin_amdgcn_wave_barrier();
            asm volatile("" ::: "memory");
            const uint8_t * const blk = raw + row * SLOT_PITCH + SLOT_FRONT;
            const float scale = half_weight_scale<TYPE>(blk) * shrink;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int unit = 4 * quarter + i;
                uint32_t words[8];
                decode16_scaled<TYPE>(blk, unit, static_cast<const std::conditional_t<TYPE == IQ2_S, Iq2sSelectors, uint2> *>(codebook), scale, words);
                uint8_t * const at = out + static_cast<int64_t>(16 * kb + unit) * 1024;
                *reinterpret_cast<uint4 *>(at) = make_uint4(words[0], words[1], words[2], words[3]);
                *reinterpret_cast<uint4 *>(at + 512) = make_uint4(words[4], words[5], words[6], words[7]);
            }
            __builtin_amdgcn_wave_barrier();
            asm volatile("" ::: "memory");
        }
    }
}

// Eight activation rows: E by a first pass over them, then quants, block scales and sums as in quantize_q8_1_scaled_kernel, brought to the
// row's exponent here instead of in the multiplying waves (one more rounding for values below 2^-14 only, as there).
template <bool K45>
TGO_DEVICE void quantize_forward_rows(const ForwardOperandArgs & args, int block, float * reach_lds, int tid) {
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int super_blocks = args.in_features / QK_K;
    const int r8 = lane >> 3, j = lane & 7;
    const int row = block * UNF_X_ROWS + r8;
    const bool present = row < args.rows;
    const uint16_t * const source = args.input + static_cast<int64_t>(min(row, args.rows - 1)) * args.in_features + j * 8;
    const auto load = [&](int kb, int i) {
        const uint4 bits = *reinterpret_cast<const uint4 *>(source + kb * QK_K + i * 64);
        return present ? bits : uint4{0, 0, 0, 0};
    };
    float largest = 0.0f;
#pragma unroll 2
    for (int kb = wave; kb < super_blocks; kb += 4) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float x[8];
            unpack_bf16x8(load(kb, i), x);
#pragma unroll
            for (int e = 0; e < 8; ++e) largest = fmaxf(largest, fabsf(x[e]));
        }
    }
    largest = fmaxf(largest, __shfl_xor(largest, 1));
    largest = fmaxf(largest, __shfl_xor(largest, 2));
    largest = fmaxf(largest, __shfl_xor(largest, 4));
    if (j == 0) {
        reach_lds[wave * 8 + r8] = largest;
    }
    __syncthreads();
    largest = fmaxf(fmaxf(reach_lds[r8], reach_lds[8 + r8]), fmaxf(reach_lds[16 + r8], reach_lds[24 + r8]));
    // the exponent of a scale d, biased, as far as powers of two reach (the largest d is that of the largest value)
    const auto exponent_of = [](float d) { return min(max(static_cast<int>(__float_as_uint(d) >> 23), 2), 254); };
    const int row_exponent = exponent_of(largest == 0.0f ? 0.0f : largest / 127.0f);
    if (wave == 0 && j == 0) {
        args.row_power[row] = __uint_as_float(static_cast<uint32_t>(row_exponent - 1) << 23);   // 2^E
    }
    uint8_t * const out = args.x + static_cast<int64_t>(row >> 5) * args.steps * 1024 + (row & 31) * 16;
    for (int kb = wave; kb < super_blocks; kb += 4) {
        uint32_t halves[4][4];
        float d[4], total[4];
        float d_largest = 0.0f;
        int magnitude[4][8];
        uint4 bits[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) bits[i] = load(kb, i);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float x[8];
            unpack_bf16x8(bits[i], x);
            uint32_t packed[2];
            quantize_eight(bits[i], x, packed, d[i], total[i], halves[i], magnitude[i]);
            d_largest = fmaxf(d_largest, d[i]);
        }
        d_largest = fmaxf(d_largest, __shfl_xor(d_largest, 4));   // (a block's scale is the same on its four lanes)
        const int exponent = exponent_of(d_largest);
        const float inverse = __uint_as_float(static_cast<uint32_t>(255 - exponent) << 23);   // 2^-e
        const float power = __uint_as_float(static_cast<uint32_t>(exponent - 1) << 23);       // 2^e
        const _Float16 half_ratio = static_cast<_Float16>(power * __uint_as_float((254u - static_cast<uint32_t>(row_exponent - 1)) << 23));   // 2^(e - E)
        const half2_t ratio = {half_ratio, half_ratio};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float lane_scale = d[i] * inverse;
            const uint32_t words[4] = {bits[i].x, bits[i].y, bits[i].z, bits[i].w};
            uint32_t result[4];
#pragma unroll
            for (int pair = 0; pair < 4; ++pair) {
                const half2_t values = {static_cast<_Float16>(static_cast<float>(magnitude[i][2 * pair]) * lane_scale),
                                        static_cast<_Float16>(static_cast<float>(magnitude[i][2 * pair + 1]) * lane_scale)};
                result[pair] = half2_mul(__builtin_bit_cast(uint32_t, values) | (words[pair] & 0x80008000u), ratio);
            }
            // piece 8i + j of the super-block: 8 values of step (8i + j) / 2
            const int piece = 8 * i + j;
            *reinterpret_cast<uint4 *>(out + static_cast<int64_t>(unpacked_step(K45, kb, piece >> 1)) * 1024 + (piece & 1) * 512) =
                make_uint4(result[0], result[1], result[2], result[3]);
        }
        if constexpr (K45) {
            uint8_t * const sums = out + static_cast<int64_t>(17 * kb + 8) * 1024;
            if ((j & 3) == 0) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const half2_t sum = {static_cast<_Float16>(total[i] * inverse), static_cast<_Float16>(0.0f)};
                    *reinterpret_cast<uint16_t *>(sums + (2 * i + (j >> 2)) * 2) =
                        static_cast<uint16_t>(half2_mul(__builtin_bit_cast(uint32_t, sum), ratio));
                }
            } else if (j == 1) {
                *reinterpret_cast<uint4 *>(sums + 512) = make_uint4(0, 0, 0, 0);
            } else if (j < 4 && kb + 1 == super_blocks && (super_blocks & 1) != 0) {   // (lanes 2 and 3)
                *reinterpret_cast<uint4 *>(out + static_cast<int64_t>(args.steps - 1) * 1024 + (j - 2) * 512) = make_uint4(0, 0, 0, 0);
            }
        }
    }
}

// Eight rows per workgroup: the row's exponent needs all of it, and 32 rows a workgroup would leave most of the chip idle at a few hundred
// rows.  Bound by memory and, below 16 million weights, by the latency of its two passes.
template <int TYPE, bool WIDE>
__global__ __launch_bounds__(256) void forward_operands_kernel(const ForwardOperandArgs args) {
    constexpr int SLOT = TYPE == Q4_K || TYPE == Q5_K ? 1 : WIDE ? WideStage<TYPE>::PITCH : Format<TYPE>::RAW_PITCH;
    __shared__ __attribute__((aligned(16))) uint8_t shared[4 * UNF_ROWS * SLOT];
    __shared__ float reach[64];
    __shared__ std::conditional_t<TYPE == IQ2_S, Iq2sSelectors, uint2> codebook;
    const int tid = threadIdx.x;
    if (blockIdx.x == 0 && tid == 0) {
        *args.tag = 0;
    }
    if (static_cast<int>(blockIdx.x) >= args.quantize_first) {
        quantize_forward_rows<TYPE == Q4_K || TYPE == Q5_K>(args, static_cast<int>(blockIdx.x) - args.quantize_first, reach, tid);
        return;
    }
    if constexpr (TYPE == IQ2_S) {
        expand_iq2s_selectors(codebook, tid, 256);
    }
    int index = 0;
#pragma unroll
    for (int i = 1; i < UNP_SOURCES; ++i) {
        index = i < args.count && static_cast<int>(blockIdx.x) >= args.source[i].first_block ? i : index;
    }
    unpack_forward_rows<TYPE, WIDE>(args, args.source[index], static_cast<int>(blockIdx.x) - args.source[index].first_block, shared, reach, &codebook,
                                    tid);
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
    // scaled operands (forward): y is multiplied by row_power[r] * column_power[c], c counted over all tiles of w
    const float * row_power;
    const float * column_power;
};

// 32-bit address of an LDS object
TGO_DEVICE uint32_t lds_address(const void * p) {
    return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) uint8_t *)p));
}

// Requests a slab: 16 bytes per lane, from `base` + the lane's `offset` to the LDS address `to` + 16 x lane.  The load takes its LDS address from m0 as it
// issues, and one that follows a scalar write of m0 at once may still see the old value: a wait state lies between them, which the compiler
// does not add inside a piece of assembly.  m0 is one of its reserved registers, which a clobber list does not protect: nothing else in these
// kernels may use it.  (check_lds_loads.py looks for both in every build.)
TGO_DEVICE void slab_to_lds(uint32_t to, uint32_t offset, const uint8_t * base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(to), "v"(offset), "s"(base) : "memory");
}
// And the slab behind it, to the place behind it: the instruction's offset counts in both addresses.  (With a wait state for every slab the product
// of 4096 x 4096 x 2048 takes 73.9 us instead of 72.8, and forward and backward of that size 169.8 instead of 167.0; with one for every pair, and
// half as many writes of m0, 166.4 instead of 166.3.)
TGO_DEVICE void slab_pair_to_lds(uint32_t to, uint32_t offset, const uint8_t * base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\tglobal_load_lds_dwordx4 %1, %2 offset:1024" ::"s"(to), "v"(offset),
                 "s"(base)
                 : "memory");
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
    // Its workgroups (one per CU, two with 128 x 128 tiles) take the tiles of the share in turn.
    const int total = a.w_blocks * a.x_blocks;
    const int per_xcd = (total + XCDS - 1) / XCDS;
    const int first_id = static_cast<int>(blockIdx.x % XCDS) * per_xcd;
    const int slots = static_cast<int>(gridDim.x) / XCDS;
    const int slot = static_cast<int>(blockIdx.x) / XCDS;
    const int share = min(per_xcd, total - first_id);
    const int items = share > slot ? (share - slot + slots - 1) / slots : 0;
    if (items == 0) {
        return;
    }
    const auto place = [&](int item, int & w_block, int & x_block) __attribute__((always_inline)) {
        constexpr int BAND = 8;
        const int id = first_id + slot + item * slots;
        const int band = id / (BAND * a.w_blocks);
        const int band_rows = min(BAND, a.x_blocks - band * BAND);
        const int in_band = id - band * BAND * a.w_blocks;
        x_block = band * BAND + in_band % band_rows;
        w_block = in_band / band_rows;
    };
    const int stages = a.steps / SS;

    // W_PER of a wave's requests are slabs of the weights, the others the rows' share.  (Tiles past the last one repeat it; nothing of
    // what they give is stored.)
    constexpr int W_PER = W_TILES * SS / WAVES, X_PER = PER - W_PER;
    static_assert(W_TILES * SS % WAVES == 0, "every wave requests as many slabs of either kind");
    static_assert(SS == 2 && W_PER % SS == 0, "and both slabs that a tile of the weights has in a stage");
    constexpr bool X_PAIRS = !ROW_MAJOR && X_PER % SS == 0;
    constexpr int X_SOURCES = X_PAIRS ? X_PER / SS : X_PER;
    const uint8_t * w_source[W_PER / SS];
    const uint8_t * x_source[X_SOURCES];
    uint32_t x_lane[X_PER];
    const uint32_t ring_address = lds_address(ring);
    const uint32_t lane16 = lane * 16;
    int request_item = 0, requested = 0;   // the tile whose stages are being requested, and how many of them have been
    int x_block_requested = 0;
    int x_left = 0;   // ROW_MAJOR: stages until the next source begins
    int x_next = 0;   // and which one that is
    auto open_source = [&](int index) __attribute__((always_inline)) {
        const int stride = a.x_stride[index];
#pragma unroll
        for (int i = 0; i < X_PER; ++i) {
            const int slab = wave * X_PER + i;
            const int row0 = (x_block_requested * X_TILES + slab / SS) * 32 + 16 * (slab % SS);
            const int row = lane >> 2;
            const int piece = (lane & 3) ^ ((row >> 1) & 3);
            const int first = min(row0, a.rows - 1);   // (rows past the last one repeat it)
            x_source[i] = a.x_source[index] + static_cast<int64_t>(first) * stride;
            x_lane[i] = static_cast<uint32_t>(min(row, a.rows - 1 - first)) * static_cast<uint32_t>(stride) + piece * 16;
        }
        x_next = index + 1;
        x_left = (x_next < a.sources ? a.x_first_stage[x_next] : stages) - a.x_first_stage[index];
    };
    auto open_item = [&]() __attribute__((always_inline)) {
        int w_block;
        place(request_item, w_block, x_block_requested);
#pragma unroll
        for (int i = 0; i < W_PER / SS; ++i) {
            const int t = min(w_block * W_TILES + wave * (W_PER / SS) + i, a.w_tiles - 1);
            w_source[i] = a.w + static_cast<int64_t>(t) * a.steps * 1024;
        }
        if constexpr (ROW_MAJOR) {
            open_source(0);
        } else {
#pragma unroll
            for (int i = 0; i < X_SOURCES; ++i) {
                const int slab = X_PAIRS ? (wave * X_SOURCES + i) * SS : wave * X_PER + i;
                const int t = min(x_block_requested * X_TILES + slab / SS, a.x_tiles - 1);
                x_source[i] = a.x + (static_cast<int64_t>(t) * a.steps + slab % SS) * 1024;
                x_lane[i] = lane16;
            }
        }
    };
    // Requests the next stage, after a tile's last one the first of the workgroup's next tile; past the last tile its last stage again, into a
    // buffer that nobody reads any more.
    auto request = [&](int buffer) __attribute__((always_inline)) {
        const uint32_t to = ring_address + buffer * STAGE;
#pragma unroll
        for (int i = 0; i < W_PER / SS; ++i) {
            slab_pair_to_lds(to + (wave * W_PER + i * SS) * 1024, lane16, w_source[i]);
        }
#pragma unroll
        for (int i = 0; i < X_SOURCES; ++i) {
            if constexpr (X_PAIRS) {
                slab_pair_to_lds(to + (W_TILES * SS + wave * X_PER + i * SS) * 1024, x_lane[i], x_source[i]);
            } else {
                slab_to_lds(to + (W_TILES * SS + wave * X_PER + i) * 1024, x_lane[i], x_source[i]);
            }
        }
        if (++requested < stages) {
#pragma unroll
            for (int i = 0; i < W_PER / SS; ++i) w_source[i] += SS * 1024;
#pragma unroll
            for (int i = 0; i < X_SOURCES; ++i) x_source[i] += ROW_MAJOR ? SS * 32 : SS * 1024;
            if constexpr (ROW_MAJOR) {
                if (--x_left == 0) {
                    open_source(x_next);
                }
            }
        } else if (request_item + 1 < items) {
            ++request_item;
            requested = 0;
            open_item();
        }
    };
    open_item();
    // The wave's requests are complete but for those of the two youngest stages, its reads are done, and so are the others'.
    auto meet = [&]() __attribute__((always_inline)) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((UNP_RING - 2) * PER) : "memory");
    };
    const int wm = wave % WM, wn = wave / WM;
    // ROW_MAJOR: where the lane's piece of step 0 lies in a row tile
    const int x_piece = (lane & 31) * 64 + (((lane >> 5) ^ ((lane >> 1) & 3)) * 16);
    v16f acc[NT][MT];
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
    const int l32 = lane & 31, half = lane >> 5;
    int buffer = 0, free_buffer = UNP_RING - 1;
#pragma unroll 1
    for (int item = 0; item < items; ++item) {
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int m = 0; m < MT; ++m) acc[n][m] = v16f{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll 1
        for (int s = 0; s < stages; ++s) {
            // the buffer of the stage before: all waves have read it before they last met
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
        int w_block, x_block;
        place(item, w_block, x_block);
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
                if constexpr (!BF16) {
                    const float row_power = a.row_power[min(r0 + l32, a.rows - 1)];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const float4 column_power = *reinterpret_cast<const float4 *>(a.column_power + tile * 32 + 8 * j + 4 * half);
                        acc[n][m][4 * j + 0] *= row_power * column_power.x;
                        acc[n][m][4 * j + 1] *= row_power * column_power.y;
                        acc[n][m][4 * j + 2] *= row_power * column_power.z;
                        acc[n][m][4 * j + 3] *= row_power * column_power.w;
                    }
                }
                store_rows_32xn<1>(&acc[n][m], a.y[output] + static_cast<int64_t>(r0) * columns + c0, columns, a.rows - r0, columns - c0, lane);
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (nothing may arrive in the LDS of a workgroup that has ended)
}

template <bool BF16, bool ROW_MAJOR, int MT, int NT, int WM, int WN>
static hipError_t launch_product_tiled(ProductArgs args, hipStream_t stream) {
    args.w_blocks = (args.w_tiles + NT * WN - 1) / (NT * WN);
    args.x_blocks = (args.x_tiles + MT * WM - 1) / (MT * WM);
    const int64_t total = static_cast<int64_t>(args.w_blocks) * args.x_blocks;
    if (total <= 0 || total > 0x7fffff00LL) {
        return hipErrorInvalidValue;
    }
    constexpr int64_t RESIDENT = 256 * (WM * WN == 4 ? 2 : 1);   // workgroups that the chip holds
    const unsigned grid = static_cast<unsigned>(std::min(xcd_slots(total), RESIDENT));
    fragment_product_kernel<BF16, ROW_MAJOR, MT, NT, WM, WN><<<grid, 64 * WM * WN, 0, stream>>>(args);
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
    if (args.row_power != nullptr) {
        args.row_power += plan.full_rows;
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
    int64_t widths[UNP_SOURCES];
    for (int i = 0; i < count; ++i) {
        widths[i] = sources[i].out_features;
    }
    // cotangents whose rows are whole stages are multiplied as they stand
    const UnpackedGradWorkspace view = unpacked_grad_workspace(workspace, rows, count, widths, in_features);
    const bool row_major = view.row_major;
    const auto chunks_of = [&](int i) { return static_cast<int>(view.chunks_of(widths[i])); };
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

template <int TYPE>
static hipError_t launch_forward_operands(ForwardOperandArgs args, hipStream_t stream) {
    args.row_bytes = static_cast<int64_t>(args.in_features / QK_K) * Format<TYPE>::BLOCK_BYTES;
    int64_t tiles = 0;
    for (int i = 0; i < args.count; ++i) {
        tiles += (args.source[i].out_features + 31) / 32;
    }
    // Two workgroups per tile of 32 weight rows, more where those do not fill the chip, each with four super-blocks at least.
    args.spans = static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(512 / (2 * tiles), args.in_features / QK_K / 4)));
    bool wide = Format<TYPE>::BLOCK_BYTES % 16 != 0 && args.row_bytes < (1 << 24);
    int64_t blocks = 0;
    for (int i = 0; i < args.count; ++i) {
        ForwardOperandSource & source = args.source[i];
        source.first_block = static_cast<int>(blocks);
        source.unpack_blocks = (source.out_features + 31) / 32 * 2 * args.spans;
        blocks += source.unpack_blocks;
        wide = wide && wide_stage_ok(source.packed, source.out_features * args.row_bytes);
    }
    args.quantize_first = static_cast<int>(blocks);
    blocks += pad_rows(args.rows) / UNF_X_ROWS;
    if (blocks > 0x7fffffffLL) {
        return hipErrorInvalidValue;
    }
    if constexpr (Format<TYPE>::BLOCK_BYTES % 16 != 0) {
        if (wide) {
            forward_operands_kernel<TYPE, true><<<static_cast<unsigned>(blocks), 256, 0, stream>>>(args);
            return hipGetLastError();
        }
    }
    forward_operands_kernel<TYPE, false><<<static_cast<unsigned>(blocks), 256, 0, stream>>>(args);
    return hipGetLastError();
}

hipError_t launch_forward_unpacked(const uint16_t * input, void * workspace, const DenseSource * sources, uint16_t * const * outputs, int count,
                                   void * scratch, int64_t rows, int64_t in_features, hipStream_t stream) {
    if (count < 1 || count > UNP_SOURCES) {
        return hipErrorInvalidValue;
    }
    const int quant_type = sources[0].quant_type;
    ForwardOperandArgs operands = {};
    operands.count = count;
    operands.in_features = static_cast<int>(in_features);
    operands.rows = static_cast<int>(rows);
    operands.steps = static_cast<int>(unpacked_forward_steps(quant_type, in_features));
    operands.input = input;
    operands.x = static_cast<uint8_t *>(workspace);
    operands.row_power = reinterpret_cast<float *>(operands.x + pad_rows(rows) * operands.steps * 32);
    operands.tag = q8_workspace_view(workspace, rows, in_features, false, OPERAND_SCALED).tag;
    int tiles = 0;
    int64_t columns = 0;
    for (int i = 0; i < count; ++i) {
        tiles += static_cast<int>((sources[i].out_features + 31) / 32);
    }
    float * const column_power = reinterpret_cast<float *>(static_cast<uint8_t *>(scratch) + static_cast<int64_t>(tiles) * operands.steps * 1024);
    ProductArgs args = {};
    args.w_tiles = tiles;
    tiles = 0;
    for (int i = 0; i < count; ++i) {
        if (sources[i].quant_type != quant_type) {
            return hipErrorInvalidValue;
        }
        operands.source[i].packed = sources[i].packed;
        operands.source[i].weights = static_cast<uint8_t *>(scratch) + static_cast<int64_t>(tiles) * operands.steps * 1024;
        operands.source[i].column_power = column_power + tiles * 32;
        operands.source[i].out_features = static_cast<int>(sources[i].out_features);
        args.y[i] = outputs[i];
        args.first_tile[i] = tiles;
        args.columns[i] = static_cast<int>(sources[i].out_features);
        tiles += static_cast<int>((sources[i].out_features + 31) / 32);
    }
    columns = static_cast<int64_t>(tiles) * 32;
    {
        const ProfileScope scope(0, stream);
        hipError_t status = hipErrorInvalidValue;
        switch (quant_type) {
            case Q3_K: status = launch_forward_operands<Q3_K>(operands, stream); break;
            case Q4_K: status = launch_forward_operands<Q4_K>(operands, stream); break;
            case Q5_K: status = launch_forward_operands<Q5_K>(operands, stream); break;
            case Q6_K: status = launch_forward_operands<Q6_K>(operands, stream); break;
            case IQ2_S: status = launch_forward_operands<IQ2_S>(operands, stream); break;
            default: break;
        }
        if (status != hipSuccess) {
            return status;
        }
    }
    const ProfileScope scope(2, stream);
    args.w = static_cast<const uint8_t *>(scratch);
    args.x = operands.x;
    args.steps = operands.steps;
    args.outputs = count;
    args.row_power = operands.row_power;
    args.column_power = column_power;
    return launch_product<false, false>(args, rows, columns, stream);
}

}  // namespace tgo
