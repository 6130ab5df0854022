// What the forward kernels with scaled fp16 operands share: operand arithmetic and the epilogue's stores.
#pragma once

#include "tgo_device.h"

namespace tgo {

typedef float v16f __attribute__((ext_vector_type(16)));

// Slot of one packed block in LDS: Q4_K/Q5_K blocks are whole 16-byte units and lie back to back (16-byte reads of 32
// consecutive rows then cover all banks); the other formats take the larger of their two staging pitches.
template <int TYPE>
struct ScaledSlot {
    static constexpr bool K45 = TYPE == Q4_K || TYPE == Q5_K;
    static constexpr int BYTES = K45 ? Format<TYPE>::BLOCK_BYTES
                                     : (Format<TYPE>::RAW_PITCH > WideStage<TYPE>::PITCH ? Format<TYPE>::RAW_PITCH
                                                                                          : WideStage<TYPE>::PITCH);
};

// 6-bit scale and minimum of 32-value group G of a Q4_K/Q5_K block from its 12 scale bytes (three words)
template <int G>
TGO_DEVICE void k45_group_scale_min(uint32_t w1, uint32_t w2, uint32_t w3, int & sc, int & mn) {
    if constexpr (G < 4) {
        sc = static_cast<int>((w1 >> (8 * G)) & 63u);
        mn = static_cast<int>((w2 >> (8 * G)) & 63u);
    } else {
        constexpr int J = G - 4;
        sc = static_cast<int>(((w3 >> (8 * J)) & 15u) | (((w1 >> (8 * J + 6)) & 3u) << 4));
        mn = static_cast<int>(((w3 >> (8 * J + 4)) & 15u) | (((w2 >> (8 * J + 6)) & 3u) << 4));
    }
}

// (1024 + byte) pairs times an fp16 multiplier h, minus the bias: fma(1024 + b, h, -1024 h) is evaluated with one
// rounding and -1024 h is a power-of-two multiple of h, so the result is fp16(b * h).
TGO_DEVICE HalfScale half_scale_of(float value) {
    const _Float16 h = static_cast<_Float16>(value);
    const _Float16 offset = static_cast<_Float16>(-1024.0f) * h;
    return HalfScale{half2_t{h, h}, half2_t{offset, offset}};
}

// Largest magnitude a weight of the format can take per unit of its super-block scale d.
template <int TYPE>
constexpr float weight_reach() {
    return TYPE == Q4_K ? 63.0f * 15.0f : TYPE == Q5_K ? 63.0f * 31.0f : TYPE == Q3_K ? 32.0f * 4.0f
           : TYPE == Q6_K ? 128.0f * 32.0f : 31.0f * 43.0f / 8.0f;
}

// Byte offset of the fp16 super-block scale d inside a block (Q4_K/Q5_K: d, then dmin).
template <int TYPE>
constexpr int scale_offset() { return TYPE == Q3_K ? 108 : TYPE == Q6_K ? 208 : 0; }


// Values 16u .. 16u + 15 of a super-block as the scaled fp16 operand fp16(v * h): v the exact integer sub-scale x quant, `scale`
// = h = 2^-S times the super-block's scale (half_weight_scale), which is exact in fp16 in the range that S leaves it in.
// out[i] holds values 2i and 2i + 1.  Q4_K/Q5_K have their own code in the kernels.
//   Q3_K   b = quant + 4 in 0..7 is placed as b << 5 under the bits of 32.0, whose mantissa counts bit 5 as one:
//          (32 + b) * sub - 36 * sub is exact (sub has six bits, 9 * sub ten), one multiply-add where an addition and a
//          multiplication stood
//   Q6_K   sub * quant has up to 13 bits, so h * sub is split into an fp16 number and its exact rest (19 bits in all): quant * rest
//          is rounded at 2^-22 of the result, then one multiply-add rounds the sum.  (The split of the integer into two operands
//          cost six instructions per pair of values, this one four.)
//   IQ2_S  a unit's values are +-h * (2s + 1) times one of three magnitudes: the three are rounded, every value picks its own
// The kernels that multiply few rows per unpacked weight are bound by these instructions.  Against the exact-integer operand of
// decode16_half with a multiplication behind every pair, 256 experts of 2048 x 512, gate and up: Q6_K, 64 rows each 346 -> 317 us,
// 256 rows 526 -> 500; IQ2_S, 16 rows 147 -> 134, 64 rows 262 -> 252; dense Q6_K 4096 x 4096 x 4096 forward and quantizing 220 -> 202.
template <int TYPE, typename Codebook>
TGO_DEVICE void decode16_scaled(const uint8_t * blk, int u, const Codebook * codebook, float scale, uint32_t (&out)[8]) {
    static_assert(TYPE == Q3_K || TYPE == Q6_K || TYPE == IQ2_S, "formats with 16-value scale groups");
    if constexpr (TYPE == Q3_K) {
        const int i0 = 16 * u;
        const uint8_t * qs = blk + 32 + (i0 >> 7) * 32 + (i0 & 31);
        const uint8_t * hm = blk + (i0 & 31);
        const int shift_l = 2 * ((i0 & 127) >> 5);
        const int shift_h = i0 >> 5;
        const uint8_t * scales = blk + 96;
        const int low = scales[u & 7] >> (4 * (u >> 3));
        const int high = scales[8 + (u & 3)] >> (2 * (u >> 2));
        const int sub = ((low & 0x0f) | ((high & 3) << 4)) - 32;
        const half2_t multiplier = half2_of(sub);
        const half2_t offset = half2_of(-36 * sub);
        const _Float16 h = static_cast<_Float16>(scale);
        const half2_t scale2 = {h, h};
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const uint32_t low_word = lds_u32(qs + 4 * t);
            const uint32_t high_word = lds_u32(hm + 4 * t);
            const uint32_t low_bits = shift_l < 6 ? low_word << (5 - shift_l) : low_word >> 1;
            const uint32_t b = (low_bits & 0x60606060u) | ((high_word << (7 - shift_h)) & 0x80808080u);
            const uint32_t p = __builtin_amdgcn_perm(0x50505050u, b, 0x04010400u);
            const uint32_t q = __builtin_amdgcn_perm(0x50505050u, b, 0x04030402u);
            out[2 * t] = half2_mul(half2_fma(p, multiplier, offset), scale2);
            out[2 * t + 1] = half2_mul(half2_fma(q, multiplier, offset), scale2);
        }
    } else if constexpr (TYPE == Q6_K) {
        const int chunk = u >> 3;
        const int rem = (16 * u) & 127;
        const uint8_t * ql = blk + chunk * 64 + (rem & 63);
        const uint8_t * qh = blk + 128 + chunk * 32 + ((16 * u) & 31);
        const int shift_l = 4 * (rem >> 6);
        const int shift_h = 2 * ((rem >> 5) & 3);
        const float product = scale * static_cast<float>(static_cast<int8_t>(blk[192 + u]));
        const _Float16 head = static_cast<_Float16>(product);
        const _Float16 rest = static_cast<_Float16>(product - static_cast<float>(head));
        const half2_t head2 = {head, head}, rest2 = {rest, rest};
        const half2_t unbias = half2_of(-1056);      // 1024 + the quant's offset of 32
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const uint32_t low = lds_u32(ql + 4 * t) >> shift_l;
            const uint32_t high_word = lds_u32(qh + 4 * t);
            const uint32_t high = shift_h < 4 ? high_word << (4 - shift_h) : high_word >> (shift_h - 4);
            const uint32_t b = (low & 0x0f0f0f0fu) | (high & 0x30303030u);
            uint32_t p, q;
            bytes_to_biased_halves(b, p, q);
            p = half2_add(p, unbias);
            q = half2_add(q, unbias);
            out[2 * t] = half2_fma(p, head2, __builtin_bit_cast(half2_t, half2_mul(p, rest2)));
            out[2 * t + 1] = half2_fma(q, head2, __builtin_bit_cast(half2_t, half2_mul(q, rest2)));
        }
    } else {
        const uint8_t * qs = blk + 2;
        const uint32_t idx_pair = lds_u16(qs + 2 * u);
        const uint32_t sign_pair = lds_u16(qs + 32 + 2 * u);
        const uint32_t qh = blk[66 + (u >> 1)] >> (4 * (u & 1));
        const half2_t multiplier = half2_of(2 * static_cast<int>((blk[74 + (u >> 1)] >> (4 * (u & 1))) & 0x0f) + 1);
        const _Float16 h = static_cast<_Float16>(scale);
        const half2_t scale2 = {h, h};
        const uint32_t low_pair = half2_mul(half2_mul(__builtin_bit_cast(uint32_t, multiplier), half2_t{static_cast<_Float16>(8.0f), static_cast<_Float16>(25.0f)}), scale2);
        const uint32_t high = half2_mul(half2_mul(__builtin_bit_cast(uint32_t, multiplier), half2_t{static_cast<_Float16>(43.0f), static_cast<_Float16>(0.0f)}), scale2);
        const uint32_t spread = (sign_pair & 0x5555u) | ((sign_pair & 0xaaaau) << 15);
#pragma unroll
        for (int gsel = 0; gsel < 2; ++gsel) {
            const uint32_t index = ((idx_pair >> (8 * gsel)) & 0xff) | (((qh >> (2 * gsel)) & 3) << 8);
            const uint4 selector = codebook->entry[index];
            const uint32_t words[4] = {selector.x, selector.y, selector.z, selector.w};
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                const int i = 4 * gsel + p;
                const uint32_t picked = __builtin_amdgcn_perm(high, low_pair, words[p]);
                out[i] = picked ^ ((spread << (15 - 2 * i)) & 0x80008000u);   // (the scale may be negative)
            }
        }
    }
}

// The lane's number computed from nothing, and opaque: what is derived from it is derived where it is used instead of
// being kept in a register through a loop (where such a register is spilled, its reload waits for every load in flight).
TGO_DEVICE int lane_afresh() {
    int lane = static_cast<int>(__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)));
    asm volatile("" : "+v"(lane));
    return lane;
}

// Stores the wave's 32 rows x (32 * TILES) columns of results, which the matrix instructions left transposed (weights as the
// A operand: the lane holds row l32 and, as element v of tile t, column 32 t + 8 (v / 4) + 4 (lane / 32) + v % 4), as
// bf16.  The two half-waves exchange runs of four columns, after which a lane holds eight neighbouring columns and
// stores 16 bytes; a row gets 32 contiguous bytes per instruction.  `dst` points at row 0, column 0; rows >=
// valid_rows and columns >= valid_cols are skipped.  The 16-byte path needs row_stride % 8 == 0 (dst is then 16-byte
// aligned: the tensor is, and column tiles start at multiples of 128).
template <int TILES>
TGO_DEVICE void store_rows_32xn(const v16f * tiles, uint16_t * dst, int64_t row_stride, int valid_rows, int valid_cols, int lane) {
    const int l32 = lane & 31;
    const int half = lane >> 5;
    const bool wide = (row_stride & 7) == 0;
    uint16_t * const row = dst + l32 * row_stride;
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            // runs 2m and 2m + 1 of the tile: the lower half-wave keeps its run 2m and takes the upper one's,
            // the upper half-wave keeps its run 2m + 1 and takes the lower one's
            const uint32_t p0 = pack_bf16x2(tiles[t][8 * m + 0], tiles[t][8 * m + 1]);
            const uint32_t p1 = pack_bf16x2(tiles[t][8 * m + 2], tiles[t][8 * m + 3]);
            const uint32_t q0 = pack_bf16x2(tiles[t][8 * m + 4], tiles[t][8 * m + 5]);
            const uint32_t q1 = pack_bf16x2(tiles[t][8 * m + 6], tiles[t][8 * m + 7]);
            const auto s0 = __builtin_amdgcn_permlane32_swap(p0, q0, false, false);
            const auto s1 = __builtin_amdgcn_permlane32_swap(p1, q1, false, false);
            const uint32_t words[4] = {s0[0], s1[0], s0[1], s1[1]};
            const int c = 32 * t + 16 * m + 8 * half;
            if (l32 < valid_rows && c < valid_cols) {
                if (wide && c + 8 <= valid_cols) {
                    *reinterpret_cast<uint4 *>(row + c) = make_uint4(words[0], words[1], words[2], words[3]);
                } else {
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        if (c + e < valid_cols) {
                            row[c + e] = static_cast<uint16_t>(words[e >> 1] >> (16 * (e & 1)));
                        }
                    }
                }
            }
        }
    }
}

}  // namespace tgo
