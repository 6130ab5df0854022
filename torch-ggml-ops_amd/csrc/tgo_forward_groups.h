// Grouped forward tasks of at most FGR_ROWS rows with scaled fp16 operands: groups of four waves that all unpack and multiply.  Three
// such groups make a workgroup of tgo_forward_scaled.hip's launch, behind its role-split workgroups.
//
// The role-split workgroups unpack with four of their twelve waves, which bounds a task of 64 rows as it does one of 256.  Here a wave
// owns 32 weight rows of the column tile and up to four tiles of 32 activation rows (64 accumulator registers), from the packed blocks
// to the stored results.  Its fp16 weights never leave its registers: the lane that unpacks k-half h of a 32-value block of weight row n
// holds exactly the two matrix-instruction fragments of reduction step 2 * block + h, and one exchange between the half-waves
// (v_permlane32_swap) per register puts them where the instruction wants them; every fragment then serves all row tiles.  The four
// waves share the activation fragments, which they bring to LDS in turn, 8 KiB a stage, rescaled to the row's exponent on the way
// (once per group instead of by each wave that multiplies with them).
// The algebra and the operands are the role-split routine's.  S of a weight row is not scanned for ahead of the row (which would fetch a
// line of every block for four bytes of it) but follows its super-blocks, see FGR_BASE: tasks of more than 32 rows add in the
// role-split routine's order and have its results bit for bit, unless a weight underflows there; tasks of at most 32 rows normalise
// every super-block by itself and add its sums to the row's.
// 256 experts of 2048 x 512 IQ2_S with 128 rows each, gate and up: 0.64 PFLOP/s (0.53 by role-split tasks); under that load the chip's
// clock is below 2 GHz (counted cycles over traced time), and neither the order of a stage's instructions nor 64 weight rows per wave (half the fragment reads, two
// waves per SIMD) changed the time.
#pragma once

#include <type_traits>

#include "tgo_device.h"
#include "tgo_forward_args.h"
#include "tgo_launch.h"
#include "tgo_scaled_operand.h"

namespace tgo {

constexpr int FGR_WAVES = 4;
constexpr int FGR_ROWS = FORWARD_LATE_ROWS;
constexpr int FGR_GROUPS = 3;   // in a workgroup
constexpr int FGR_SPIN_LIMIT = 1 << 20;   // polls of the group's counters before a wave gives up waiting (a few hundred ms)

// The four waves of a group meet through counters in LDS (LDS executes a wave's accesses in issue order: a count written after the data,
// or after the last read, needs no wait of its own): the groups of a workgroup run side by side like workgroups of their own, which the
// workgroup's barrier would hold in step.  A wave that has polled FGR_SPIN_LIMIT times stops waiting, so that a lost count ends in wrong
// results rather than in a workgroup that never finishes.
struct GroupBarrier {
    typedef int i32x4_t __attribute__((ext_vector_type(4)));
    int * arrived;
    int count, seen;
    __device__ __forceinline__ void arrive(int lane, int wave) {
        ++count;
        asm volatile("" ::: "memory");   // (the data accesses stay before the count)
        if (lane == 0) {
            *(volatile __attribute__((address_space(3))) int *)&arrived[wave] = count;
        }
    }
    // until every wave has arrived as often as this one
    __device__ __forceinline__ void wait() {
        if (seen < count) {
            for (int polls = 0; polls < FGR_SPIN_LIMIT; ++polls) {
                const i32x4_t v = *(const volatile __attribute__((address_space(3))) i32x4_t *)arrived;
                seen = __builtin_amdgcn_readfirstlane(min(min(v.x, v.y), min(v.z, v.w)));
                if (seen >= count) {
                    break;
                }
                __builtin_amdgcn_s_sleep(1);
            }
        }
        asm volatile("" ::: "memory");   // (the data accesses stay after the count)
    }
};

// Blocks of 32 values per stage: the activation fragments of a stage are 8 KiB
template <int R> constexpr int group_stage_blocks() { return R == 1 ? 4 : R == 2 ? 2 : 1; }

template <int TYPE>
struct GroupLds {
    alignas(16) uint8_t raw[FGR_WAVES][32 * ScaledSlot<TYPE>::BYTES];   // per wave: the packed blocks of one super-block
    alignas(16) uint8_t x[2][8 * 1024];                                     // activation fragments of two stages
    alignas(16) uint8_t sums[ScaledSlot<TYPE>::K45 ? 4 * 512 : 16];         // block sums of the super-block, per row tile
    alignas(16) float column_power[FGR_WAVES][32];                      // 2^S of the wave's weight rows, or what S grew by
    alignas(16) float row_power[FGR_ROWS];                         // 2^E of the task's rows
    alignas(16) int arrived[FGR_WAVES];                                 // stages that each wave is done with
    int next_chunk;                                                     // the chunk of column tiles that the group has taken
    std::conditional_t<TYPE == IQ2_S, Iq2sSelectors, uint2> codebook;
};

// S puts the largest possible weight of a super-block in [2^FGR_BASE, 2^(FGR_BASE + 1)), as the role-split routine does for a row's
// largest (Q4_K/Q5_K's -1024 * scale allows no more).
//  - R = 1: every super-block has an S of its own, and no weight loses bits to a larger super-block of its row; 2^S of the super-block
//    goes into the multiply-add that joins its sums to the row's.
//  - R > 1: S is that of the largest super-block so far, and where it grows the sums so far are divided accordingly (a power of two):
//    a weight never has fewer bits than under the row's maximum, which costs 16 R multiplications in the few super-blocks that bring
//    one of the wave's 32 rows a new one.
// Against one S from a row's first super-block with room of 2^4 to grow, in which weights 2^14 below the row's largest lost bits: a
// prefill layer of 2048 tokens, 256 experts 354.7 -> 355.7 us, a training layer of 4096 tokens 1167 -> 1173.
constexpr int FGR_BASE = 8;

template <int TYPE, bool WIDE, int R>
TGO_DEVICE void group_task(const ForwardArgs & a, GroupLds<TYPE> & lds, GroupBarrier & barrier, const int tid, int expert, int row_start,
                           int row_end, int tile_first, int tile_count) {
    using F = Format<TYPE>;
    constexpr bool K45 = TYPE == Q4_K || TYPE == Q5_K;
    constexpr int BS = group_stage_blocks<R>();
    constexpr int STAGES = 8 / BS;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31;
    const int half = lane >> 5;
    const int super_blocks = a.in_features / QK_K;
    const int blocks_per_row = a.in_features / 32;

    // ---- packed blocks
    constexpr int RAW_UNITS = K45 ? F::BLOCK_BYTES / 16 : 1;
    constexpr int RAW_REGS = K45 ? (32 * RAW_UNITS + 63) / 64 : 1;
    using W = WideStage<TYPE>;
    constexpr int WIDE_REGS = WIDE ? W::template regs<32, 64>() : 1;
    constexpr int SLOT_PITCH = K45 ? F::BLOCK_BYTES : (WIDE ? W::PITCH : F::RAW_PITCH);
    constexpr int SLOT_FRONT = K45 ? 0 : (WIDE ? W::FRONT : F::RAW_SHIFT);
    uint8_t * const slot = lds.raw[wave];
    struct Cursor {
        int tile, kb;
        const uint8_t * weights;
        const uint8_t * rows;
        int n0, rows_valid;
    };
    auto open = [&](Cursor & c, int tile) {
        c.tile = tile;
        c.kb = 0;
        const bool second = tile >= a.n_tiles;
        c.weights = (second ? a.packed_second : a.packed) + static_cast<int64_t>(expert) * a.bytes_per_expert;
        c.n0 = (second ? tile - a.n_tiles : tile) * FWD_TN + 32 * wave;
        c.rows_valid = max(1, min(32, a.out_features - c.n0));
        c.rows = c.weights + static_cast<int64_t>(min(c.n0, a.out_features - 1)) * a.row_bytes;
    };
    auto step = [&](Cursor & c) {
        if (c.kb + 1 < super_blocks) {
            ++c.kb;
        } else if (c.tile + 1 < tile_first + tile_count) {
            open(c, c.tile + 1);
        }
    };
    struct RawSet {
        u32x4_t units[RAW_REGS];
        WideRegs<WIDE_REGS> wide;
    };
    RawSet pending;
    auto request = [&](const Cursor & c) __attribute__((always_inline)) {
        const int lane = lane_afresh();
        if constexpr (K45) {
            const uint8_t * base = c.rows + static_cast<int64_t>(c.kb) * F::BLOCK_BYTES;
#pragma unroll
            for (int i = 0; i < RAW_REGS; ++i) {
                const int id = min(lane + 64 * i, 32 * RAW_UNITS - 1);
                const int row = id / RAW_UNITS;
                const int unit = id - row * RAW_UNITS;
                const uint32_t offset = __umul24(min(row, c.rows_valid - 1), static_cast<uint32_t>(a.row_bytes)) + unit * 16;
                pending.units[i] = *reinterpret_cast<const u32x4_t *>(base + offset);
            }
        } else if constexpr (WIDE) {
            wide_fetch<TYPE, 32, 64, WIDE_REGS>(pending.wide, c.rows, static_cast<int>(a.row_bytes), c.rows_valid, c.kb, lane);
        }
    };
    auto park = [&](const Cursor & c) __attribute__((always_inline)) {
        const int lane = lane_afresh();
        asm volatile("" ::: "memory");
        if constexpr (K45) {
#pragma unroll
            for (int i = 0; i < RAW_REGS; ++i) {
                const int id = min(lane + 64 * i, 32 * RAW_UNITS - 1);
                *reinterpret_cast<u32x4_t *>(slot + id * 16) = pending.units[i];
            }
        } else if constexpr (WIDE) {
            wide_park<TYPE, 32, 64, WIDE_REGS>(slot, pending.wide, c.rows, static_cast<int>(a.row_bytes), c.rows_valid, c.kb, lane);
        } else {
            stage_blocks<TYPE>(slot, c.weights, a.row_bytes, min(c.n0, a.out_features - 1), a.out_features, c.kb, 32, lane, 64);
        }
        asm volatile("" ::: "memory");
    };

    // ---- activations: a stage is 2 R BS fragments of 1 KiB, fragment f = block (f / 2R), reduction step (f / R) % 2, row tile f % R;
    // wave w brings fragments w and w + 4
    constexpr int FRAGMENTS = 2 * R * BS;
    constexpr int NX = (FRAGMENTS + FGR_WAVES - 1) / FGR_WAVES;
    const int first_tile = row_start >> 5;
    const uint8_t * const x_base = reinterpret_cast<const uint8_t *>(a.qx) + static_cast<int64_t>(first_tile) * blocks_per_row * 2048;
    const uint8_t * const sums_base = reinterpret_cast<const uint8_t *>(a.block_sums) + static_cast<int64_t>(first_tile) * super_blocks * 512;
    // (R = 1, 2, 4: all fragments of a wave are of one row tile)
    constexpr int NT = FGR_WAVES % R == 0 ? 1 : NX;
    uint32_t x_lane[NT], power_lane[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) {
        const int f = wave + FGR_WAVES * i;
        int first = row_start + 32 * (f % R) + l32;
        first = first < a.rows_padded ? first : a.rows_padded - 1;
        x_lane[i] = static_cast<uint32_t>((first >> 5) - first_tile) * blocks_per_row * 2048u + static_cast<uint32_t>(((first & 31) + 32 * half) * 16) +
                    min(f / R, 2 * BS - 1) * 1024u;
        power_lane[i] = static_cast<uint32_t>(first) * 4u;
    }
    const auto fragment_offset = [&](int i) __attribute__((always_inline)) {
        return NT == 1 ? x_lane[0] + i * (FGR_WAVES / R) * 1024u : x_lane[NT == 1 ? 0 : i];
    };
    int sums_row = row_start + 32 * (wave % R) + l32;
    sums_row = sums_row < a.rows_padded ? sums_row : a.rows_padded - 1;
    const uint32_t sums_lane = static_cast<uint32_t>((sums_row >> 5) - first_tile) * super_blocks * 512u + static_cast<uint32_t>((sums_row & 31) * 16);
    struct Incoming {
        half8_t x[NX];
    };
    auto load_x = [&](int kb, int stage) __attribute__((always_inline)) {
        Incoming in;
#pragma unroll
        for (int i = 0; i < NX; ++i) {
            in.x[i] = *reinterpret_cast<const half8_t *>(x_base + static_cast<int64_t>(kb * 16 + 2 * BS * stage) * 1024 + fragment_offset(i));
        }
        return in;
    };
    struct Ratio {
        float r[NT];
        uint4 sums;
    };
    auto load_ratio = [&](int kb) __attribute__((always_inline)) {
        Ratio out;
        const uint8_t * base = reinterpret_cast<const uint8_t *>(a.power + static_cast<int64_t>(kb) * a.rows_padded);
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            out.r[i] = *reinterpret_cast<const float *>(base + power_lane[i]);
        }
        out.sums = make_uint4(0, 0, 0, 0);
        if constexpr (K45) {
            out.sums = *reinterpret_cast<const uint4 *>(sums_base + static_cast<int64_t>(kb) * 512 + sums_lane);
        }
        return out;
    };
    auto rescale = [&](uint4 words, float ratio) __attribute__((always_inline)) {
        const half2_t h = {static_cast<_Float16>(ratio), static_cast<_Float16>(ratio)};
        return make_uint4(half2_mul(words.x, h), half2_mul(words.y, h), half2_mul(words.z, h), half2_mul(words.w, h));
    };
    auto publish = [&](const Incoming & in, const Ratio & ratio, int buffer) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NX; ++i) {
            const int f = wave + FGR_WAVES * i;
            if (FRAGMENTS % FGR_WAVES == 0 || f < FRAGMENTS) {
                *reinterpret_cast<uint4 *>(&lds.x[buffer][f * 1024 + lane * 16]) = rescale(__builtin_bit_cast(uint4, in.x[i]), ratio.r[NT == 1 ? 0 : i]);
            }
        }
    };
    auto publish_sums = [&](const Ratio & ratio) __attribute__((always_inline)) {
        if constexpr (K45) {
            // (fragment i = 0 is of row tile wave % R)
            if (wave < R && half == 0) {
                *reinterpret_cast<uint4 *>(&lds.sums[wave * 512 + l32 * 16]) = rescale(ratio.sums, ratio.r[0]);
            }
        }
    };

    const v16f zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    constexpr bool APART = R == 1;   // super-blocks normalised by themselves
    v16f acc[R];                     // (APART: of the super-block)
    v16f row_sums = zero;            // APART: sum over the super-blocks so far of 2^S * acc
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = zero;

    // ---- unpacking
    struct Row {
        u32x4_t header;
        uint32_t plane_word[4];
        u32x4_t nibbles;
        float scale;
        int exponent;    // biased exponent that S of the lane's weight row stands for
        float shrink;    // 2^-S
    };
    Row row;
    const uint8_t * const blk = slot + l32 * SLOT_PITCH + SLOT_FRONT;
    // Reads the super-block's scales.  Returns whether S of some row changes, after leaving in LDS what the row's sums have to be
    // multiplied with (`fresh`: there are none yet).
    auto open_super_block = [&](bool fresh) __attribute__((always_inline)) {
        Row & w = row;
        float reach;
        if constexpr (K45) {
            w.header = *reinterpret_cast<const u32x4_t *>(blk);
            if constexpr (TYPE == Q5_K) {
                const u32x4_t planes = *reinterpret_cast<const u32x4_t *>(blk + 16 + 16 * half);
                w.plane_word[0] = planes.x; w.plane_word[1] = planes.y; w.plane_word[2] = planes.z; w.plane_word[3] = planes.w;
            }
            reach = fmaxf(fabsf(half_bits_to_float(w.header.x & 0xffffu)) * weight_reach<TYPE>(),
                          fabsf(half_bits_to_float(w.header.x >> 16)) * 63.0f);
        } else {
            reach = fabsf(half_bits_to_float(lds_u16(blk + scale_offset<TYPE>()))) * weight_reach<TYPE>();
        }
        int exponent = static_cast<int>(__float_as_uint(reach) >> 23);
        exponent = min(max(exponent, 9), 254);
        const bool grow = fresh || APART || exponent > w.exponent;
        bool changed = false;
        if (__any(grow)) {
            if (!fresh && !APART) {
                changed = true;
                if (half == 0) {
                    lds.column_power[wave][l32] = grow ? __uint_as_float(static_cast<uint32_t>(max(127 + w.exponent - exponent, 0)) << 23) : 1.0f;
                }
            }
            if (grow) {
                w.exponent = exponent;
                w.shrink = __uint_as_float(static_cast<uint32_t>(254 + FGR_BASE - exponent) << 23);
            }
        }
        w.scale = (K45 ? half_bits_to_float(w.header.x & 0xffffu) : half_weight_scale<TYPE>(blk)) * w.shrink;
        return changed;
    };
    // block B of the super-block -> the two matrix-instruction fragments of the 32 weight rows
    struct Weights {
        half8_t step[2];
    };
    auto unpack = [&](auto block_tag) __attribute__((always_inline)) {
        constexpr int B = decltype(block_tag)::value;
        Row & w = row;
        uint32_t values[8];
        if constexpr (K45) {
            constexpr int QS = TYPE == Q4_K ? 16 : 48;
            if constexpr ((B & 1) == 0) {
                w.nibbles = *reinterpret_cast<const u32x4_t *>(blk + QS + (B >> 1) * 32 + 16 * half);
            }
            int sc, mn;
            k45_group_scale_min<B>(w.header.y, w.header.z, w.header.w, sc, mn);
            const HalfScale half_scales = half_scale_of(w.scale * static_cast<float>(sc));
            const uint32_t word[4] = {w.nibbles.x, w.nibbles.y, w.nibbles.z, w.nibbles.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                uint32_t bytes = (word[i] >> ((B & 1) * 4)) & 0x0f0f0f0fu;
                if constexpr (TYPE == Q5_K) {
                    bytes |= (B <= 4 ? w.plane_word[i] << (B <= 4 ? 4 - B : 0) : w.plane_word[i] >> (B > 4 ? B - 4 : 0)) & 0x10101010u;
                }
                scaled_halves(bytes, half_scales, values[2 * i], values[2 * i + 1]);
            }
        } else {
            decode16_scaled<TYPE>(blk, 2 * B + half, &lds.codebook, w.scale, values);
        }
        // the lane has 16 values of its weight row, k-half `half` of the block: registers 0-3 and 4-7 are the fragments of
        // reduction step `half`; the half-waves exchange what the other one multiplies
        uint32_t first[4], other[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const auto swapped = __builtin_amdgcn_permlane32_swap(values[i], values[4 + i], false, false);
            first[i] = swapped[0];
            other[i] = swapped[1];
        }
        Weights out;
        out.step[0] = __builtin_bit_cast(half8_t, make_uint4(first[0], first[1], first[2], first[3]));
        out.step[1] = __builtin_bit_cast(half8_t, make_uint4(other[0], other[1], other[2], other[3]));
        return out;
    };
    // the extra reduction step of a Q4_K/Q5_K super-block: block minima x block sums
    auto minima_fragment = [&]() __attribute__((always_inline)) {
        const u32x4_t header = row.header;
        const float minus = -half_bits_to_float(header.x >> 16) * row.shrink;
        uint32_t packed[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float m[2];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int g = 2 * i + e;
                const uint32_t mn = g < 4 ? (header.z >> (8 * (g & 3))) & 63u
                                          : ((header.w >> (8 * (g & 3) + 4)) & 15u) | (((header.z >> (8 * (g & 3) + 6)) & 3u) << 4);
                m[e] = minus * static_cast<float>(static_cast<int>(mn));
            }
            const half2_t pair = {static_cast<_Float16>(m[0]), static_cast<_Float16>(m[1])};
            packed[i] = half != 0 ? 0u : __builtin_bit_cast(uint32_t, pair);
        }
        return __builtin_bit_cast(half8_t, make_uint4(packed[0], packed[1], packed[2], packed[3]));
    };
    // sums[4 j + e] *= of_row * lds.column_power[its weight row]
    auto scale_sums = [&](v16f & sums, float of_row, int half_here) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float4 power = *reinterpret_cast<const float4 *>(&lds.column_power[wave][8 * j + 4 * half_here]);
            sums[4 * j + 0] *= of_row * power.x;
            sums[4 * j + 1] *= of_row * power.y;
            sums[4 * j + 2] *= of_row * power.z;
            sums[4 * j + 3] *= of_row * power.w;
        }
    };

    // ---- start
    Cursor ahead;   // of the packed blocks in flight
    open(ahead, tile_first);
    request(ahead);
    Ratio ratio = load_ratio(0);
    constexpr bool DEEP = R < 4;   // activation fragments two stages ahead in registers instead of one
    Incoming x_stage0 = load_x(0, 0), x_a = load_x(0, 1), x_b = {};
    if constexpr (DEEP) {
        x_b = load_x(STAGES > 2 ? 0 : (super_blocks > 1 ? 1 : 0), STAGES > 2 ? 2 : 0);
    }
    if (tid < 32 * R) {
        lds.row_power[tid] = a.row_power[min(row_start + tid, a.rows_padded - 1)];
    }
    park(ahead);
    publish(x_stage0, ratio, 0);
    publish_sums(ratio);
    Ratio ratio_next = ratio;
    open_super_block(true);
    barrier.arrive(lane, wave);   // (stage 0 is published)
    const int total = tile_count * super_blocks;
    int kb = 0, tile = tile_first;
#pragma unroll 1
    for (int q = 0; q < total; ++q) {
        const int kb_next = kb + 1 < super_blocks ? kb + 1 : 0;
        const int kb_after = kb_next + 1 < super_blocks ? kb_next + 1 : 0;
        auto stage = [&](auto stage_tag) __attribute__((always_inline)) {
            constexpr int S = decltype(stage_tag)::value;
            auto block = [&](auto block_tag) __attribute__((always_inline)) {
                constexpr int OF_STAGE = decltype(block_tag)::value;
                constexpr int B = S * BS + OF_STAGE;
                const Weights w = unpack(std::integral_constant<int, B>{});
                if constexpr (OF_STAGE == 0) {
                    // (the weights are unpacked before the wait: the counters' round trip through LDS passes beside them)
                    __builtin_amdgcn_sched_barrier(0);
                    barrier.wait();   // stage S is published, and every wave is done with stage S - 1
                    publish(x_a, S == STAGES - 1 ? ratio_next : ratio, (S + 1) & 1);
                    if constexpr (S == STAGES - 1) {
                        publish_sums(ratio_next);
                    }
                    if constexpr (DEEP) {
                        x_a = x_b;
                    }
                    constexpr int AHEAD = DEEP ? 3 : 2;
                    Incoming & x_new = DEEP ? x_b : x_a;
                    x_new = S + AHEAD < STAGES ? load_x(kb, S + AHEAD)
                            : S + AHEAD - STAGES < STAGES ? load_x(kb_next, S + AHEAD - STAGES)
                                                          : load_x(kb_after, S + AHEAD - 2 * STAGES);
                    if constexpr (S == 0) {
                        ratio_next = load_ratio(kb_next);
                        step(ahead);
                        request(ahead);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                half8_t x[R];
                const auto read_step = [&](int step, int r) __attribute__((always_inline)) {
                    x[r] = *reinterpret_cast<const half8_t *>(&lds.x[S & 1][((OF_STAGE * 2 + step) * R + r) * 1024 + lane * 16]);
                };
#pragma unroll
                for (int r = 0; r < R; ++r) read_step(0, r);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    acc[r] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w.step[0], x[r], acc[r], 0, 0, 0);
                    read_step(1, r);
                }
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (OF_STAGE == BS - 1 && !(K45 && B == 3)) {
                    barrier.arrive(lane, wave);
                }
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    acc[r] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w.step[1], x[r], acc[r], 0, 0, 0);
                }
                if constexpr (K45 && B == 3) {
                    const half8_t minima = minima_fragment();
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        uint4 sums = *reinterpret_cast<const uint4 *>(&lds.sums[r * 512 + l32 * 16]);
                        if (half != 0) {
                            sums = make_uint4(0, 0, 0, 0);
                        }
                        acc[r] = __builtin_amdgcn_mfma_f32_32x32x16_f16(minima, __builtin_bit_cast(half8_t, sums), acc[r], 0, 0, 0);
                    }
                    if constexpr (OF_STAGE == BS - 1) {
                        barrier.arrive(lane, wave);
                    }
                }
            };
            block(std::integral_constant<int, 0>{});
            if constexpr (BS > 1) block(std::integral_constant<int, 1>{});
            if constexpr (BS > 2) { block(std::integral_constant<int, 2>{}); block(std::integral_constant<int, 3>{}); }
        };
        stage(std::integral_constant<int, 0>{});
        stage(std::integral_constant<int, 1>{});
        if constexpr (STAGES > 2) { stage(std::integral_constant<int, 2>{}); stage(std::integral_constant<int, 3>{}); }
        if constexpr (STAGES > 4) {
            stage(std::integral_constant<int, 4>{}); stage(std::integral_constant<int, 5>{});
            stage(std::integral_constant<int, 6>{}); stage(std::integral_constant<int, 7>{});
        }
        park(ahead);   // (everything of this super-block has been read from the slot)
        ratio = ratio_next;
        kb = kb_next;
        if (APART || kb == 0) {
            if (half == 0) {
                lds.column_power[wave][l32] = __uint_as_float(static_cast<uint32_t>(row.exponent - FGR_BASE) << 23);
            }
            asm volatile("" ::: "memory");
        }
        if constexpr (APART) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float4 power = *reinterpret_cast<const float4 *>(&lds.column_power[wave][8 * j + 4 * half]);
                row_sums[4 * j + 0] = __builtin_fmaf(acc[0][4 * j + 0], power.x, row_sums[4 * j + 0]);
                row_sums[4 * j + 1] = __builtin_fmaf(acc[0][4 * j + 1], power.y, row_sums[4 * j + 1]);
                row_sums[4 * j + 2] = __builtin_fmaf(acc[0][4 * j + 2], power.z, row_sums[4 * j + 2]);
                row_sums[4 * j + 3] = __builtin_fmaf(acc[0][4 * j + 3], power.w, row_sums[4 * j + 3]);
            }
            acc[0] = zero;
            asm volatile("" ::: "memory");
        }
        if (kb == 0) {
            // the item is complete: scale by 2^(E[r] + S[n]) (APART: the sums have their 2^S) and store
            const bool second = tile >= a.n_tiles;
            const int n0 = (second ? tile - a.n_tiles : tile) * FWD_TN + 32 * wave;
            uint16_t * const y = second ? a.y_second : a.y;
            const int lane_here = lane_afresh();
            const int l32_here = lane_here & 31, half_here = lane_here >> 5;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int first = row_start + 32 * r;
                if (first < row_end) {
                    if constexpr (APART) {
#pragma unroll
                        for (int v = 0; v < 16; ++v) {
                            acc[r][v] = row_sums[v] * lds.row_power[l32_here];
                        }
                    } else {
                        scale_sums(acc[r], lds.row_power[32 * r + l32_here], half_here);
                    }
                    store_rows_32xn<1>(&acc[r], y + static_cast<int64_t>(first) * a.out_stride + n0, a.out_stride, row_end - first,
                                       a.out_features - n0, lane_here);
                    __builtin_amdgcn_sched_barrier(0);
                }
                acc[r] = zero;
            }
            row_sums = zero;
            asm volatile("" ::: "memory");
            ++tile;
        }
        if (open_super_block(kb == 0)) {
            // (a super-block far above those before it: the sums so far are brought to the new S)
            asm volatile("" ::: "memory");
#pragma unroll
            for (int r = 0; r < R; ++r) {
                scale_sums(acc[r], 1.0f, half);
            }
            asm volatile("" ::: "memory");
        }
    }
}

// `tid`: the thread's index in its group of FGR_WAVES waves; `group`: which of the groups that share the workgroup this is; `blocks`
// workgroups run such groups.
template <int TYPE, bool WIDE>
TGO_DEVICE void group_tasks(const ForwardArgs & a, GroupLds<TYPE> & lds, const int tid, const int group, const int blocks) {
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    if constexpr (TYPE == IQ2_S) {
        expand_iq2s_selectors(lds.codebook, tid, 64 * FGR_WAVES);
    }
    if (tid < FGR_WAVES) {
        lds.arrived[tid] = 0;
    }
    __syncthreads();   // (of the whole workgroup: its groups are still in step here, and part ways behind it)
    GroupBarrier barrier = {lds.arrived, 0, 0};
    const int tasks = a.task_count[0];
    const int first_late = min(a.task_early[0], tasks);
    const int total_tiles = a.n_tiles * a.projections;
    // A chunk: column tiles of one task, eight super-blocks of work where that leaves a chunk for every group of the chip, else four.
    // Each of the TASK_CURSORS lists holds a contiguous eighth of the chunks, so that a task's activations and an expert's weights stay
    // with the workgroups of one XCD; its cursor counts the chunks taken from it.  (Atomic operations on one address complete one after
    // the other, at some tens of nanoseconds each.)  A group starts with the list of its workgroup's number and goes on to the others
    // when that is used up.
    const int late = tasks - first_late;
    const int super_blocks = a.in_features / QK_K;
    int run = max(1, 8 / super_blocks);
    if (static_cast<int64_t>(late) * ((total_tiles + run - 1) / run) < blocks * FGR_GROUPS) {
        run = max(1, 4 / super_blocks);
    }
    const int per_task = (total_tiles + run - 1) / run;
    const int chunks = late * per_task;
    const int home = static_cast<int>(blockIdx.x) % TASK_CURSORS;
    const int blocks_per_list = max(1, blocks / TASK_CURSORS);
    bool started = false;
#pragma unroll 1
    for (;;) {
        if (tid == 0) {
            int chunk = -1;
            for (int k = 0; k < TASK_CURSORS && chunk < 0; ++k) {
                const int list = (home + k) % TASK_CURSORS;
                int32_t * const cursor = a.task_cursor + list * TASK_CURSOR_STRIDE;
                const int list_first = static_cast<int>(static_cast<int64_t>(chunks) * list / TASK_CURSORS);
                const int in_list = static_cast<int>(static_cast<int64_t>(chunks) * (list + 1) / TASK_CURSORS) - list_first;
                // Three groups on a CU each take more than twice as long as one that is alone there.  So a list that does not fill the
                // chip goes one or two to a CU, and towards a list's end (an estimate of what is left decides, the count itself is
                // exact) the later groups of the workgroups stop: the first ones, one more chunk each, finish it.
                const int left = in_list - __hip_atomic_load(cursor, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (left > 0 && (started ? left : in_list) > group * blocks_per_list) {
                    const int taken = atomicAdd(cursor, 1);
                    if (taken < in_list) {
                        chunk = list_first + taken;
                    }
                }
            }
            *(volatile __attribute__((address_space(3))) int *)&lds.next_chunk = chunk;
        }
        barrier.arrive(lane, wave);   // (and every wave is done with the chunk before)
        barrier.wait();
        const int chunk = __builtin_amdgcn_readfirstlane(*(const volatile __attribute__((address_space(3))) int *)&lds.next_chunk);
        if (chunk < 0) {
            break;
        }
        started = true;
        const int task = first_late + chunk / per_task;
        const int tile_first = chunk % per_task * run;
        const int tile_count = min(run, total_tiles - tile_first);
        const int expert = __builtin_amdgcn_readfirstlane(a.task_expert[task]);
        const int row_start = __builtin_amdgcn_readfirstlane(a.task_row_start[task]);
        const int row_end = __builtin_amdgcn_readfirstlane(a.task_row_end[task]);
        const int rows = row_end - row_start;
        if (rows > 96) {
            group_task<TYPE, WIDE, 4>(a, lds, barrier, tid, expert, row_start, row_end, tile_first, tile_count);
        } else if (rows > 64) {
            group_task<TYPE, WIDE, 3>(a, lds, barrier, tid, expert, row_start, row_end, tile_first, tile_count);
        } else if (rows > 32) {
            group_task<TYPE, WIDE, 2>(a, lds, barrier, tid, expert, row_start, row_end, tile_first, tile_count);
        } else {
            group_task<TYPE, WIDE, 1>(a, lds, barrier, tid, expert, row_start, row_end, tile_first, tile_count);
        }
    }
}

}  // namespace tgo
