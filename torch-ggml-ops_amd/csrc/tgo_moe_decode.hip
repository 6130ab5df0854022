// A mixture-of-experts layer of a few tokens in two launches, without a sorted list of its slots.
//
// Routing, quantizing, gate and up, SwiGLU, down and combine were five or six dependent launches of 2 to 20 us whose time is not the packed
// bytes (6 tokens x 8 of 256 experts, 66 MB: 13 us of memory time in 53 us) but each launch's chain of round trips: the group list, the row
// index, the activations, the weights, one after the other, in two rounds of workgroups.  Here a workgroup finds what it needs from the
// choices themselves, has all its weights in flight at once, and is small enough for the whole layer to be resident together:
//
// 6 tokens x 8 of 256 experts of 2048 x 512, IQ2_S and Q6_K, in a graph: 50.9 -> 31.5 us a layer; one token called from Python 21.8 -> 10.9.
//
//   moe_gate_up_kernel   one (slot, eight rows of gate and of up): the first slot of an expert takes the expert's other slots along, two at
//                        a time, so that its weights are read once; activated = silu(gate) * up, both rounded to bf16 first
//   moe_down_kernel      one (token, eight columns): the token's experts side by side as one reduction of top_k x intermediate values, whose
//                        activations carry the routing weights; the sum over the experts is the reduction's own and rounded once
//
// A wave loads its weight rows as 16-byte pieces at their own addresses (BlockPieces), through registers into LDS of its own, and multiplies
// with the q8_1 activations that the workgroup quantizes meanwhile; arithmetic as in tgo_gemv.hip.
#include <algorithm>
#include <type_traits>

#include "tgo_device.h"
#include "tgo_launch.h"

namespace tgo {

constexpr int MDE_THREADS = 256;
constexpr int MDE_WAVES = MDE_THREADS / 64;
constexpr int MDE_COLUMNS = 2 * MDE_WAVES;   // weight rows of a projection per workgroup, two per wave
constexpr int MDE_MAX_SLOTS = MOE_DECODE_SLOTS;
static_assert(MDE_MAX_SLOTS <= 64, "a slot per lane");

// IQ2_S: the codebook's magnitudes as bytes, and for a byte of signs 0xff in the bytes to negate.  In memory as the workgroups want them in LDS:
// expanding the packed codebook is 140 vector instructions per wave, a seventh of a gate and up workgroup's.
struct Iq2sBytes {
    uint32_t grid[TGO_IQ2S_GRID_ENTRIES][2];
    uint32_t sign[256][2];
};
constexpr Iq2sBytes iq2s_bytes_of_packed() {
    Iq2sBytes t = {};
    for (int i = 0; i < TGO_IQ2S_GRID_ENTRIES; ++i) {
        for (int e = 0; e < 8; ++e) {
            const uint32_t digit = (tgo_iq2s_packed[i] >> (2 * e)) & 3u;
            t.grid[i][e / 4] |= (8u + 17u * digit + (digit >> 1)) << (8 * (e % 4));
        }
    }
    for (int i = 0; i < 256; ++i) {
        for (int e = 0; e < 8; ++e) {
            t.sign[i][e / 4] |= ((i >> e) & 1) != 0 ? 0xffu << (8 * (e % 4)) : 0u;
        }
    }
    return t;
}
static constexpr __device__ __attribute__((aligned(16))) Iq2sBytes iq2s_bytes = iq2s_bytes_of_packed();
struct Iq2sLds {
    uint2 grid[TGO_IQ2S_GRID_ENTRIES];
    uint2 sign[256];
};
static_assert(sizeof(Iq2sBytes) == sizeof(Iq2sLds) && sizeof(Iq2sLds) % 512 == 0, "copied 16 bytes at a time");
// The thread's share of the tables, requested and written: 640 pieces of 16 bytes for 256 threads.
struct Iq2sRequest {
    u32x4_t piece[3];
    __device__ __forceinline__ void request(int tid) {
        const u32x4_t * const from = reinterpret_cast<const u32x4_t *>(&iq2s_bytes);
        piece[0] = from[tid];
        piece[1] = from[tid + 256];
        piece[2] = from[512 + (tid & 127)];
    }
    __device__ __forceinline__ void write(Iq2sLds & tables, int tid) const {
        u32x4_t * const to = reinterpret_cast<u32x4_t *>(&tables);
        to[tid] = piece[0];
        to[tid + 256] = piece[1];
        if (tid < 128) {
            to[512 + tid] = piece[2];
        }
    }
};

TGO_DEVICE int mde_dot4(uint32_t a, uint32_t b, int c) { return __builtin_amdgcn_sdot4(static_cast<int>(a), static_cast<int>(b), c, false); }

// ---- a lane's share of a super-block ---------------------------------------------------------------------------------
// Q3_K, Q6_K, IQ2_S: 16 consecutive values (16 lanes per super-block); Q4_K / Q5_K: 16 values each of two neighbouring 32-value groups,
// which share their bytes (8 lanes).
template <int TYPE>
struct LaneUnit {
    static constexpr bool K45 = TYPE == Q4_K || TYPE == Q5_K;
    static constexpr int PER_BLOCK = K45 ? 8 : 16;
    static constexpr int PARTS = K45 ? 2 : 1;   // runs of 16 values
    // first value of run `part` of unit `u` within the super-block
    __device__ __forceinline__ static int first_value(int u, int part) { return K45 ? (u >> 1) * 64 + part * 32 + (u & 1) * 16 : u * 16; }
};

// The activations that meet a unit: quants, block scales, and what the formats' offsets are multiplied with: the sum of the quants, or for
// Q4_K / Q5_K the block's sum (on the first of the two lanes that hold a group).
template <int TYPE>
struct UnitInput {
    uint4 q[LaneUnit<TYPE>::PARTS];
    float d[LaneUnit<TYPE>::PARTS], offset[LaneUnit<TYPE>::PARTS];
};

// `q`: the row's int8 values, `d` and `sum`: fp32 per 32 values, `value`: first value of the unit's super-block
template <int TYPE>
TGO_DEVICE UnitInput<TYPE> unit_input(const int8_t * q, const float * d, const float * sum, int value, int u) {
    using U = LaneUnit<TYPE>;
    UnitInput<TYPE> x;
#pragma unroll
    for (int part = 0; part < U::PARTS; ++part) {
        const int first = value + U::first_value(u, part);
        x.q[part] = *reinterpret_cast<const uint4 *>(q + first);
        x.d[part] = d[first >> 5];
        if constexpr (U::K45) {
            x.offset[part] = (u & 1) == 0 ? sum[first >> 5] : 0.0f;
        } else if constexpr (TYPE != IQ2_S) {
            int total = mde_dot4(0x01010101u, x.q[part].x, 0);
            total = mde_dot4(0x01010101u, x.q[part].y, total);
            total = mde_dot4(0x01010101u, x.q[part].z, total);
            total = mde_dot4(0x01010101u, x.q[part].w, total);
            x.offset[part] = static_cast<float>(total);
        }
    }
    return x;
}

TGO_DEVICE int dot16(const uint32_t (&w)[4], const uint4 q) {
    int dot = mde_dot4(w[0], q.x, 0);
    dot = mde_dot4(w[1], q.y, dot);
    dot = mde_dot4(w[2], q.z, dot);
    return mde_dot4(w[3], q.w, dot);
}

// acc[r] += unit `u` of the block at `blk` (BlockPieces order) times row r's activations.
template <int TYPE, int ROWS>
TGO_DEVICE void unit_product(const uint8_t * blk, int u, const Iq2sLds * tables, const UnitInput<TYPE> (&x)[ROWS], float (&acc)[ROWS]) {
    if constexpr (LaneUnit<TYPE>::K45) {
        constexpr int QS = TYPE == Q4_K ? 16 : 48;
        const int pair = u >> 1, half = u & 1;
        const uint4 header = *reinterpret_cast<const uint4 *>(blk);
        const uint4 nibbles = *reinterpret_cast<const uint4 *>(blk + QS + pair * 32 + half * 16);
        const uint32_t word[4] = {nibbles.x, nibbles.y, nibbles.z, nibbles.w};
        uint32_t low[4], high[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            low[t] = word[t] & 0x0f0f0f0fu;
            high[t] = (word[t] >> 4) & 0x0f0f0f0fu;
        }
        if constexpr (TYPE == Q5_K) {
            const uint4 planes = *reinterpret_cast<const uint4 *>(blk + 16 + half * 16);
            const uint32_t plane[4] = {planes.x, planes.y, planes.z, planes.w};
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const uint32_t bits = plane[t] >> (2 * pair);
                low[t] |= (bits & 0x01010101u) << 4;
                high[t] |= (bits << 3) & 0x10101010u;
            }
        }
        // groups 2 pair and 2 pair + 1, 16 bits of each of the scale words
        const int shift = 16 * (pair & 1);
        const uint32_t w1 = header.y >> shift, w2 = header.z >> shift, w3 = header.w >> shift;
        const uint32_t scales = pair < 2 ? w1 & 0x3f3fu : (w3 & 0x0f0fu) | ((w1 >> 2) & 0x3030u);
        const uint32_t minima = pair < 2 ? w2 & 0x3f3fu : ((w3 >> 4) & 0x0f0fu) | ((w2 >> 2) & 0x3030u);
        const float d = half_bits_to_float(header.x & 0xffffu), dmin = half_bits_to_float(header.x >> 16);
        const float s0 = d * static_cast<float>(scales & 0xffu), s1 = d * static_cast<float>(scales >> 8 & 0xffu);
        const float m0 = dmin * static_cast<float>(minima & 0xffu), m1 = dmin * static_cast<float>(minima >> 8 & 0xffu);
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            float sum = acc[r];
            sum = fmaf(s0 * x[r].d[0], static_cast<float>(dot16(low, x[r].q[0])), sum);
            sum = fmaf(s1 * x[r].d[1], static_cast<float>(dot16(high, x[r].q[1])), sum);
            sum = fmaf(-m0, x[r].offset[0], sum);
            acc[r] = fmaf(-m1, x[r].offset[1], sum);
        }
        return;
    } else {
        uint32_t w[4], mask[4];
        float scale, bias = 0.0f;
        if constexpr (TYPE == Q6_K) {
            const uint4 low = *reinterpret_cast<const uint4 *>(blk + (u >> 3) * 64 + (u & 3) * 16);
            const uint4 high = *reinterpret_cast<const uint4 *>(blk + 128 + (u >> 3) * 32 + (u & 1) * 16);
            const int shift_low = u & 4, shift_high = u & 6;   // 4 ((u >> 2) & 1), 2 ((u >> 1) & 3)
            const uint32_t lows[4] = {low.x, low.y, low.z, low.w}, highs[4] = {high.x, high.y, high.z, high.w};
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                w[t] = ((lows[t] >> shift_low) & 0x0f0f0f0fu) | (((highs[t] >> shift_high) & 0x03030303u) << 4);
            }
            scale = half_bits_to_float(lds_u16(blk + 222)) * static_cast<float>(static_cast<int8_t>(blk[192 + u]));
            bias = 32.0f;
        } else if constexpr (TYPE == Q3_K) {
            const uint4 low = *reinterpret_cast<const uint4 *>(blk + 32 + (u >> 3) * 32 + (u & 1) * 16);
            const uint4 high = *reinterpret_cast<const uint4 *>(blk + (u & 1) * 16);
            const int shift_low = u & 6, shift_high = u >> 1;
            const uint32_t lows[4] = {low.x, low.y, low.z, low.w}, highs[4] = {high.x, high.y, high.z, high.w};
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                w[t] = ((lows[t] >> shift_low) & 0x03030303u) | (((highs[t] >> shift_high) & 0x01010101u) << 2);
            }
            // (the last piece starts two bytes into the quants' end: scales from 98, d at 110)
            const int sub = ((blk[98 + (u & 7)] >> (4 * (u >> 3))) & 0x0f) | (((blk[106 + (u & 3)] >> (2 * (u >> 2))) & 3) << 4);
            scale = half_bits_to_float(lds_u16(blk + 110)) * static_cast<float>(sub - 32);
            bias = 4.0f;
        } else {
            const uint32_t idx_pair = lds_u16(blk + 2 * u), sign_pair = lds_u16(blk + 32 + 2 * u);
            const uint32_t qh = blk[64 + (u >> 1)] >> (4 * (u & 1));
            // the magnitudes, those to negate inverted (-m - 1): what is missing to the sum of a row's products is the sum of the
            // activations there, and the masks, bytes of -1, are the operand that gives it
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                const uint2 magnitudes = tables->grid[((idx_pair >> (8 * g)) & 0xffu) | (((qh >> (2 * g)) & 3u) << 8)];
                const uint2 negated = tables->sign[(sign_pair >> (8 * g)) & 0xffu];
                mask[2 * g] = negated.x;
                mask[2 * g + 1] = negated.y;
                w[2 * g] = magnitudes.x ^ negated.x;
                w[2 * g + 1] = magnitudes.y ^ negated.y;
            }
            const int sub = (blk[72 + (u >> 1)] >> (4 * (u & 1))) & 0x0f;
            scale = half_bits_to_float(lds_u16(blk + 80)) * 0.125f * static_cast<float>(2 * sub + 1);
        }
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            float dot;
            if constexpr (TYPE == IQ2_S) {
                dot = static_cast<float>(dot16(w, x[r].q[0]) - dot16(mask, x[r].q[0]));
            } else {
                dot = fmaf(-bias, x[r].offset[0], static_cast<float>(dot16(w, x[r].q[0])));   // (integers below 2^24: exact)
            }
            acc[r] = fmaf(scale * x[r].d[0], dot, acc[r]);
        }
    }
}

// ---- weights: memory -> registers -> the wave's LDS --------------------------------------------------------------------
// One weight row (or several that follow one another) of `blocks` super-blocks; `PIECES` 16-byte pieces per lane at most.
typedef uint32_t u32x4_even_t __attribute__((ext_vector_type(4), aligned(2)));   // blocks start on any even address
template <int TYPE, int PIECES>
struct RowPieces {
    u32x4_t piece[PIECES];   // (a native vector type: arrays of the uint4 struct end up in scratch memory)
    __device__ __forceinline__ void request(const uint8_t * row, int blocks, int lane) {
        using B = BlockPieces<TYPE>;
#pragma unroll
        for (int i = 0; i < PIECES; ++i) {
            if (64 * i < blocks * B::UNITS) {   // uniform
                const int id = min(lane + 64 * i, blocks * B::UNITS - 1);   // (past the end: the last piece again)
                const int block = id / B::UNITS, unit = id - block * B::UNITS;
                const int offset = B::ALIGNED ? 16 * unit
                                   : TYPE == IQ2_S ? (unit == B::UNITS - 1 ? 0 : 2 + 16 * unit)
                                                   : (unit == B::UNITS - 1 ? B::BLOCK - 16 : 16 * unit);
                piece[i] = *reinterpret_cast<const u32x4_even_t *>(row + block * B::BLOCK + offset);
            }
        }
    }
    __device__ __forceinline__ void park(uint8_t * lds, int blocks, int lane) const {
        using B = BlockPieces<TYPE>;
#pragma unroll
        for (int i = 0; i < PIECES; ++i) {
            if (64 * i < blocks * B::UNITS) {
                const int id = min(lane + 64 * i, blocks * B::UNITS - 1);
                const int block = id / B::UNITS, unit = id - block * B::UNITS;
                *reinterpret_cast<u32x4_t *>(lds + block * B::PITCH + unit * 16) = piece[i];
            }
        }
    }
};
template <int TYPE>
constexpr int pieces_per_lane(int blocks) { return (blocks * BlockPieces<TYPE>::UNITS + 63) / 64; }

// Eight values of a row to q8_1 in LDS, by four neighbouring lanes per block.  `scale`: multiplies block scale and sum.
TGO_DEVICE void quantize_to_lds(const uint4 bits, int8_t * q, float * d, float * sum, int value, float scale) {
    float x[8], d_block, total;
    uint32_t packed[2], halves[4];
    int magnitude[8];
    unpack_bf16x8(bits, x);
    quantize_eight(bits, x, packed, d_block, total, halves, magnitude);
    *reinterpret_cast<uint2 *>(q + value) = make_uint2(packed[0], packed[1]);
    if ((value & 31) == 0) {
        d[value >> 5] = d_block * scale;
        sum[value >> 5] = total * scale;
    }
}

// Sum over the wave by data-parallel-primitive additions (no LDS crossbar); the total is lane 63's.
template <int CONTROL, int ROWS>
TGO_DEVICE float dpp_add(float v) {
    return v + __uint_as_float(static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(__float_as_uint(v)), CONTROL, ROWS, 0xf, true)));
}
TGO_DEVICE float wave_sum(float v) {
    v = dpp_add<0x111, 0xf>(v);   // row_shr:1
    v = dpp_add<0x112, 0xf>(v);   // row_shr:2
    v = dpp_add<0x114, 0xf>(v);   // row_shr:4
    v = dpp_add<0x118, 0xf>(v);   // row_shr:8: lane 15 of every row of 16 has its row's sum
    v = dpp_add<0x142, 0xa>(v);   // row_bcast:15 into rows 1 and 3
    return dpp_add<0x143, 0xc>(v);   // row_bcast:31 into rows 2 and 3
}

// The choice of a slot; -1 for none or one that is not an expert.
TGO_DEVICE int choice(const MoeDecodeArgs & a, int slot) {
    const int64_t expert = slot < a.slots ? a.slot_experts[slot] : -1;
    return expert >= 0 && expert < a.experts ? static_cast<int>(expert) : -1;
}

// ---- gate and up -------------------------------------------------------------------------------------------------------
// BLOCKS: super-blocks of K at most.  Bound by latency at a token (7 us), by unpacking at six (IQ2_S, 42 of 256 experts of 2048 x 512: vector
// unit and LDS half of the time each).  Two weight rows of either projection per wave: with four, which spare half of what a workgroup does
// besides unpacking, every size measured slower (6 tokens of 128 experts, 1024 x 512, layer 19.7 -> 23.9 us), as it did with four slots at a
// time instead of two (170 registers instead of 112 with Q4_K: 30.8 -> 33.4).
template <int TYPE, int BLOCKS>
__global__ __launch_bounds__(MDE_THREADS) void moe_gate_up_kernel(const MoeDecodeArgs a) {
    using B = BlockPieces<TYPE>;
    using U = LaneUnit<TYPE>;
    constexpr int PIECES = pieces_per_lane<TYPE>(BLOCKS);
    constexpr int ROW_LDS = BLOCKS * B::PITCH;
    constexpr int VALUES = BLOCKS * QK_K;
    __shared__ __attribute__((aligned(16))) uint8_t raw[MDE_WAVES][4][ROW_LDS];   // gate, gate, up, up
    __shared__ __attribute__((aligned(16))) int8_t xq[2][VALUES];
    __shared__ __attribute__((aligned(16))) float xd[2][VALUES / 32], xs[2][VALUES / 32];
    __shared__ __attribute__((aligned(16))) std::conditional_t<TYPE == IQ2_S, Iq2sLds, uint2> table_lds;
    const Iq2sLds * const tables = reinterpret_cast<const Iq2sLds *>(&table_lds);
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int row_groups = a.intermediate / MDE_COLUMNS;
    const int slot = static_cast<int>(blockIdx.x) / row_groups;
    const int n0 = (static_cast<int>(blockIdx.x) - slot * row_groups) * MDE_COLUMNS + 2 * wave;   // the wave's first weight row
    const int blocks = a.features / QK_K;
    Iq2sRequest table;
    if constexpr (TYPE == IQ2_S) {
        table.request(tid);
    }
    // the slots of this expert, and whether this one is the first of them
    const int own = __builtin_amdgcn_readfirstlane(choice(a, slot));
    const int theirs = choice(a, lane);
    if (own < 0) {
        return;
    }
    uint64_t slots = __ballot(theirs == own);
    if (__builtin_ctzll(slots) != slot) {
        return;
    }
    RowPieces<TYPE, PIECES> weights[4];
    const int64_t row_bytes = static_cast<int64_t>(blocks) * B::BLOCK;
    const int64_t at = (static_cast<int64_t>(own) * a.intermediate + n0) * row_bytes;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        weights[i].request((i < 2 ? a.gate : a.up) + at + (i & 1) * row_bytes, blocks, lane);
    }
    const auto quantize = [&](int of_slot, int row) {
        const uint16_t * const source = a.hidden + static_cast<int64_t>(of_slot / a.top_k) * a.features;
#pragma unroll
        for (int pass = 0; pass < (VALUES + 2047) / 2048; ++pass) {
            const int value = pass * 2048 + tid * 8;
            if (value < a.features) {   // (whole blocks of four lanes)
                quantize_to_lds(*reinterpret_cast<const uint4 *>(source + value), xq[row], xd[row], xs[row], value, 1.0f);
            }
        }
    };
    if constexpr (TYPE == IQ2_S) {
        table.write(table_lds, tid);
    }
    bool parked = false;
    while (slots != 0) {   // two slots at a time
        const int first = __builtin_ctzll(slots);
        slots &= slots - 1;
        const int second = slots != 0 ? __builtin_ctzll(slots) : -1;
        slots &= slots - 1;   // (0 stays 0)
        if (parked) {
            __syncthreads();   // (the activations in LDS have been read)
        }
        quantize(first, 0);
        if (second >= 0) {
            quantize(second, 1);
        }
        if (!parked) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                weights[i].park(raw[wave][i], blocks, lane);
            }
            parked = true;
        }
        __syncthreads();
        const auto multiply = [&](auto rows_tag) __attribute__((always_inline)) {
            constexpr int ROWS = decltype(rows_tag)::value;
            float acc[4][ROWS] = {};
#pragma unroll
            for (int j = 0; j < (BLOCKS * U::PER_BLOCK + 63) / 64; ++j) {
                const int id = lane + 64 * j;
                if (id < blocks * U::PER_BLOCK) {
                    const int block = id / U::PER_BLOCK, u = id % U::PER_BLOCK;
                    UnitInput<TYPE> x[ROWS];
#pragma unroll
                    for (int r = 0; r < ROWS; ++r) {
                        x[r] = unit_input<TYPE>(xq[r], xd[r], xs[r], block * QK_K, u);
                    }
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        unit_product<TYPE, ROWS>(raw[wave][i] + block * B::PITCH, u, tables, x, acc[i]);
                    }
                }
            }
#pragma unroll
            for (int r = 0; r < ROWS; ++r) {
                uint32_t both = 0;
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const uint16_t gate = to_bf16_bits(wave_sum(acc[i][r])), up = to_bf16_bits(wave_sum(acc[2 + i][r]));
                    both |= static_cast<uint32_t>(swiglu_bf16(gate, up)) << (16 * i);
                }
                if (lane == 63) {
                    *reinterpret_cast<uint32_t *>(a.activated + static_cast<int64_t>(r == 0 ? first : second) * a.intermediate + n0) = both;
                }
            }
        };
        if (second >= 0) {
            multiply(std::integral_constant<int, 2>{});
        } else {
            multiply(std::integral_constant<int, 1>{});
        }
    }
}

// ---- down and combine --------------------------------------------------------------------------------------------------
// BLOCKS: super-blocks of the intermediate features, exactly.  Bound by latency (six tokens: 13 us for 41 MB; vector unit 0.30 of the time, LDS 0.27);
// with all eight experts' weights in LDS at once 15.2, in four of six workgroups' worth of it per CU.
template <int TYPE, int BLOCKS>
__global__ __launch_bounds__(MDE_THREADS) void moe_down_kernel(const MoeDecodeArgs a) {
    using B = BlockPieces<TYPE>;
    using U = LaneUnit<TYPE>;
    constexpr int PIECES = pieces_per_lane<TYPE>(2 * BLOCKS);
    constexpr int VALUES = BLOCKS * QK_K;
    constexpr int UNITS = BLOCKS * U::PER_BLOCK;   // of one expert's row
    constexpr int EXPERTS = MOE_DECODE_TOP_K;
    constexpr int AT_ONCE = EXPERTS / 2;   // experts whose weights are in LDS at a time: the workgroups of six tokens are then all resident
    __shared__ __attribute__((aligned(16))) uint8_t raw[MDE_WAVES][AT_ONCE][2 * BLOCKS * B::PITCH];
    __shared__ __attribute__((aligned(16))) int8_t xq[EXPERTS * VALUES];
    __shared__ __attribute__((aligned(16))) float xd[EXPERTS * VALUES / 32], xs[EXPERTS * VALUES / 32];
    __shared__ __attribute__((aligned(16))) std::conditional_t<TYPE == IQ2_S, Iq2sLds, uint2> table_lds;
    const Iq2sLds * const tables = reinterpret_cast<const Iq2sLds *>(&table_lds);
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int column_groups = a.features / MDE_COLUMNS;
    const int token = static_cast<int>(blockIdx.x) / column_groups;
    const int c0 = (static_cast<int>(blockIdx.x) - token * column_groups) * MDE_COLUMNS + 2 * wave;
    const int first_slot = token * a.top_k;
    const int mine = lane < a.top_k ? choice(a, first_slot + lane) : -1;
    const float weight = lane < a.top_k ? a.slot_weights[first_slot + lane] : 0.0f;
    const uint32_t valid = static_cast<uint32_t>(__ballot(mine >= 0));
    constexpr int64_t row_bytes = static_cast<int64_t>(BLOCKS) * B::BLOCK;
    RowPieces<TYPE, PIECES> weights[EXPERTS];
#pragma unroll
    for (int j = 0; j < EXPERTS; ++j) {
        if ((valid >> j & 1) != 0) {   // uniform
            const int expert = __builtin_amdgcn_readlane(mine, j);
            weights[j].request(a.down + (static_cast<int64_t>(expert) * a.features + c0) * row_bytes, 2 * BLOCKS, lane);
        }
    }
    if constexpr (TYPE == IQ2_S) {
        Iq2sRequest table;
        table.request(tid);
        table.write(table_lds, tid);
    }
    // the token's activated rows lie one behind the other (those of slots without an expert were never written)
    const uint16_t * const source = a.activated + static_cast<int64_t>(first_slot) * VALUES;
#pragma unroll
    for (int pass = 0; pass < EXPERTS * VALUES / 2048; ++pass) {
        const int value = pass * 2048 + tid * 8;
        const int j = value / VALUES;
        const float factor = __shfl(weight, j);
        if (j < a.top_k && (valid >> j & 1) != 0) {
            quantize_to_lds(*reinterpret_cast<const uint4 *>(source + value), xq, xd, xs, value, factor);
        }
    }
    __syncthreads();
    float acc[2][1] = {};
    // (lanes read what other lanes of their wave have parked: LDS executes a wave's accesses in order, the compiler has to keep them so)
    const auto wave_sync = [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
#pragma unroll
    for (int first = 0; first < EXPERTS; first += AT_ONCE) {
        if (first != 0) {
            wave_sync();   // the experts before have been read
        }
#pragma unroll
        for (int j = 0; j < AT_ONCE; ++j) {
            if ((valid >> (first + j) & 1) != 0) {
                weights[first + j].park(raw[wave][j], 2 * BLOCKS, lane);
            }
        }
        wave_sync();   // parked
#pragma unroll
        for (int i = 0; i < (AT_ONCE * UNITS + 63) / 64; ++i) {
            const int id = lane + 64 * i;
            const int j = id / UNITS, unit = id - j * UNITS;
            const int block = unit / U::PER_BLOCK, u = unit % U::PER_BLOCK;
            if (j < AT_ONCE && (valid >> (first + j) & 1) != 0) {   // (no bit beyond the token's choices)
                const UnitInput<TYPE> x[1] = {unit_input<TYPE>(xq, xd, xs, (first + j) * VALUES + block * QK_K, u)};
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    unit_product<TYPE, 1>(raw[wave][j] + (c * BLOCKS + block) * B::PITCH, u, tables, x, acc[c]);
                }
            }
        }
    }
    const float sums[2] = {wave_sum(acc[0][0]), wave_sum(acc[1][0])};
    if (lane == 63) {
        *reinterpret_cast<uint32_t *>(a.output + static_cast<int64_t>(token) * a.features + c0) = pack_bf16x2(sums[0], sums[1]);
    }
}

template <int TYPE>
static hipError_t launch_gate_up(const MoeDecodeArgs & a, hipStream_t stream) {
    const unsigned grid = static_cast<unsigned>(a.slots * (a.intermediate / MDE_COLUMNS));
    if (a.features <= 8 * QK_K) {
        moe_gate_up_kernel<TYPE, 8><<<grid, MDE_THREADS, 0, stream>>>(a);
    } else {
        moe_gate_up_kernel<TYPE, 16><<<grid, MDE_THREADS, 0, stream>>>(a);
    }
    return hipGetLastError();
}

template <int TYPE>
static hipError_t launch_down(const MoeDecodeArgs & a, hipStream_t stream) {
    const unsigned grid = static_cast<unsigned>(a.tokens * (a.features / MDE_COLUMNS));
    switch (a.intermediate / QK_K) {
        case 1: moe_down_kernel<TYPE, 1><<<grid, MDE_THREADS, 0, stream>>>(a); break;
        case 2: moe_down_kernel<TYPE, 2><<<grid, MDE_THREADS, 0, stream>>>(a); break;
        case 3: moe_down_kernel<TYPE, 3><<<grid, MDE_THREADS, 0, stream>>>(a); break;
        case 4: moe_down_kernel<TYPE, 4><<<grid, MDE_THREADS, 0, stream>>>(a); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_moe_decode(const MoeDecodeArgs & a, int gate_up_type, int down_type, hipStream_t stream) {
    if (a.slots > MDE_MAX_SLOTS || a.top_k > MOE_DECODE_TOP_K || a.features > 16 * QK_K || a.intermediate > 4 * QK_K || a.features % QK_K != 0 ||
        a.intermediate % QK_K != 0) {
        return hipErrorInvalidValue;
    }
    const ProfileScope scope(5, stream);
    hipError_t status = hipErrorInvalidValue;
    switch (gate_up_type) {
        case Q3_K: status = launch_gate_up<Q3_K>(a, stream); break;
        case Q4_K: status = launch_gate_up<Q4_K>(a, stream); break;
        case Q5_K: status = launch_gate_up<Q5_K>(a, stream); break;
        case Q6_K: status = launch_gate_up<Q6_K>(a, stream); break;
        case IQ2_S: status = launch_gate_up<IQ2_S>(a, stream); break;
        default: break;
    }
    if (status != hipSuccess) {
        return status;
    }
    switch (down_type) {
        case Q3_K: return launch_down<Q3_K>(a, stream);
        case Q4_K: return launch_down<Q4_K>(a, stream);
        case Q5_K: return launch_down<Q5_K>(a, stream);
        case Q6_K: return launch_down<Q6_K>(a, stream);
        case IQ2_S: return launch_down<IQ2_S>(a, stream);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace tgo
