// Decode-regime forward kernel for tasks of several rows (up to 16): every weight is read and unpacked once per task and
// multiplied on the matrix cores.
//
//   y[r, n] = sum over super-blocks s of d[n, s] * sum over 32-value blocks b of dx[r, b] * dot_b(v[n, :], q[r, :])
//             - sum over b of dmin[n, s] * m[n, b] * sx[r, b]                                    (Q4_K / Q5_K)
//
// Same algebra as the matrix-core kernels with exact fp16 operands: the weight operand v = sub-scale x quant and the
// quantized activations q are integers that fp16 holds exactly (Q6_K: two numbers whose products accumulate in the same
// result), so v_mfma_f32_16x16x32_f16 returns the integer dot product of a 32-value block without rounding, already
// as a float.  What is left per block and result is one multiply-add with the activation scale, per super-block one with
// the weight scale; the minimum term is a small fp32 matrix product of its own.
//
// Layout.  The instruction's A operand is 16 weight rows x 32 values of K: lane (col, part) holds values 8 part .. + 7 of
// weight row col.  Its B operand is 32 values of K x 16 activation rows: lane (col, part) holds the same values of row col.
// Neighbouring lanes therefore hold different rows, and a load from memory in that arrangement costs the address unit a
// cycle per lane (measured: the kernel then waits for that unit alone, at 2 TB/s).  So a wave fetches the packed
// blocks of its 16 weight rows as 16-byte pieces, neighbouring lanes neighbouring pieces, two steps ahead into registers,
// parks them in LDS of its own, and reads each lane's bytes from there; the activations go the same way, once per
// super-block.  LDS executes a wave's accesses in order, so no barrier is needed anywhere in the loop.
// A wave walks a range of super-blocks (the four waves of a workgroup split K, up to four ways) and, for each, its R tiles of
// 16 weight rows.  The waves' sums meet in LDS at the end and are added in a fixed order.
//
// What it takes: a vector instruction per weight of a lane for the unpacking (Q4_K: 217 per 256 x 16 weights and wave), however many
// rows a task has.  No unit is full (28672 x 8192 Q4_K, five rows, 37 us: vector units busy 44 % of the time, LDS 35 %, matrix
// cores 11 %, 3.5 TB/s of packed bytes); what is left is each wave's own chain of fetch, park, read back, unpack and multiply at two workgroups per CU,
// and a fetch ring of four steps or a third workgroup changed nothing.  The kernels of tgo_gemv.hip
// pay four v_dot4 plus scaling per 16 weights and activation row instead and need no whole tiles: better for one to three
// rows.  Calls of more tasks than the decode regime has, up to 128 dense rows, come here too (dense_takes_tiles, grouped_takes_tiles).
// Measured against them in a layer of 97 tokens of eight choices among 256 experts (kernel time, the fused SwiGLU on top of it
// not counted): gate and up (2048 x 512) Q3_K 179 -> 75 us, Q5_K 135 -> 92, IQ2_S 140 -> 91; down (512 x 2048) Q4_K 100 -> 42, Q6_K
// 91 -> 84.  Dense 28672 x 8192, 16 rows: Q3_K 230 -> 44, Q4_K 65 -> 46, Q6_K 160 -> 69.
#include <algorithm>
#include <type_traits>

#include "tgo_device.h"
#include "tgo_launch.h"

namespace tgo {

constexpr int TILES_THREADS = 256;
constexpr int TILES_WAVES = TILES_THREADS / 64;
constexpr int TILES_RING = 2;         // steps fetched ahead (four measured the same)
constexpr int TILES_RED_PITCH = 20;   // floats per activation row of a tile's sums in LDS: 16-byte aligned, rows spread over the banks

typedef float v4f __attribute__((ext_vector_type(4)));

struct TilesArgs {
    const uint8_t * packed;
    const uint8_t * packed_second;   // second projection of a pair, or nullptr
    int64_t bytes_per_expert;
    // activations: quants, block scales and block sums, in the kernel's LAYOUT
    const int8_t * qx;
    const float * dx;
    const float * sx;
    uint16_t * y;
    uint16_t * y_second;             // (SWIGLU: silu(gate) * up)
    const int32_t * task_count;      // task list, or nullptr (dense)
    const int32_t * task_expert;
    const int32_t * task_row_start;
    const int32_t * task_row_end;
    uint32_t row_bytes;
    int rows;
    int rows_padded;
    int in_features;
    int out_features; // a multiple of 16
    int out_stride;   // values from one row of y to the next (out_features, or more)
    int k_split;      // waves that share a tile's K: 1, 2 or 4, by the length of K alone; the workgroup's other waves take other tiles
    int n_groups;     // workgroups per task and projection
    int projections;  // 1, or 2 for a pair (SWIGLU: 1, a workgroup holds the tiles of both)
};

// ---- a lane's share of a super-block --------------------------------------------------------------------------------
// Eight values (8 part .. + 7) of each of the super-block's eight 32-value blocks, packed, and the scales.
template <int TYPE> struct LaneBlock;
template <> struct LaneBlock<Q4_K> { uint4 header; uint2 q[4]; };
template <> struct LaneBlock<Q5_K> { uint4 header; uint2 q[4]; uint2 high; };
template <> struct LaneBlock<Q3_K> { uint2 q[2], high; uint4 scales; };
template <> struct LaneBlock<Q6_K> { uint2 low[4], high[2]; uint4 scales; uint16_t d; };
template <> struct LaneBlock<IQ2_S> { uint4 index[2], sign[2]; uint2 high, scales; uint16_t d; };

// `row`: the lane's block in LDS as BlockPieces lays it out; `mine`: row + 8 * part.
template <int TYPE>
TGO_DEVICE void lane_load(LaneBlock<TYPE> & r, const uint8_t * row, const uint8_t * mine) {
    if constexpr (TYPE == Q4_K || TYPE == Q5_K) {
        r.header = *reinterpret_cast<const uint4 *>(row);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            r.q[j] = *reinterpret_cast<const uint2 *>(mine + (TYPE == Q4_K ? 16 : 48) + 32 * j);
        }
        if constexpr (TYPE == Q5_K) {
            r.high = *reinterpret_cast<const uint2 *>(mine + 16);
        }
    } else if constexpr (TYPE == Q3_K) {
        r.q[0] = *reinterpret_cast<const uint2 *>(mine + 32);
        r.q[1] = *reinterpret_cast<const uint2 *>(mine + 64);
        r.high = *reinterpret_cast<const uint2 *>(mine);
        // (two bytes of quants, the scales, d)
        const uint4 tail = *reinterpret_cast<const uint4 *>(row + 96);
        r.scales = make_uint4(__builtin_amdgcn_alignbyte(tail.y, tail.x, 2), __builtin_amdgcn_alignbyte(tail.z, tail.y, 2),
                              __builtin_amdgcn_alignbyte(tail.w, tail.z, 2), tail.w >> 16);
    } else if constexpr (TYPE == Q6_K) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            r.low[j] = *reinterpret_cast<const uint2 *>(mine + 32 * j);
        }
        r.high[0] = *reinterpret_cast<const uint2 *>(mine + 128);
        r.high[1] = *reinterpret_cast<const uint2 *>(mine + 160);
        r.scales = *reinterpret_cast<const uint4 *>(row + 192);
        r.d = *reinterpret_cast<const uint16_t *>(row + 222);
    } else {
        // (a lane's eight values of a block are one codebook index byte, one sign byte and two index bits: it takes the
        // words that hold those of all four lanes of its row)
        r.d = *reinterpret_cast<const uint16_t *>(row + 80);
        r.index[0] = *reinterpret_cast<const uint4 *>(row);
        r.index[1] = *reinterpret_cast<const uint4 *>(row + 16);
        r.sign[0] = *reinterpret_cast<const uint4 *>(row + 32);
        r.sign[1] = *reinterpret_cast<const uint4 *>(row + 48);
        r.high = *reinterpret_cast<const uint2 *>(row + 64);
        r.scales = *reinterpret_cast<const uint2 *>(row + 72);
    }
}

// Sub-scales of the lane's values in the eight blocks, one byte each, and the super-block's scale(s).
struct LaneScales {
    uint32_t sub[2];   // Q4_K/Q5_K: 6-bit scales; Q3_K: 6-bit scale (+ 32); Q6_K: int8; IQ2_S: the 4-bit scale
    uint32_t min[2];   // Q4_K/Q5_K: 6-bit minima
    float d, dmin;
};
template <int TYPE>
TGO_DEVICE LaneScales lane_scales(const LaneBlock<TYPE> & r, int part) {
    LaneScales s = {};
    const uint32_t halves = part >= 2 ? 0x07050301u : 0x06040200u;   // 16-value units: the lane's is unit 2 b + part / 2 of block b
    if constexpr (TYPE == Q4_K || TYPE == Q5_K) {
        s.d = half_bits_to_float(r.header.x & 0xffffu);
        s.dmin = half_bits_to_float(r.header.x >> 16);
        s.sub[0] = r.header.y & 0x3f3f3f3fu;
        s.sub[1] = (r.header.w & 0x0f0f0f0fu) | ((r.header.y >> 2) & 0x30303030u);
        s.min[0] = r.header.z & 0x3f3f3f3fu;
        s.min[1] = ((r.header.w >> 4) & 0x0f0f0f0fu) | ((r.header.z >> 2) & 0x30303030u);
    } else if constexpr (TYPE == Q3_K) {
        // units 0-3, 4-7, 8-11, 12-15: nibbles of the first eight bytes, two bits each of the last four
        const uint32_t u0 = (r.scales.x & 0x0f0f0f0fu) | ((r.scales.z << 4) & 0x30303030u);
        const uint32_t u1 = (r.scales.y & 0x0f0f0f0fu) | ((r.scales.z << 2) & 0x30303030u);
        const uint32_t u2 = ((r.scales.x >> 4) & 0x0f0f0f0fu) | (r.scales.z & 0x30303030u);
        const uint32_t u3 = ((r.scales.y >> 4) & 0x0f0f0f0fu) | ((r.scales.z >> 2) & 0x30303030u);
        s.sub[0] = __builtin_amdgcn_perm(u1, u0, halves);
        s.sub[1] = __builtin_amdgcn_perm(u3, u2, halves);
        s.d = half_bits_to_float(r.scales.w & 0xffffu) * 0x1p14f;   // (lane_unpack)
    } else if constexpr (TYPE == Q6_K) {
        s.sub[0] = __builtin_amdgcn_perm(r.scales.y, r.scales.x, halves);
        s.sub[1] = __builtin_amdgcn_perm(r.scales.w, r.scales.z, halves);
        s.d = half_bits_to_float(r.d);
    } else {
        const int shift = part >= 2 ? 4 : 0;
        s.sub[0] = (r.scales.x >> shift) & 0x0f0f0f0fu;
        s.sub[1] = (r.scales.y >> shift) & 0x0f0f0f0fu;
        s.d = half_bits_to_float(r.d) * 0.125f;
    }
    return s;
}

// The codebook as fp16 magnitudes: what a lane multiplies by its odd multiplier 2 s + 1.
struct HalfCodebook {
    uint4 entry[TGO_IQ2S_GRID_ENTRIES];
};
TGO_DEVICE void expand_half_codebook(HalfCodebook & table, const uint32_t (&packed)[TGO_IQ2S_GRID_ENTRIES / TILES_THREADS], int tid) {
#pragma unroll
    for (int j = 0; j < TGO_IQ2S_GRID_ENTRIES / TILES_THREADS; ++j) {
        uint32_t words[4];
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            // fp16 of 8, 25, 43: 0x4800, 0x4e40, 0x5160
            const uint32_t first = (packed[j] >> (4 * p)) & 3u, second = (packed[j] >> (4 * p + 2)) & 3u;
            const uint32_t a = first == 0 ? 0x4800u : first == 1 ? 0x4e40u : 0x5160u;
            const uint32_t b = second == 0 ? 0x4800u : second == 1 ? 0x4e40u : 0x5160u;
            words[p] = a | (b << 16);
        }
        table.entry[tid + j * TILES_THREADS] = make_uint4(words[0], words[1], words[2], words[3]);
    }
}

TGO_DEVICE half8_t as_half8(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
    return __builtin_bit_cast(half8_t, make_uint4(a, b, c, d));
}
// {value, value} as fp16 of byte B of `bytes`: 1024 + byte, minus 1024
template <int B>
TGO_DEVICE uint32_t byte_as_halves(uint32_t bytes, int bias) {
    constexpr uint32_t selector = 0x04000400u + B * 0x00010001u;
    return half2_add(__builtin_amdgcn_perm(0x64646464u, bytes, selector), half2_of(-1024 - bias));
}

// The lane's eight values of block B as the fp16 operand; Q6_K: `fine` is its second operand.
template <int TYPE, int B>
TGO_DEVICE half8_t lane_unpack(const LaneBlock<TYPE> & r, const LaneScales & s, int part, const HalfCodebook * codebook, half8_t & fine) {
    const uint32_t sub_bytes = s.sub[B >> 2];
    if constexpr (TYPE == Q4_K || TYPE == Q5_K) {
        const uint32_t scale = byte_as_halves<B & 3>(sub_bytes, 0);
        const half2_t m = __builtin_bit_cast(half2_t, scale);
        const half2_t offset = __builtin_bit_cast(half2_t, half2_mul(scale, half2_of(-1024)));
        const uint32_t words[2] = {r.q[B >> 1].x, r.q[B >> 1].y};
        uint32_t out[4];
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            uint32_t bytes = (words[w] >> (4 * (B & 1))) & 0x0f0f0f0fu;
            if constexpr (TYPE == Q5_K) {
                const uint32_t high = w == 0 ? r.high.x : r.high.y;
                bytes |= (B <= 4 ? high << (4 - B) : high >> (B - 4)) & 0x10101010u;
            }
            uint32_t a, b;
            bytes_to_biased_halves(bytes, a, b);
            out[2 * w] = half2_fma(a, m, offset);
            out[2 * w + 1] = half2_fma(b, m, offset);
        }
        return as_half8(out[0], out[1], out[2], out[3]);
    } else if constexpr (TYPE == Q3_K) {
        // A zero byte above a byte b is the fp16 number b * 2^-24: one multiply-add makes (b - 4) * sub-scale * 2^-14 of it,
        // exactly (the weight scale carries the 2^14 back).
        const uint32_t scale = byte_as_halves<B & 3>(sub_bytes, 32);
        const half2_t m = __builtin_bit_cast(half2_t, half2_mul(scale, half2_of(1024)));
        const half2_t offset = __builtin_bit_cast(half2_t, half2_mul(scale, half2_t{static_cast<_Float16>(-0x1p-12f), static_cast<_Float16>(-0x1p-12f)}));
        uint32_t out[4];
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            const uint32_t low = (w == 0 ? r.q[B >> 2].x : r.q[B >> 2].y) >> (2 * (B & 3));
            const uint32_t high = w == 0 ? r.high.x : r.high.y;
            const uint32_t bytes = (low & 0x03030303u) | ((B <= 2 ? high << (2 - B) : high >> (B - 2)) & 0x04040404u);
            out[2 * w] = half2_fma(__builtin_amdgcn_perm(0u, bytes, 0x04010400u), m, offset);
            out[2 * w + 1] = half2_fma(__builtin_amdgcn_perm(0u, bytes, 0x04030402u), m, offset);
        }
        return as_half8(out[0], out[1], out[2], out[3]);
    } else if constexpr (TYPE == Q6_K) {
        // sign-magnitude split of the sub-scale (decode16_half): both parts have its sign, every product is exact
        const int sc = static_cast<int>(sub_bytes << (24 - 8 * (B & 3))) >> 24;
        const int magnitude = sc < 0 ? -sc : sc;
        const uint32_t sign = static_cast<uint32_t>(sc >> 31) & 0x80008000u;
        const uint32_t coarse_pair = (static_cast<uint32_t>(magnitude & ~15) * 0x00010001u) | 0x64006400u;
        const uint32_t fine_pair = (static_cast<uint32_t>(magnitude & 15) * 0x00010001u) | 0x64006400u;
        const half2_t coarse = __builtin_bit_cast(half2_t, half2_add(coarse_pair, half2_of(-1024)) | sign);
        const half2_t fine_scale = __builtin_bit_cast(half2_t, half2_add(fine_pair, half2_of(-1024)) | sign);
        const half2_t unbias = half2_of(-1056);
        constexpr int CHUNK = B >> 2, J = B & 3;
        uint32_t first[4], second[4];
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            const uint2 & low_words = r.low[2 * CHUNK + (J & 1)];
            const uint32_t low = (w == 0 ? low_words.x : low_words.y) >> (4 * (J >> 1));
            const uint32_t high = w == 0 ? r.high[CHUNK].x : r.high[CHUNK].y;
            const uint32_t bytes = (low & 0x0f0f0f0fu) | ((J <= 2 ? high << (4 - 2 * J) : high >> 2) & 0x30303030u);
            uint32_t a, b;
            bytes_to_biased_halves(bytes, a, b);
            a = half2_add(a, unbias);
            b = half2_add(b, unbias);
            first[2 * w] = half2_mul(a, coarse);
            first[2 * w + 1] = half2_mul(b, coarse);
            second[2 * w] = half2_mul(a, fine_scale);
            second[2 * w + 1] = half2_mul(b, fine_scale);
        }
        fine = as_half8(second[0], second[1], second[2], second[3]);
        return as_half8(first[0], first[1], first[2], first[3]);
    } else {
        const uint4 & index_words = r.index[B >> 2];
        const uint4 & sign_words = r.sign[B >> 2];
        constexpr int J = B & 3;
        const uint32_t index_word = J == 0 ? index_words.x : J == 1 ? index_words.y : J == 2 ? index_words.z : index_words.w;
        const uint32_t sign_word = J == 0 ? sign_words.x : J == 1 ? sign_words.y : J == 2 ? sign_words.z : sign_words.w;
        const uint32_t high = ((B < 4 ? r.high.x : r.high.y) >> (8 * J)) >> (2 * part);
        const uint32_t index = __builtin_amdgcn_ubfe(index_word, 8 * part, 8) | ((high & 3u) << 8);
        const uint32_t signs = sign_word >> (8 * part);
        // 2 s + 1: twice the byte plus one
        const uint32_t scale = byte_as_halves<J>(2 * sub_bytes + 0x01010101u, 0);
        const half2_t m = __builtin_bit_cast(half2_t, scale);
        // sign of value 2i at bit 2i, of value 2i + 1 at bit 2i + 16
        const uint32_t spread = (signs & 0x55u) | ((signs & 0xaau) << 15);
        const uint4 entry = codebook->entry[index];
        const uint32_t magnitude[4] = {entry.x, entry.y, entry.z, entry.w};
        uint32_t out[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            out[i] = ((spread << (15 - 2 * i)) & 0x80008000u) | half2_mul(magnitude[i], m);
        }
        return as_half8(out[0], out[1], out[2], out[3]);
    }
}

// ---- activations: 256 values of a row as fp16, rows TILES_X_PITCH bytes apart, then block scales and sums
constexpr int TILES_X_PITCH = 512 + 16;
constexpr int TILES_XS_PITCH = 20;   // floats: eight scales, eight sums, padding

template <int TYPE>
struct TileWaveLds {
    alignas(16) uint8_t raw[16 * BlockPieces<TYPE>::PITCH];
    alignas(16) uint8_t x[GEMV_TILES_ROWS * TILES_X_PITCH];
    alignas(16) float scales[GEMV_TILES_ROWS * TILES_XS_PITCH];
};

// R: tiles of 16 weight rows per wave and pass over K (more tiles: fewer fetches of the activations, fewer workgroups).
// SWIGLU (pair): half of a wave's tiles are gate rows, the other half the same rows of up; the workgroup stores
// silu(gate) * up, both rounded to bf16 first, and the gate.
// LAYOUT: of the activations.  The tile layouts are those of a workspace that is quantized before its weights are known
// (tgo_quantize_q8_1) or for several of them, which the matrix-core kernels may read as well; dense calls only.  The same quants, scales
// and sums reach LDS from any of them, so the results are the same bits.  2048 x 2048, 33 rows, us: Q6_K 22.4 by the matrix-core kernel's ranges
// of K, 10.9 here from int8 tiles (10.9 from rows); IQ2_S 21.7 and 9.5; 4096 x 4096, 64 rows: Q4_K 18.6 and 17.2.
template <int TYPE, int R, bool SWIGLU, int LAYOUT>
__global__ __launch_bounds__(TILES_THREADS, 2) void mmq_gemv_tiles_kernel(const TilesArgs a) {
    using S = BlockPieces<TYPE>;
    constexpr int REGS = (16 * S::UNITS + 63) / 64;
    constexpr bool K45 = TYPE == Q4_K || TYPE == Q5_K;
    constexpr int SIDES = SWIGLU ? 2 : 1;
    static_assert(R % SIDES == 0, "as many gate as up tiles");
    constexpr int COLUMN_TILES = R / SIDES;   // tiles of output columns per wave
    constexpr bool BY_ROWS = LAYOUT == LAYOUT_ROWS, HALVES = LAYOUT == LAYOUT_HALF_TILES;
    static_assert(BY_ROWS || LAYOUT == LAYOUT_INT8_TILES || HALVES, "the scaled tiles hold no quants");
    union WaveLds {
        TileWaveLds<TYPE> walk;
        alignas(16) float reduction[R * 16 * TILES_RED_PITCH];
    };
    __shared__ WaveLds lds[TILES_WAVES];
    using Codebook = std::conditional_t<TYPE == IQ2_S, HalfCodebook, uint2>;
    __shared__ Codebook codebook_storage;
    const HalfCodebook * const codebook = reinterpret_cast<const HalfCodebook *>(&codebook_storage);

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15;
    const int part = lane >> 4;
    const int per_task = a.n_groups * a.projections;
    const int task = blockIdx.x / per_task;
    int n_group = blockIdx.x - task * per_task;
    const bool second = n_group >= a.n_groups;
    n_group -= second ? a.n_groups : 0;
    TileWaveLds<TYPE> & mine = lds[wave].walk;

    uint32_t packed_grid[TGO_IQ2S_GRID_ENTRIES / TILES_THREADS];
    if constexpr (TYPE == IQ2_S) {   // (travels while the task is looked up)
        request_iq2s_grid(packed_grid, tid);
    }
    int expert = 0, row_start = 0, row_end = a.rows;
    if (a.task_count != nullptr) {
        // all four loads go out together (slot `task` exists in the list's arrays whatever the count says)
        const int count = a.task_count[0];
        expert = a.task_expert[task];
        row_start = a.task_row_start[task];
        row_end = a.task_row_end[task];
        if (task >= count) {
            return;
        }
    } else {
        row_start = task * GEMV_TILES_ROWS;
        row_end = min(row_start + GEMV_TILES_ROWS, a.rows);
    }
    const int nrows = row_end - row_start;

    // ---- this wave's share: super-blocks [sb_begin, sb_end) of tiles tile0 ..
    const int super_blocks = a.in_features / QK_K;
    const int split = a.k_split;
    const int share = wave % split;
    const int sb_begin = super_blocks * share / split, sb_end = super_blocks * (share + 1) / split;
    const int columns = 16 * COLUMN_TILES * (TILES_WAVES / split);   // output columns per workgroup
    const int n0 = n_group * columns;
    const int tile0 = wave / split * COLUMN_TILES;
    const uint8_t * const side_weights[2] = {
        (second ? a.packed_second : a.packed) + static_cast<int64_t>(expert) * a.bytes_per_expert,
        SWIGLU ? a.packed_second + static_cast<int64_t>(expert) * a.bytes_per_expert : nullptr};

    // A tile's pieces of a super-block, neighbouring lanes neighbouring pieces of a row (lanes past the tile repeat its last
    // piece, tiles past the matrix its last tile).
    struct __attribute__((packed, aligned(2))) Piece { u32x4_t value; };
    struct Units {
        u32x4_t value[REGS];
    };
    auto tile_base = [&](int sb, int r) __attribute__((always_inline)) {
        const int n = min(n0 + (tile0 + r % COLUMN_TILES) * 16, a.out_features - 16);
        return side_weights[SWIGLU ? r / COLUMN_TILES : 0] + static_cast<int64_t>(n) * a.row_bytes + static_cast<int64_t>(sb) * S::BLOCK;
    };
    uint32_t piece_from[REGS], piece_to[REGS];   // bytes from the tile's first block; place in `raw`
#pragma unroll
    for (int i = 0; i < REGS; ++i) {
        const int id = min(lane + 64 * i, 16 * S::UNITS - 1);
        const int row = id / S::UNITS, unit = id - row * S::UNITS;
        piece_from[i] = static_cast<uint32_t>(row) * a.row_bytes + S::offset(unit);
        piece_to[i] = row * S::PITCH + 16 * unit;
    }
    auto fetch = [&](Units & units, int sb, int r) __attribute__((always_inline)) {
        const uint8_t * const base = tile_base(sb, r);
#pragma unroll
        for (int i = 0; i < REGS; ++i) {
            if constexpr (S::ALIGNED) {
                units.value[i] = *reinterpret_cast<const u32x4_t *>(base + piece_from[i]);
            } else {
                units.value[i] = reinterpret_cast<const Piece *>(base + piece_from[i])->value;
            }
        }
    };
    auto park = [&](const Units & units) __attribute__((always_inline)) {
        asm volatile("" ::: "memory");   // (written as pieces, read as other types: the compiler must keep the order)
#pragma unroll
        for (int i = 0; i < REGS; ++i) {
            *reinterpret_cast<u32x4_t *>(mine.raw + piece_to[i]) = units.value[i];
        }
        asm volatile("" ::: "memory");
    };
    const uint8_t * const my_block = mine.raw + col * S::PITCH;
    Units ring[TILES_RING];
#pragma unroll
    for (int i = 0; i < TILES_RING; ++i) {
        fetch(ring[i], min(sb_begin + i / R, sb_end - 1), i % R);
    }

    if constexpr (TYPE == IQ2_S) {
        expand_half_codebook(codebook_storage, packed_grid, tid);
        __syncthreads();
    }

    // ---- activations of a super-block, one super-block ahead in registers.  Rows: 16 lanes fetch a row.  Tiles: 16 lanes fetch the same
    // 16 bytes of the task's 16 rows, which lie side by side (the task starts at row 0 or 16 of a tile, and the rows that it does not
    // have are there as zeros).
    constexpr int X_REGS = (HALVES ? 2 : 1) * GEMV_TILES_ROWS / 4;
    struct Incoming {
        uint4 bytes[X_REGS];
        float4 scales;   // rows: row lane / 4, piece lane % 4 of its eight block scales and eight block sums; tiles: rows 4 (lane % 4) .. + 3
                         // of block lane / 4 % 8, scales (lanes 0-31) or sums
    };
    constexpr int TILE_STEP = HALVES ? 8 * 2048 : 8 * 1024;   // bytes of a 32-row tile's super-block
    uint32_t x_offset[X_REGS];
#pragma unroll
    for (int i = 0; i < X_REGS; ++i) {
        x_offset[i] = BY_ROWS ? static_cast<uint32_t>(min(4 * i + part, nrows - 1)) * static_cast<uint32_t>(a.in_features) + col * 16
                              : static_cast<uint32_t>((4 * i + part) * 512 + ((row_start & 31) + col) * 16);
    }
    const int8_t * const x_rows = a.qx + (BY_ROWS ? static_cast<int64_t>(row_start) * a.in_features
                                                  : static_cast<int64_t>(row_start >> 5) * super_blocks * TILE_STEP);
    const float * const my_scales =
        BY_ROWS ? ((lane & 2) == 0 ? a.dx : a.sx) + static_cast<int64_t>(row_start + min(lane >> 2, nrows - 1)) * (a.in_features / 32) + 4 * (lane & 1)
                : (lane < 32 ? a.dx : a.sx) + static_cast<int64_t>((lane >> 2) & 7) * a.rows_padded + row_start + 4 * (lane & 3);
    auto x_request = [&](Incoming & in, int sb) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < X_REGS; ++i) {
            if (!BY_ROWS || 4 * i < nrows) {   // uniform
                in.bytes[i] = *reinterpret_cast<const uint4 *>(x_rows + static_cast<int64_t>(sb) * (BY_ROWS ? QK_K : TILE_STEP) + x_offset[i]);
            }
        }
        in.scales = *reinterpret_cast<const float4 *>(my_scales + static_cast<int64_t>(sb) * 8 * (BY_ROWS ? 1 : a.rows_padded));
    };
    auto x_park = [&](const Incoming & in) __attribute__((always_inline)) {
        asm volatile("" ::: "memory");
#pragma unroll
        for (int i = 0; i < X_REGS; ++i) {
            if constexpr (HALVES) {
                // (word by word: copied whole, the structure that holds them goes through scratch memory)
                *reinterpret_cast<uint4 *>(mine.x + col * TILES_X_PITCH + (4 * i + part) * 16) =
                    make_uint4(in.bytes[i].x, in.bytes[i].y, in.bytes[i].z, in.bytes[i].w);
            } else if (!BY_ROWS || 4 * i < nrows) {
                const uint32_t words[4] = {in.bytes[i].x, in.bytes[i].y, in.bytes[i].z, in.bytes[i].w};
                uint32_t halves[8];
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    uint32_t first, second_pair;
                    bytes_to_biased_halves(words[w] ^ 0x80808080u, first, second_pair);
                    halves[2 * w] = half2_add(first, half2_of(-1152));
                    halves[2 * w + 1] = half2_add(second_pair, half2_of(-1152));
                }
                uint8_t * const to = mine.x + (BY_ROWS ? (4 * i + part) * TILES_X_PITCH + col * 32 : col * TILES_X_PITCH + (4 * i + part) * 32);
                *reinterpret_cast<uint4 *>(to) = make_uint4(halves[0], halves[1], halves[2], halves[3]);
                *reinterpret_cast<uint4 *>(to + 16) = make_uint4(halves[4], halves[5], halves[6], halves[7]);
            }
        }
        if constexpr (BY_ROWS) {
            *reinterpret_cast<float4 *>(&mine.scales[(lane >> 2) * TILES_XS_PITCH + 4 * (lane & 3)]) = in.scales;
        } else {
            float * const to = &mine.scales[4 * (lane & 3) * TILES_XS_PITCH + (lane >> 2)];   // (scale or sum of block lane / 4 % 8)
            to[0] = in.scales.x;
            to[TILES_XS_PITCH] = in.scales.y;
            to[2 * TILES_XS_PITCH] = in.scales.z;
            to[3 * TILES_XS_PITCH] = in.scales.w;
        }
        asm volatile("" ::: "memory");
    };
    half8_t x[8];
    float dx[8];
    float block_sum[2] = {};   // of blocks part and 4 + part
    const int my_row = min(col, nrows - 1);   // (rows the task does not have repeat its last one: nothing of them is stored)
    const uint8_t * const my_x = mine.x + my_row * TILES_X_PITCH + 16 * part;
    const float * const my_dx = &mine.scales[my_row * TILES_XS_PITCH];
    auto x_read = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            x[b] = *reinterpret_cast<const half8_t *>(my_x + 64 * b);
        }
        const float4 low = *reinterpret_cast<const float4 *>(my_dx), high = *reinterpret_cast<const float4 *>(my_dx + 4);
        dx[0] = low.x; dx[1] = low.y; dx[2] = low.z; dx[3] = low.w;
        dx[4] = high.x; dx[5] = high.y; dx[6] = high.z; dx[7] = high.w;
        if constexpr (K45) {
            block_sum[0] = my_dx[8 + part];
            block_sum[1] = my_dx[12 + part];
        }
    };

    v4f total[R];
    const v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int r = 0; r < R; ++r) {
        total[r] = zero;
    }
    auto multiply = [&](const LaneBlock<TYPE> & block, int r) __attribute__((always_inline)) {
        const LaneScales scales = lane_scales<TYPE>(block, part);
        v4f acc = zero;
        auto one = [&](auto block_tag) __attribute__((always_inline)) {
            constexpr int B = decltype(block_tag)::value;
            half8_t fine;
            const half8_t w = lane_unpack<TYPE, B>(block, scales, part, codebook, fine);
            v4f dot = __builtin_amdgcn_mfma_f32_16x16x32_f16(w, x[B], zero, 0, 0, 0);
            if constexpr (TYPE == Q6_K) {
                dot = __builtin_amdgcn_mfma_f32_16x16x32_f16(fine, x[B], dot, 0, 0, 0);
            }
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                acc[v] = __builtin_fmaf(dot[v], dx[B], acc[v]);
            }
        };
        one(std::integral_constant<int, 0>{});
        one(std::integral_constant<int, 1>{});
        one(std::integral_constant<int, 2>{});
        one(std::integral_constant<int, 3>{});
        one(std::integral_constant<int, 4>{});
        one(std::integral_constant<int, 5>{});
        one(std::integral_constant<int, 6>{});
        one(std::integral_constant<int, 7>{});
        // the results of lane (col, part) belong to weight rows 4 part .. + 3: their scales come from the lanes that hold them
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const float d = __uint_as_float(static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(
                (4 * part + v) * 4, static_cast<int>(__float_as_uint(scales.d)))));
            total[r][v] = __builtin_fmaf(acc[v], d, total[r][v]);
        }
        if constexpr (K45) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const float weight = -scales.dmin * static_cast<float>((scales.min[h] >> (8 * part)) & 0xffu);
                total[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(weight, block_sum[h], total[r], 0, 0, 0);
            }
        }
    };

    Incoming incoming;
    x_request(incoming, sb_begin);
    constexpr int UNROLL = TILES_RING > R ? TILES_RING / R : 1;   // (the ring's slot follows from the position in the unrolled body)
#pragma unroll 1
    for (int first = sb_begin; first < sb_end; first += UNROLL) {
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            const int sb = first + u;
            if (u > 0 && sb >= sb_end) {   // uniform
                break;
            }
            x_park(incoming);
            x_read();
            x_request(incoming, min(sb + 1, sb_end - 1));
#pragma unroll
            for (int r = 0; r < R; ++r) {
                Units & units = ring[(u * R + r) % TILES_RING];
                park(units);
                LaneBlock<TYPE> block;
                lane_load<TYPE>(block, my_block, my_block + 8 * part);
                fetch(units, min(sb + (r + TILES_RING) / R, sb_end - 1), (r + TILES_RING) % R);
                multiply(block, r);
            }
        }
    }

    // ---- the waves' sums meet in LDS, each in its own part of it: [tile][activation row][16 weight rows]
    asm volatile("" ::: "memory");
#pragma unroll
    for (int r = 0; r < R; ++r) {
        *reinterpret_cast<v4f *>(&lds[wave].reduction[(r * 16 + col) * TILES_RED_PITCH + 4 * part]) = total[r];
    }
    __syncthreads();
    auto joined = [&](int side, int column, int m) __attribute__((always_inline)) {
        const int tile = column >> 4;
        const int first_wave = tile / COLUMN_TILES * split;
        const int r = side * COLUMN_TILES + tile % COLUMN_TILES;
        const int at = (r * 16 + m) * TILES_RED_PITCH + (column & 15);
        float sum = lds[first_wave].reduction[at];
        for (int s = 1; s < split; ++s) {
            sum += lds[first_wave + s].reduction[at];
        }
        return sum;
    };
    for (int id = tid; id < nrows * columns; id += TILES_THREADS) {
        const int m = id / columns;
        const int column = id - m * columns;
        if (n0 + column < a.out_features) {
            const int64_t at = static_cast<int64_t>(row_start + m) * a.out_stride + n0 + column;
            const uint16_t value = to_bf16_bits(joined(0, column, m));
            if constexpr (SWIGLU) {
                a.y[at] = value;
                a.y_second[at] = swiglu_bf16(value, to_bf16_bits(joined(1, column, m)));
            } else {
                (second ? a.y_second : a.y)[at] = value;
            }
        }
    }
}

// ---- launch ------------------------------------------------------------------------------------------------------------
template <int TYPE, bool SWIGLU, int LAYOUT>
static hipError_t launch_tiles_typed(TilesArgs args, int64_t task_slots, hipStream_t stream) {
    const int super_blocks = args.in_features / QK_K;
    args.k_split = super_blocks >= 4 ? 4 : super_blocks >= 2 ? 2 : 1;
    args.projections = args.packed_second != nullptr && !SWIGLU ? 2 : 1;
    const auto workgroups = [&](int tiles) {
        const int columns = 16 * (SWIGLU ? tiles / 2 : tiles) * (TILES_WAVES / args.k_split);
        args.n_groups = (args.out_features + columns - 1) / columns;
        return static_cast<int64_t>(args.n_groups) * args.projections * task_slots;
    };
    // four tiles per pass over the activations measured up to a tenth faster than two (28672 x 8192 Q4_K, 16 rows: 46 and
    // 52 us) while the launch still has a workgroup or two for every CU, half as fast on a matrix of 4096 x 2048
    const int tiles = workgroups(4) >= GEMV_TILES_WORKGROUPS ? 4 : 2;
    const int64_t total = workgroups(tiles);
    if (total <= 0 || total > 0x7fffffffLL) {
        return hipErrorInvalidValue;
    }
    const unsigned grid = static_cast<unsigned>(total);
    const ProfileScope scope(5, stream);
    if (tiles == 4) {
        mmq_gemv_tiles_kernel<TYPE, 4, SWIGLU, LAYOUT><<<grid, TILES_THREADS, 0, stream>>>(args);
    } else {
        mmq_gemv_tiles_kernel<TYPE, 2, SWIGLU, LAYOUT><<<grid, TILES_THREADS, 0, stream>>>(args);
    }
    return hipGetLastError();
}

hipError_t launch_mmq_gemv_tiles(const uint8_t * packed, const uint8_t * packed_second, int64_t bytes_per_expert,
                                 const Q8Workspace & ws, uint16_t * output, uint16_t * output_second,
                                 const TaskList * tasks, int rows, int in_features, int out_features,
                                 int quant_type, bool swiglu, hipStream_t stream, int output_stride) {
    const int64_t row_bytes = static_cast<int64_t>(in_features / QK_K) * block_bytes(quant_type);
    if (ws.scaled_tiles() || (!ws.by_rows() && (tasks != nullptr || swiglu)) || out_features % 16 != 0 || 16 * row_bytes > 0x7fffffffLL || (swiglu && packed_second == nullptr)) {
        return hipErrorInvalidValue;
    }
    TilesArgs args = {};
    args.packed = packed;
    args.packed_second = packed_second;
    args.bytes_per_expert = bytes_per_expert;
    args.qx = ws.q;
    args.dx = ws.d;
    args.sx = ws.sum;
    args.y = output;
    args.y_second = output_second;
    args.row_bytes = static_cast<uint32_t>(row_bytes);
    args.rows = rows;
    args.rows_padded = static_cast<int>(ws.rows_padded);
    args.in_features = in_features;
    args.out_features = out_features;
    args.out_stride = output_stride > 0 ? output_stride : out_features;
    int64_t task_slots = (rows + GEMV_TILES_ROWS - 1) / GEMV_TILES_ROWS;
    if (tasks != nullptr) {
        args.task_count = tasks->count;
        args.task_expert = tasks->expert;
        args.task_row_start = tasks->row_start;
        args.task_row_end = tasks->row_end;
        task_slots = std::min(tasks->max_tasks, rows);
    }
    const auto typed = [&](auto type) {
        constexpr int TYPE = decltype(type)::value;
        return swiglu            ? launch_tiles_typed<TYPE, true, LAYOUT_ROWS>(args, task_slots, stream)
               : ws.by_rows()    ? launch_tiles_typed<TYPE, false, LAYOUT_ROWS>(args, task_slots, stream)
               : ws.half_tiles() ? launch_tiles_typed<TYPE, false, LAYOUT_HALF_TILES>(args, task_slots, stream)
                                 : launch_tiles_typed<TYPE, false, LAYOUT_INT8_TILES>(args, task_slots, stream);
    };
    switch (quant_type) {
        case Q3_K: return typed(std::integral_constant<int, Q3_K>{});
        case Q4_K: return typed(std::integral_constant<int, Q4_K>{});
        case Q5_K: return typed(std::integral_constant<int, Q5_K>{});
        case Q6_K: return typed(std::integral_constant<int, Q6_K>{});
        case IQ2_S: return typed(std::integral_constant<int, IQ2_S>{});
        default: return hipErrorInvalidValue;
    }
}

}  // namespace tgo
