// Packing of a cotangent into MFMA fragment order, shared by the kernel that does nothing else (tgo_backward.hip) and the one that
// unpacks weights in the same launch (tgo_unpacked.hip).
#pragma once

#include "tgo_device.h"

namespace tgo {

constexpr int PACK_COLUMNS = 128;             // columns that one workgroup of 256 threads packs for 32 rows
constexpr int PACK_TILE_BYTES = 8 * 1024;     // its LDS

TGO_DEVICE uint32_t scale_bf16x2(uint32_t pair, float scale) {
    return pack_bf16x2(scale * bf16_bits_to_float(pair & 0xffffu), scale * bf16_bits_to_float(pair >> 16));
}

// 32 rows x 128 columns (8 slabs): coalesced row reads, transpose through LDS, one contiguous 8 KiB write.
// With `gather` set (single cotangent only), row r of the cotangent is bf16(scale[r] * grad[gather[r], :]):
// the routing-weighted return of a mixture-of-experts layer run backwards, read straight from the per-token
// cotangent (rows whose index lies outside [0, gather_rows) are zeros), so the expert-sorted cotangent that the
// caller would otherwise build (rows x out_features bf16 written and read again) never exists.
// `packed`: slab 0 of row tile 0; a row tile has `row_chunks` slabs, of which `n_chunks` belong to this cotangent.
TGO_DEVICE void pack_cotangent_tile(uint8_t * tile, const uint16_t * grad, uint8_t * packed, int row_tile, int chunk0, int rows,
                                    int out_features, int n_chunks, int row_chunks, const int64_t * gather, const float * scale,
                                    int64_t gather_rows, int tid) {
    const int rr = tid >> 3;            // row inside the tile
    const int c = tid & 7;              // 16-column chunk inside this workgroup
    const int row = row_tile * 32 + rr;
    const int n = (chunk0 + c) * 16;
    uint4 lo = make_uint4(0, 0, 0, 0), hi = make_uint4(0, 0, 0, 0);
    int64_t source_row = row;
    float factor = 1.0f;
    bool present = row < rows && n < out_features;
    if (gather != nullptr && present) {   // (uniform: one launch either gathers or does not)
        source_row = gather[row];
        factor = scale[row];
        present = source_row >= 0 && source_row < gather_rows;
    }
    if (present) {
        const uint16_t * src = grad + source_row * out_features + n;
        if ((out_features & 7) == 0 && n + 16 <= out_features) {
            lo = *reinterpret_cast<const uint4 *>(src);
            hi = *reinterpret_cast<const uint4 *>(src + 8);
        } else {
            uint32_t e[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                e[i] = n + i < out_features ? src[i] : 0u;
            }
            lo = make_uint4(e[0] | (e[1] << 16), e[2] | (e[3] << 16), e[4] | (e[5] << 16), e[6] | (e[7] << 16));
            hi = make_uint4(e[8] | (e[9] << 16), e[10] | (e[11] << 16), e[12] | (e[13] << 16), e[14] | (e[15] << 16));
        }
        if (gather != nullptr) {
            lo = make_uint4(scale_bf16x2(lo.x, factor), scale_bf16x2(lo.y, factor), scale_bf16x2(lo.z, factor), scale_bf16x2(lo.w, factor));
            hi = make_uint4(scale_bf16x2(hi.x, factor), scale_bf16x2(hi.y, factor), scale_bf16x2(hi.z, factor), scale_bf16x2(hi.w, factor));
        }
    }
    *reinterpret_cast<uint4 *>(tile + c * 1024 + rr * 16) = lo;
    *reinterpret_cast<uint4 *>(tile + c * 1024 + (32 + rr) * 16) = hi;
    __syncthreads();
    const int chunks_here = min(8, n_chunks - chunk0);
    uint4 * dst = reinterpret_cast<uint4 *>(packed + (static_cast<int64_t>(row_tile) * row_chunks + chunk0) * 1024);
    const uint4 * src4 = reinterpret_cast<const uint4 *>(tile);
    if (tid < chunks_here * 64) {
        dst[tid] = src4[tid];
    }
    if (tid + 256 < chunks_here * 64) {
        dst[tid + 256] = src4[tid + 256];
    }
}

}  // namespace tgo
