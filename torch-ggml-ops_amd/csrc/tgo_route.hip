// The steps of a mixture-of-experts layer that move slots, rows and tokens around: the routing sort, and what the
// backward pass of the weighted return to tokens needs (the inverse of the slot map, the routing weights' gradients, the
// rows that no group covers).
#include <algorithm>

#include "tgo_device.h"
#include "tgo_launch.h"

namespace tgo {

// ---- routing: the (token, choice) slots sorted by expert, stably -------------------------------------------------
//   slot_rows[i]      sorted row of slot i (-1 for a slot whose expert is out of range)
//   row_index[r]      token of sorted row r (slot / top_k); -1 behind the last row
//   expert_offsets[e] rows of experts 0..e (the grouped operators' offsets with one group per expert),
//   expert_indices[e] = e
// A counting sort.  Slots are dealt to waves in runs of slot order: a wave counts its run per expert, a prefix over the
// waves (and, in a call of several workgroups, over the workgroups) gives each wave its first row of every expert, and a
// second walk hands the rows out.  Within 64 slots the lanes that name the same expert find one another with one ballot
// per bit of the expert number, so a slot's place among them is a population count: no serial walk over earlier slots.
// Bound by latency: up to ROUTE_SINGLE_SLOTS slots one workgroup does everything (776 slots over 256 experts: 17.4 us
// with a walk over the earlier slots of a batch of 256, 5.5 us now); above that the slots are cut over up to
// ROUTE_MAX_BLOCKS workgroups in two launches, counts first (16384 slots over 256 experts: 11 us; sorted with
// tensor operations those are twenty launches and 140 us).
// A call of at most ROUTE_SMALL_SLOTS slots takes a workgroup of four waves, which is quicker to start and to synchronise
// than one of sixteen.
constexpr int ROUTE_THREADS = 1024;
constexpr int64_t ROUTE_SMALL_SLOTS = 256;

// Lanes of the wave whose key equals this lane's (`bits` bits of it).
TGO_DEVICE uint64_t lanes_with_key(int key, int bits) {
    uint64_t same = ~0ull;
    for (int b = 0; b < bits; ++b) {
        const uint64_t set = __ballot((key >> b) & 1);
        same &= ((key >> b) & 1) != 0 ? set : ~set;
    }
    return same;
}

// expert of slot i, or num_experts for a slot without one
TGO_DEVICE int slot_key(const int64_t * slot_experts, int64_t i, int64_t end, int num_experts) {
    if (i >= end) {
        return num_experts;
    }
    const int64_t expert = slot_experts[i];
    return expert >= 0 && expert < num_experts ? static_cast<int>(expert) : num_experts;
}

// First launch of a call of several workgroups: counts[workgroup][expert].
template <int CAPACITY>
__global__ __launch_bounds__(ROUTE_THREADS) void route_count_kernel(const int64_t * __restrict__ slot_experts, int64_t slots,
                                                                    int64_t block_slots, int num_experts,
                                                                    int32_t * __restrict__ counts) {
    __shared__ int count[CAPACITY];
    const int tid = threadIdx.x;
    for (int e = tid; e < num_experts; e += ROUTE_THREADS) {
        count[e] = 0;
    }
    __syncthreads();
    const int64_t begin = blockIdx.x * block_slots, end = min(slots, begin + block_slots);
    for (int64_t i = begin + tid; i < end; i += ROUTE_THREADS) {
        const int key = slot_key(slot_experts, i, end, num_experts);
        if (key < num_experts) {
            atomicAdd(&count[key], 1);
        }
    }
    __syncthreads();
    for (int e = tid; e < num_experts; e += ROUTE_THREADS) {
        counts[static_cast<int64_t>(blockIdx.x) * num_experts + e] = count[e];
    }
}

// `counts`: of route_count_kernel, or nullptr when one workgroup holds all slots.
template <int CAPACITY, int THREADS>
__global__ __launch_bounds__(THREADS) void route_place_kernel(const int64_t * __restrict__ slot_experts, int64_t slots,
                                                                    int64_t block_slots, int top_k, int num_experts, int bits,
                                                                    const int32_t * __restrict__ counts,
                                                                    int64_t * __restrict__ row_index,
                                                                    int64_t * __restrict__ slot_rows,
                                                                    int64_t * __restrict__ expert_indices,
                                                                    int32_t * __restrict__ expert_offsets) {
    constexpr int WAVES = THREADS / 64;
    __shared__ uint16_t taken[WAVES][CAPACITY];         // slots per wave and expert, then the wave's next place
    __shared__ int first_row[CAPACITY];                 // of the expert in this workgroup
    __shared__ int wave_total[WAVES];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t begin = blockIdx.x * block_slots, end = min(slots, begin + block_slots);
    // the wave's run of slots: whole rounds of 64
    const int64_t wave_slots = (end - begin + THREADS - 1) / THREADS * 64;
    const int64_t wave_begin = begin + wave * wave_slots, wave_end = min(end, wave_begin + wave_slots);
    // (the first round's slots are looked up once: all there are when a workgroup has one slot per thread)
    const int first_key = slot_key(slot_experts, wave_begin + lane, wave_end, num_experts);
    const uint64_t first_same = lanes_with_key(first_key, bits);
    for (int e = lane; e < num_experts; e += 64) {
        taken[wave][e] = 0;
    }
    // (a wave touches only its own counters until the barrier below, and LDS runs a wave's accesses in order: the fences
    // keep the compiler from moving the reads of one round across the writes of the one before it)
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    for (int64_t i = wave_begin; i < wave_end; i += 64) {
        const int key = i == wave_begin ? first_key : slot_key(slot_experts, i + lane, wave_end, num_experts);
        const uint64_t same = i == wave_begin ? first_same : lanes_with_key(key, bits);
        const bool leader = (same & ((1ull << lane) - 1)) == 0;
        if (leader && key < num_experts) {
            taken[wave][key] = static_cast<uint16_t>(taken[wave][key] + __popcll(same));
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    __syncthreads();
    // A thread owns a run of consecutive experts: their rows in this workgroup, before it and in all, then the prefix over
    // the experts.
    constexpr int RUN = (CAPACITY + THREADS - 1) / THREADS;
    const int run = (num_experts + THREADS - 1) / THREADS;
    int all[RUN], before[RUN];
    int mine = 0;
#pragma unroll
    for (int j = 0; j < RUN; ++j) {
        const int e = tid * run + j;
        all[j] = 0;
        before[j] = 0;
        if (j < run && e < num_experts) {
            int next = 0;
#pragma unroll
            for (int w = 0; w < WAVES; ++w) {
                const int count = taken[w][e];
                taken[w][e] = static_cast<uint16_t>(next);
                next += count;
            }
            all[j] = next;
            if (counts != nullptr) {
                all[j] = 0;
                // (eight requests in flight: one at a time, the walk over the workgroups is a chain of round trips)
                const int blocks = gridDim.x;
                for (int block = 0; block < blocks; block += 8) {
                    int count[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u) {
                        count[u] = counts[static_cast<int64_t>(min(block + u, blocks - 1)) * num_experts + e];
                    }
#pragma unroll
                    for (int u = 0; u < 8; ++u) {
                        const int value = block + u < blocks ? count[u] : 0;
                        before[j] += block + u < static_cast<int>(blockIdx.x) ? value : 0;
                        all[j] += value;
                    }
                }
            }
        }
        mine += all[j];
    }
    int inclusive = mine;
#pragma unroll
    for (int offset = 1; offset < 64; offset <<= 1) {
        const int add = __shfl_up(inclusive, offset);
        inclusive += lane >= offset ? add : 0;
    }
    if (lane == 63) {
        wave_total[wave] = inclusive;
    }
    __syncthreads();
    int start = inclusive - mine, total = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
        start += w < wave ? wave_total[w] : 0;
        total += wave_total[w];
    }
#pragma unroll
    for (int j = 0; j < RUN; ++j) {
        const int e = tid * run + j;
        if (j < run && e < num_experts) {
            first_row[e] = start + before[j];
            start += all[j];
            if (blockIdx.x == 0) {
                expert_offsets[e] = start;
                expert_indices[e] = e;
            }
        }
    }
    // rows behind the last one name no token (every workgroup clears its share: nobody else writes those)
    for (int64_t i = max(begin, static_cast<int64_t>(total)) + tid; i < end; i += THREADS) {
        row_index[i] = -1;
    }
    __syncthreads();
    for (int64_t i = wave_begin; i < wave_end; i += 64) {
        const int key = i == wave_begin ? first_key : slot_key(slot_experts, i + lane, wave_end, num_experts);
        const uint64_t same = i == wave_begin ? first_same : lanes_with_key(key, bits);
        const uint64_t earlier = same & ((1ull << lane) - 1);
        int row = -1;
        if (key < num_experts) {
            row = first_row[key] + taken[wave][key] + __popcll(earlier);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if (earlier == 0 && key < num_experts) {
            taken[wave][key] = static_cast<uint16_t>(taken[wave][key] + __popcll(same));
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if (i + lane < wave_end) {
            slot_rows[i + lane] = row;
            if (row >= 0) {
                row_index[row] = (i + lane) / top_k;
            }
        }
    }
}

int route_blocks(int64_t slots) {
    return slots <= ROUTE_SINGLE_SLOTS ? 1 : static_cast<int>(std::min<int64_t>((slots + ROUTE_THREADS - 1) / ROUTE_THREADS, ROUTE_MAX_BLOCKS));
}

template <int CAPACITY>
static hipError_t launch_route_sized(const int64_t * slot_experts, int64_t slots, int top_k, int num_experts, int32_t * counts,
                                     int64_t * row_index, int64_t * slot_rows, int64_t * expert_indices,
                                     int32_t * expert_offsets, hipStream_t stream) {
    const int blocks = route_blocks(slots);
    const int64_t block_slots = ((slots + blocks - 1) / blocks + ROUTE_THREADS - 1) / ROUTE_THREADS * ROUTE_THREADS;
    int bits = 1;
    while ((1 << bits) <= num_experts) {   // (keys 0 .. num_experts)
        ++bits;
    }
    if constexpr (CAPACITY <= 1024) {
        if (slots <= ROUTE_SMALL_SLOTS) {
            route_place_kernel<CAPACITY, 256><<<1, 256, 0, stream>>>(slot_experts, slots, slots, top_k, num_experts, bits, nullptr,
                                                                     row_index, slot_rows, expert_indices, expert_offsets);
            return hipGetLastError();
        }
    }
    if (blocks > 1) {
        route_count_kernel<CAPACITY><<<blocks, ROUTE_THREADS, 0, stream>>>(slot_experts, slots, block_slots, num_experts, counts);
    }
    route_place_kernel<CAPACITY, ROUTE_THREADS><<<blocks, ROUTE_THREADS, 0, stream>>>(
        slot_experts, slots, block_slots, top_k, num_experts, bits, blocks > 1 ? counts : nullptr, row_index, slot_rows,
                                                                       expert_indices, expert_offsets);
    return hipGetLastError();
}

hipError_t launch_route(const int64_t * slot_experts, int64_t slots, int top_k, int num_experts, int32_t * counts,
                        int64_t * row_index, int64_t * slot_rows, int64_t * expert_indices, int32_t * expert_offsets,
                        hipStream_t stream) {
    if (slots <= 0 || slots > ROUTE_SLOT_LIMIT || num_experts <= 0 || num_experts > ROUTE_EXPERT_LIMIT ||
        (route_blocks(slots) > 1 && counts == nullptr)) {
        return hipErrorInvalidValue;
    }
    // (a workgroup clears and walks LDS for as many experts as it is compiled for: 10, 36 or 144 KiB of it)
    const auto launch = num_experts <= 256 ? launch_route_sized<256> : num_experts <= 1024 ? launch_route_sized<1024>
                                                                                           : launch_route_sized<ROUTE_EXPERT_LIMIT>;
    return launch(slot_experts, slots, top_k, num_experts, counts, row_index, slot_rows, expert_indices, expert_offsets, stream);
}

// ---- the slot map inverted ------------------------------------------------------------------------------------
// row_token[r], row_weight[r] = token and routing weight of the slot that names row r; -1 and 0 for a row that none does.
__global__ __launch_bounds__(256) void clear_rows_kernel(int64_t * __restrict__ row_token, float * __restrict__ row_weight,
                                                         int64_t num_rows) {
    const int64_t row = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (row < num_rows) {
        row_token[row] = -1;
        row_weight[row] = 0.0f;
    }
}
__global__ __launch_bounds__(256) void invert_slots_kernel(const int64_t * __restrict__ slot_rows,
                                                           const float * __restrict__ slot_weights, int64_t slots, int top_k,
                                                           int64_t num_rows, int64_t * __restrict__ row_token,
                                                           float * __restrict__ row_weight) {
    const int64_t slot = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (slot >= slots) {
        return;
    }
    const int64_t row = slot_rows[slot];
    if (row >= 0 && row < num_rows) {
        row_token[row] = slot / top_k;
        row_weight[row] = slot_weights[slot];
    }
}

hipError_t launch_invert_slots(const int64_t * slot_rows, const float * slot_weights, int64_t slots, int top_k,
                               int64_t num_rows, int64_t * row_token, float * row_weight, hipStream_t stream) {
    clear_rows_kernel<<<static_cast<unsigned>((num_rows + 255) / 256), 256, 0, stream>>>(row_token, row_weight, num_rows);
    invert_slots_kernel<<<static_cast<unsigned>((slots + 255) / 256), 256, 0, stream>>>(slot_rows, slot_weights, slots, top_k,
                                                                                       num_rows, row_token, row_weight);
    return hipGetLastError();
}

// ---- gradient of the routing weights ------------------------------------------------------------------------------
// grad_weights[t, j] = sum over f of rows[slot_rows[t, j], f] * grad_tokens[t, f]: bf16 operands, fp32 sums in a fixed
// order, 0 for a slot without a row.  One wave per slot: the rows are read once (the token's gradient stays in the L1 for
// its choices), so the kernel runs at the rate of memory: 32768 slots of 2048 values 38 us, where the gather, the
// fp32 copies, their product and its sum were 480 us.
__global__ __launch_bounds__(256) void slot_weight_grad_kernel(const uint16_t * __restrict__ rows,
                                                               const uint16_t * __restrict__ grad_tokens,
                                                               const int64_t * __restrict__ slot_rows,
                                                               float * __restrict__ grad_weights, int64_t slots, int top_k,
                                                               int64_t num_rows, int features) {
    const int64_t slot = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (slot >= slots) {
        return;
    }
    const int64_t row = slot_rows[slot];
    float sum = 0.0f;
    if (row >= 0 && row < num_rows) {   // uniform in the wave
        const uint16_t * const a = rows + row * features;
        const uint16_t * const b = grad_tokens + slot / top_k * features;
#pragma unroll 4
        for (int f = lane * 8; f < features; f += 64 * 8) {
            const uint4 x = *reinterpret_cast<const uint4 *>(a + f);
            const uint4 y = *reinterpret_cast<const uint4 *>(b + f);
            const uint32_t xs[4] = {x.x, x.y, x.z, x.w}, ys[4] = {y.x, y.y, y.z, y.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                sum = __builtin_fmaf(bf16_bits_to_float(xs[i] & 0xffffu), bf16_bits_to_float(ys[i] & 0xffffu), sum);
                sum = __builtin_fmaf(bf16_bits_to_float(xs[i] >> 16), bf16_bits_to_float(ys[i] >> 16), sum);
            }
        }
    }
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1) {
        sum += __shfl_xor(sum, offset);
    }
    if (lane == 0) {
        grad_weights[slot] = sum;
    }
}

hipError_t launch_slot_weight_grad(const uint16_t * rows, const uint16_t * grad_tokens, const int64_t * slot_rows,
                                   float * grad_weights, int64_t slots, int top_k, int64_t num_rows, int features,
                                   hipStream_t stream) {
    const ProfileScope scope(7, stream);
    slot_weight_grad_kernel<<<static_cast<unsigned>((slots + 3) / 4), 256, 0, stream>>>(rows, grad_tokens, slot_rows, grad_weights,
                                                                                       slots, top_k, num_rows, features);
    return hipGetLastError();
}

// ---- rows that no valid group covers ---------------------------------------------------------------------------------
// Zeros in the rows of `rows` [num_rows, features] that lie in no valid group (the rule of build_tasks): what a
// grad-input leaves unwritten and a sum over all rows must not see.  A workgroup checks 256 rows against the whole group
// list and writes only where there is something to clear, so a call whose groups cover every row reads the list and
// leaves (5 us), where filling the whole tensor beforehand wrote it once more than needed.
__global__ __launch_bounds__(256) void clear_uncovered_kernel(uint16_t * __restrict__ rows, int64_t num_rows, int features,
                                                              const int64_t * __restrict__ expert_indices,
                                                              const int32_t * __restrict__ expert_offsets, int num_groups,
                                                              int num_experts) {
    __shared__ int change[257];   // groups that begin minus groups that end at each of the workgroup's rows
    __shared__ int wave_total[4];
    __shared__ uint8_t uncovered[256];
    const int tid = threadIdx.x;
    const int64_t first = static_cast<int64_t>(blockIdx.x) * 256;
    change[tid] = 0;
    __syncthreads();
    for (int group = tid; group < num_groups; group += 256) {
        const int64_t begin = group == 0 ? 0 : expert_offsets[group - 1];
        const int64_t end = expert_offsets[group];
        const int64_t expert = expert_indices[group];
        if (expert >= 0 && expert < num_experts && begin >= 0 && end > begin && end <= num_rows && begin < first + 256 && end > first) {
            atomicAdd(&change[max(begin, first) - first], 1);
            atomicAdd(&change[min(end, first + 256) - first], -1);
        }
    }
    __syncthreads();
    int cover = change[tid];
#pragma unroll
    for (int offset = 1; offset < 64; offset <<= 1) {
        const int add = __shfl_up(cover, offset);
        cover += (tid & 63) >= offset ? add : 0;
    }
    if ((tid & 63) == 63) {
        wave_total[tid >> 6] = cover;
    }
    __syncthreads();
    for (int w = 0; w < (tid >> 6); ++w) {
        cover += wave_total[w];
    }
    const bool covered = first + tid >= num_rows || cover > 0;
    uncovered[tid] = covered ? 0 : 1;
    if (__syncthreads_or(covered ? 0 : 1) == 0) {
        return;
    }
    for (int r = 0; r < 256; ++r) {
        if (uncovered[r] != 0) {   // uniform
            uint16_t * const dst = rows + (first + r) * features;
            for (int f = tid; f < features; f += 256) {
                dst[f] = 0;
            }
        }
    }
}

hipError_t launch_clear_uncovered(uint16_t * rows, int64_t num_rows, int features, const int64_t * expert_indices,
                                  const int32_t * expert_offsets, int num_groups, int num_experts, hipStream_t stream) {
    clear_uncovered_kernel<<<static_cast<unsigned>((num_rows + 255) / 256), 256, 0, stream>>>(
        rows, num_rows, features, expert_indices, expert_offsets, num_groups, num_experts);
    return hipGetLastError();
}

}  // namespace tgo
