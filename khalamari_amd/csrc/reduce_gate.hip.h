// Log-sum-exp Reduce kernels and the sigmoid gate for gfx950.
//
// split_kv_reduce_kernel replaces gqa_sdpa_sliced_kv_reduce_bf16
// (crates/inference-backend-metal/src/components/metal/gqa_sdpa_sliced_kv_reduce.metal:10-56) and
// gqa_sdpa_sliced_q_reduce (.../gqa_sdpa_sliced_q_reduce.metal:4-63):
//     gmax = max_p max_p;  w_p = exp(max_p - gmax) * sum_p  (0 for an empty partial);
//     out  = sum_p w_p * partial_p / sum_p w_p              (0 when the denominator is 0)
// One block owns one output row; its threads are arranged as
// (partial-slice, 8-dim octet): every slice walks a strided subset of the row's partials with
// its own running maximum, and the slices are merged through LDS.  Long rows (a 131072-token
// context has 64 partials at 2048-token partitions) therefore reduce in parallel instead of in
// one thread's serial loop.
//
// The optional gate epilogue is gqa_activation_gate_bf16 (.../gqa_activation_gate.metal:19-39)
// applied to the bf16-rounded attention value, which is what the reference's separate kernel sees.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device_math.hip.h"
#include "device_params.h"
#include "lse_merge.hip.h"

namespace khm {

constexpr int kReduceThreads = 256;

// RANGED = false: sliced-KV flat reduce, grid (tokens, heads).
// RANGED = true : sliced-Q reduce, grid (Q ranges * max_q_tokens, heads): one block per token slot of a range, so the
//                 tokens of a range reduce side by side rather than in a serial loop of dependent loads.
// Few rows with many partials: bound by the round trips to memory one after the other.  D/8 threads of 16 bytes share a
// partial, so a block has eight (D 256) or sixteen slices of the list and 64 partials are requested at once, with the gate
// values (four 131072-token contexts at Hq24/D256, 64
// partials a row: 7.3 us with 8-byte loads, four slices and two batches each, 5.2 us now).
template <int D, bool RANGED>
__global__ __launch_bounds__(kReduceThreads) void split_kv_reduce_kernel(const ReduceParams p) {
    constexpr int OCTETS = D / 8;                    // threads per partial
    constexpr int SLICES = kReduceThreads / OCTETS;  // partial slices per block
    constexpr int BATCH = 64 / SLICES;
    __shared__ float slice_stats[SLICES * 2];
    __shared__ __align__(16) float slice_acc[SLICES * D];

    const uint32_t unit = RANGED ? blockIdx.x / p.max_q_tokens : blockIdx.x;
    const uint32_t head = blockIdx.y;
    const uint32_t begin = load_uniform_u32(p.cu_partial_outputs, unit);
    const uint32_t end = load_uniform_u32(p.cu_partial_outputs, (uint64_t)unit + 1);
    uint32_t flat_begin = unit, num_q = 1, max_q = 1;
    if constexpr (RANGED) {
        flat_begin = load_uniform_u32(p.q_token_ranges, 2 * (uint64_t)unit);
        num_q = load_uniform_u32(p.q_token_ranges, 2 * (uint64_t)unit + 1) - flat_begin;
        max_q = p.max_q_tokens;
        if (num_q > max_q) num_q = max_q;
    }
    uint32_t active = p.num_active.value;
    if (p.num_active.is_parameter) active = load_uniform_u32(p.replay_parameters, active);
    if (unit >= active) return;
    const uint32_t local = RANGED ? blockIdx.x - unit * p.max_q_tokens : 0u;
    if (local >= num_q) return;

    const int octet = threadIdx.x % OCTETS;
    const uint32_t slice = threadIdx.x / OCTETS;
    // the first D/4 threads write four dims each
    const uint64_t out_index = ((uint64_t)(flat_begin + local) * p.num_q_heads + head) * D + threadIdx.x * 4;
    const bool writes = threadIdx.x < D / 4;
    const GateBits<1> gates = request_gates(writes ? p.gates : nullptr, out_index);
    const uint64_t row0 = (uint64_t)head * max_q + local, row_step = (uint64_t)p.num_q_heads * max_q;
    MergeStateOf<2> state = merge_state_empty<2>();
    if (end > begin) {
        if (p.partial_is_f32)
            merge_partial_octets<D, true, BATCH>(state, p.max_logits, p.exp_sums, p.partial, begin + slice, end, SLICES, begin, row0, row_step, octet);
        else
            merge_partial_octets<D, false, BATCH>(state, p.max_logits, p.exp_sums, p.partial, begin + slice, end, SLICES, begin, row0, row_step, octet);
    }
    if (octet == 0) {
        slice_stats[slice * 2] = state.run_max;
        slice_stats[slice * 2 + 1] = state.run_sum;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) *reinterpret_cast<f32x4*>(slice_acc + slice * D + octet * 8 + i * 4) = state.acc[i];
    __syncthreads();
    if (writes) merge_store_output(merge_combine_slices<D>(slice_stats, slice_acc, 0, SLICES, threadIdx.x), p.output, gates, out_index);
}

// The same merge for rows with few partials (speculative-verify tiles have about ten): D/8 threads own one (token, head) row
// and walk all of its partials themselves, BATCH partials requested at once and 16 bytes per lane, so nothing passes through
// LDS.  `blocks_per_unit` blocks serve one token (flat) or Q range (ranged), so everything about the unit is block-uniform
// and read with scalar loads; the live rows of a range are numbered tokens fastest, as the partial states lie in memory: the
// 4-byte maxima and sums of neighbouring rows share cache lines, and a range with one token of 32 takes blocks for its heads
// only.  Bound by the bytes of the partial states (which the Map left in the caches).  The batch follows the average number
// of partials: with sixteen for every row most loads were repeats of a row's first partial.  Before (eight bytes per lane,
// sixteen requests per row, rows numbered heads first) and now: 1025 tokens of a mixed batch at Hq64/D128 with two to three
// partials 48.1 -> 20.0 us; 511 tokens at Hq24/D256 with fourteen 26.4 -> 21.3 us; 640 tokens at Hq32/D128 with thirteen
// 21.5 -> 16.1 us; 61 verify tokens at Hq64/D128 with eight 7.5 -> 5.5 us.  The 16-byte accesses need no more than the
// 4-byte alignment that global memory instructions ask for.
template <int D, bool RANGED, int BATCH>
__global__ __launch_bounds__(kReduceThreads) void split_kv_reduce_rows_kernel(const ReduceParams p, uint32_t blocks_per_unit) {
    constexpr int OCTETS = D / 8;
    constexpr int ROWS = kReduceThreads / OCTETS;
    const uint32_t unit = blockIdx.x / blocks_per_unit;
    const uint32_t begin = load_uniform_u32(p.cu_partial_outputs, unit);
    const uint32_t end = load_uniform_u32(p.cu_partial_outputs, (uint64_t)unit + 1);
    uint32_t flat_begin = unit, num_q = 1, max_q = 1;
    if constexpr (RANGED) {
        flat_begin = load_uniform_u32(p.q_token_ranges, 2 * (uint64_t)unit);
        num_q = load_uniform_u32(p.q_token_ranges, 2 * (uint64_t)unit + 1) - flat_begin;
        max_q = p.max_q_tokens;
        if (num_q > max_q) num_q = max_q;
    }
    uint32_t active = p.num_active.value;
    if (p.num_active.is_parameter) active = load_uniform_u32(p.replay_parameters, active);
    if (unit >= active) return;
    const uint32_t row = (blockIdx.x - unit * blocks_per_unit) * ROWS + threadIdx.x / OCTETS;
    if (row >= num_q * p.num_q_heads) return;
    const int octet = threadIdx.x % OCTETS;
    const uint32_t head = RANGED ? row / num_q : row;
    const uint32_t local = RANGED ? row - head * num_q : 0u;
    const uint64_t row0 = (uint64_t)head * max_q + local, row_step = (uint64_t)p.num_q_heads * max_q;
    const uint64_t out_index = ((uint64_t)(flat_begin + local) * p.num_q_heads + head) * D + octet * 8;
    const GateBits<2> gates = request_gates<2>(p.gates, out_index);
    MergeStateOf<2> state = merge_state_empty<2>();
    if (p.partial_is_f32) {
        merge_partial_octets<D, true, BATCH / 2>(state, p.max_logits, p.exp_sums, p.partial, begin, end, 1, begin, row0, row_step, octet);
    } else if (BATCH > 8 && end - begin <= 8) {
        merge_partial_octets<D, false, 8>(state, p.max_logits, p.exp_sums, p.partial, begin, end, 1, begin, row0, row_step, octet);
    } else {
        merge_partial_octets<D, false, BATCH>(state, p.max_logits, p.exp_sums, p.partial, begin, end, 1, begin, row0, row_step, octet);
    }
    merge_store_output(state, p.output, gates, out_index);
}

// gqa_activation_gate_{f32,bf16} (gqa_activation_gate.metal:28-59): one thread per element.  For buffers that are not
// 16-byte aligned; the vector kernel below is the one that normally runs.
__global__ __launch_bounds__(256) void activation_gate_kernel(const GateParams p) {
    const uint64_t total = (uint64_t)resolve_u32(p.num_active_tokens, p.replay_parameters) * p.values_per_token;
    const uint64_t gid = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (gid >= total) return;
    if (p.is_f32) {
        const float a = reinterpret_cast<const float*>(p.attention)[gid];
        const float x = reinterpret_cast<const float*>(p.gates)[gid];
        reinterpret_cast<float*>(p.output)[gid] = a * sigmoid_f32(x);
    } else {
        const float a = bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(p.attention)[gid]);
        const float x = bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(p.gates)[gid]);
        reinterpret_cast<uint16_t*>(p.output)[gid] = f32_to_bf16_bits(a * sigmoid_bf16_steps(x));
    }
}

// The same arithmetic, 16 bytes per thread and buffer (eight bf16 or four f32 elements), the output written with streaming
// stores (it is read by the next launch, not by this one); what is left of the last group goes element by element.
constexpr int gate_elements_per_thread(bool f32) { return f32 ? 4 : 8; }
template <bool F32>
__global__ __launch_bounds__(256) void activation_gate_vector_kernel(const GateParams p) {
    constexpr int EPT = gate_elements_per_thread(F32);
    const uint64_t total = (uint64_t)resolve_u32(p.num_active_tokens, p.replay_parameters) * p.values_per_token;
    const uint64_t first = ((uint64_t)blockIdx.x * 256 + threadIdx.x) * EPT;
    if (first >= total) return;
    if (first + EPT <= total) {
        if constexpr (F32) {
            const float4 a = *reinterpret_cast<const float4*>(reinterpret_cast<const float*>(p.attention) + first);
            const float4 x = *reinterpret_cast<const float4*>(reinterpret_cast<const float*>(p.gates) + first);
            store_streaming(reinterpret_cast<float*>(p.output) + first,
                            make_float4(a.x * sigmoid_f32(x.x), a.y * sigmoid_f32(x.y), a.z * sigmoid_f32(x.z), a.w * sigmoid_f32(x.w)));
        } else {
            const uint4 a = *reinterpret_cast<const uint4*>(reinterpret_cast<const uint16_t*>(p.attention) + first);
            const uint4 x = *reinterpret_cast<const uint4*>(reinterpret_cast<const uint16_t*>(p.gates) + first);
            const uint32_t a_words[4] = {a.x, a.y, a.z, a.w}, x_words[4] = {x.x, x.y, x.z, x.w};
            uint32_t out[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float low = bf16_bits_to_f32(a_words[i] & 0xffffu) * sigmoid_bf16_steps(bf16_bits_to_f32(x_words[i] & 0xffffu));
                const float high = bf16_bits_to_f32(a_words[i] >> 16) * sigmoid_bf16_steps(bf16_bits_to_f32(x_words[i] >> 16));
                out[i] = pack_bf16x2(low, high);
            }
            store_streaming(reinterpret_cast<uint16_t*>(p.output) + first, make_uint4(out[0], out[1], out[2], out[3]));
        }
        return;
    }
    for (uint64_t i = first; i < total; ++i) {
        if constexpr (F32) {
            reinterpret_cast<float*>(p.output)[i] = reinterpret_cast<const float*>(p.attention)[i] * sigmoid_f32(reinterpret_cast<const float*>(p.gates)[i]);
        } else {
            const float a = bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(p.attention)[i]);
            const float x = bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(p.gates)[i]);
            reinterpret_cast<uint16_t*>(p.output)[i] = f32_to_bf16_bits(a * sigmoid_bf16_steps(x));
        }
    }
}

}  // namespace khm
