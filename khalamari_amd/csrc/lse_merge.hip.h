// Log-sum-exp merge of split-KV partial states, shared by the Reduce kernels and the fused Map epilogue.
//
// Contract of the reference's reducers (gqa_sdpa_sliced_kv_reduce.metal:30-55, gqa_sdpa_sliced_q_reduce.metal:27-62):
//     w_p = exp(max_p - gmax) * sum_p, 0 for an empty partial;  out = sum_p w_p * partial_p / sum_p w_p.
// Here the walk over partials is a single online pass (running max, rescale on increase) so that the loads of
// several partials can be in flight at once instead of one dependent load per step: eight per lane group in the Map's last
// block, two to sixteen in the Reduce kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device_math.hip.h"

namespace khm {

// QUADS groups of four consecutive dims per lane.
template <int QUADS>
struct MergeStateOf {
    float run_max;
    float run_sum;
    f32x4 acc[QUADS];
};
typedef MergeStateOf<1> MergeState;

template <int QUADS = 1>
__device__ __forceinline__ MergeStateOf<QUADS> merge_state_empty() {
    MergeStateOf<QUADS> state;
    state.run_max = -INFINITY;
    state.run_sum = 0.0f;
#pragma unroll
    for (int i = 0; i < QUADS; ++i) state.acc[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    return state;
}

// One more partial: its maximum, its exp-sum (both checked here: an empty partial changes nothing) and its normalized values.
template <int QUADS>
__device__ __forceinline__ void merge_one_partial(MergeStateOf<QUADS>& state, float part_max, float part_sum, const f32x4 (&value)[QUADS]) {
    if (!(part_sum > 0.0f) || !(fabsf(part_max) < INFINITY)) return;  // empty partial
    const float next_max = fmaxf(state.run_max, part_max);
    const float keep = fast_exp(state.run_max - next_max);  // 0 while run_max is still -inf
    const float weight = fast_exp(part_max - next_max) * part_sum;
    state.run_sum = state.run_sum * keep + weight;
#pragma unroll
    for (int i = 0; i < QUADS; ++i) state.acc[i] = state.acc[i] * keep + value[i] * weight;
    state.run_max = next_max;
}

__device__ __forceinline__ f32x4 bf16x4_to_f32x4(uint32_t a, uint32_t b) {
    return f32x4{bf16_bits_to_f32(a & 0xffffu), bf16_bits_to_f32(a >> 16), bf16_bits_to_f32(b & 0xffffu), bf16_bits_to_f32(b >> 16)};
}

// Merges partials first, first + step, ... < end of one (Q head, token offset) row into `state`, for the four
// dims chunk*4 .. chunk*4+3.  `safe_part` is any valid partial index (address of masked-off batch slots).  For the Map's
// last block: other blocks of the same launch wrote the partials, so the loads are device-coherent.
template <int D>
__device__ __forceinline__ void merge_partial_slice(MergeState& state, const float* max_logits, const float* exp_sums, const void* partial,
                                                    bool f32_partials, uint32_t first, uint32_t end, uint32_t step, uint32_t safe_part,
                                                    uint32_t num_q_heads, uint32_t q_head, uint32_t max_q_tokens, uint32_t token_offset,
                                                    int chunk) {
    constexpr int BATCH = 8;
    for (; first < end; first += BATCH * step) {
        float part_max[BATCH], part_sum[BATCH];
        uint64_t lo[BATCH], hi[BATCH];
#pragma unroll
        for (int k = 0; k < BATCH; ++k) {
            const uint32_t part = first + k * step;
            const bool ok = part < end;
            const uint64_t row = ((uint64_t)(ok ? part : safe_part) * num_q_heads + q_head) * max_q_tokens + token_offset;
            part_max[k] = coherent_load_f32(max_logits + row);
            part_sum[k] = ok ? coherent_load_f32(exp_sums + row) : 0.0f;
            if (f32_partials) {
                const float* source = reinterpret_cast<const float*>(partial) + row * D + chunk * 4;
                lo[k] = coherent_load_u64(source);
                hi[k] = coherent_load_u64(source + 2);
            } else {
                lo[k] = coherent_load_u64(reinterpret_cast<const uint16_t*>(partial) + row * D + chunk * 4);
                hi[k] = 0;
            }
        }
#pragma unroll
        for (int k = 0; k < BATCH; ++k) {
            f32x4 value[1];
            if (f32_partials) {
                value[0] = f32x4{__uint_as_float((uint32_t)lo[k]), __uint_as_float((uint32_t)(lo[k] >> 32)),
                                 __uint_as_float((uint32_t)hi[k]), __uint_as_float((uint32_t)(hi[k] >> 32))};
            } else {
                value[0] = bf16x4_to_f32x4((uint32_t)lo[k], (uint32_t)(lo[k] >> 32));
            }
            merge_one_partial(state, part_max[k], part_sum[k], value);
        }
    }
}

// Merges the partials begin, begin + step, ... < end of one row, eight dims per lane (dims octet * 8 .. + 8), BATCH partials
// requested at once; `safe_part` is any valid partial index (address of the requests behind the last one).
// `row0` is the row of partial 0, `row_step` the rows from one partial to the next.
template <int D, bool F32, int BATCH>
__device__ __forceinline__ void merge_partial_octets(MergeStateOf<2>& state, const float* max_logits, const float* exp_sums, const void* partial,
                                                     uint32_t begin, uint32_t end, uint32_t step, uint32_t safe_part, uint64_t row0, uint64_t row_step, int octet) {
    for (uint32_t first = begin; first < end; first += BATCH * step) {
        float part_max[BATCH], part_sum[BATCH];
        uint4 bits[BATCH], more[F32 ? BATCH : 1];
#pragma unroll
        for (int k = 0; k < BATCH; ++k) {
            const uint32_t part = first + k * step;
            const bool ok = part < end;
            const uint64_t row = row0 + (ok ? part : safe_part) * row_step;
            part_max[k] = max_logits[row];
            part_sum[k] = ok ? exp_sums[row] : 0.0f;
            const uint4* source = reinterpret_cast<const uint4*>(reinterpret_cast<const unsigned char*>(partial) + (row * D + octet * 8) * (F32 ? 4 : 2));
            bits[k] = source[0];
            if constexpr (F32) more[k] = source[1];
        }
#pragma unroll
        for (int k = 0; k < BATCH; ++k) {
            f32x4 value[2];
            if constexpr (F32) {
                value[0] = __builtin_bit_cast(f32x4, bits[k]);
                value[1] = __builtin_bit_cast(f32x4, more[k]);
            } else {
                value[0] = bf16x4_to_f32x4(bits[k].x, bits[k].y);
                value[1] = bf16x4_to_f32x4(bits[k].z, bits[k].w);
            }
            merge_one_partial(state, part_max[k], part_sum[k], value);
        }
    }
}

// Combines `count` slice states stored in LDS (stats [i][2] = (max, sum), acc [i][D]) for this lane's chunk.
template <int D>
__device__ __forceinline__ MergeState merge_combine_slices(const float* stats, const float* acc, uint32_t first, uint32_t count, int chunk) {
    float all_max = -INFINITY;
    for (uint32_t i = 0; i < count; ++i) all_max = fmaxf(all_max, stats[(first + i) * 2]);
    MergeState out = merge_state_empty();
    out.run_max = all_max;
    for (uint32_t i = 0; i < count; ++i) {
        const float slice_sum = stats[(first + i) * 2 + 1];
        if (slice_sum > 0.0f) {
            const float factor = fast_exp(stats[(first + i) * 2] - all_max);
            out.run_sum += slice_sum * factor;
            out.acc[0] += *reinterpret_cast<const f32x4*>(acc + (first + i) * D + chunk * 4) * factor;
        }
    }
    return out;
}

// The gate values of a lane's dims.  Nothing that the merge computes decides where they are, so they are requested first.
template <int QUADS>
struct GateBits {
    uint2 quad[QUADS];
    bool gated;
};
template <int QUADS = 1>
__device__ __forceinline__ GateBits<QUADS> request_gates(const uint16_t* gates, uint64_t out_index) {
    GateBits<QUADS> bits;
    bits.gated = gates != nullptr;
#pragma unroll
    for (int i = 0; i < QUADS; ++i) bits.quad[i] = bits.gated ? *reinterpret_cast<const uint2*>(gates + out_index + 4 * i) : make_uint2(0, 0);
    return bits;
}

// Normalizes, applies the optional bf16 gate (gqa_activation_gate.metal:19-39) and stores four bf16 outputs per quad.
template <int QUADS>
__device__ __forceinline__ void merge_store_output(const MergeStateOf<QUADS>& state, uint16_t* output, const GateBits<QUADS>& gates, uint64_t out_index) {
    uint32_t words[2 * QUADS];
#pragma unroll
    for (int i = 0; i < QUADS; ++i) {
        f32x4 result = {0.0f, 0.0f, 0.0f, 0.0f};
        if (state.run_sum > 0.0f) result = state.acc[i] / state.run_sum;
        if (gates.gated) result = gate_bf16x4(result, gates.quad[i]);
        words[2 * i] = pack_bf16x2(result[0], result[1]);
        words[2 * i + 1] = pack_bf16x2(result[2], result[3]);
    }
    if constexpr (QUADS == 2) {
        *reinterpret_cast<uint4*>(output + out_index) = make_uint4(words[0], words[1], words[2], words[3]);
    } else {
        static_assert(QUADS == 1, "one or two quads per lane");
        *reinterpret_cast<uint2*>(output + out_index) = make_uint2(words[0], words[1]);
    }
}

}  // namespace khm
