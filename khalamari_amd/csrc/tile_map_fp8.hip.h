// Tiled Map kernel for chunked prefill on FP8 E4M3FN pages (65..256 (q_token, q_head) coordinates), gfx950.
//
// Replaces gqa_sdpa_sliced_q_map / gqa_sdpa_sliced_q_per_head_map there
// (crates/inference-backend-metal/src/components/metal/gqa_sdpa_sliced_q_map.metal:29-284,
// gqa_sdpa_sliced_q_per_head_map.metal:25-298): same task ABI, masks, partial-state contract and direct output as the tiled Map
// kernel for bf16 pages (tile_map.hip.h).
//
// Work shape.  A block owns up to NWAVES * NTW * 16 (q_token, q_head) columns, a wave NTW column tiles for the whole KV range.  KV
// is walked 128 tokens at a time; the codes of a step go from HBM/L2 straight into LDS, one step ahead of their use, and are
// operands of v_mfma_scale_f32_16x16x128_f8f6f4 as they are:
//     S^T[128][cols] = K . Q^T       32 tokens at a time, the K rows as the A operand
//     weights                        online softmax per column, exp2 domain
//     O^T[D][cols] += V^T . P^T      one product over the 128 tokens, V through ds_read_b64_tr_b8; a lane holds the weights of the
//                                    very tokens whose scores it computed
// What bounds it: matrix and vector pipe together, which hardly overlap here (a weight costs the vector pipe nine full-rate
// instructions, four of them its exponential).  Decoding to bf16 in every wave that read a code took it two conversions
// more per product.  Layers, before and after: 3 chunks of 130..246 tokens on 35000..40000 at Hq24/Hkv4/D256 735 -> 475 us (its
// 484 GFLOP in the Map at 1.1 PFLOP/s), 9 prompts of 20..900 tokens there 227 -> 135 us, 4 chunks of 1000..2048 at
// Hq32/Hkv8/D128 823 -> 558 us.  Codes and straight-line order matter: the same with a branch around row tiles that no column
// sees took 548 us on the chunks, and with every slice's weights made before the next slice's scores the registers of twelve waves
// did not suffice.
//
// Arithmetic.  The other operand is split into E4M3 pieces that add up to it (fp8_device.hip.h).  A bf16 Q value, scaled so that
// the largest of its row lies in [2^7, 2^8), is exactly two pieces down to 2^-14 of that largest value and off by at most
// 2^-22 of it below.  A softmax weight is two pieces (relative error 6e-4 rms, a bf16 weight has 1.7e-3), and three (1.5e-5)
// in blocks with a column that sees few keys, where the tile kernel for bf16 pages has hi + lo bf16 pairs.  The product
// of two pieces takes the time of one bf16 product.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "device_math.hip.h"
#include "device_params.h"
#include "fp8_device.hip.h"
#include "split_kv_map.hip.h"
#include "tile_map.hip.h"

namespace khm {

constexpr int kFp8StepTokens = 128;
// two steps of K and V codes, or what the decode kernel's body works in (narrow ranges)
template <int D, int NWAVES>
constexpr int tile_map_fp8_smem_bytes() {
    constexpr int steps = 2 * 2 * kFp8StepTokens * D, narrow = D == 128 ? split_kv_map_smem_bytes<128, 1, NWAVES, true>() : 0;
    return steps > narrow ? steps : narrow;
}

template <int D, int NTW, int NWAVES, int MIN_BLOCKS>
__global__ __launch_bounds__(NWAVES * 64, MIN_BLOCKS) __attribute__((amdgpu_waves_per_eu(NWAVES * MIN_BLOCKS / 4, NWAVES * MIN_BLOCKS / 4)))
void tile_map_fp8_kernel(const MapParams p) {
    constexpr int STEP = kFp8StepTokens;
    constexpr int KD = D / 128;                  // 128-dim products per 16-token row tile
    constexpr int MT = D / 16;                   // 16-dim tiles of the output
    constexpr int CHUNKS = D / 16;               // 16-byte chunks per row
    constexpr int ROWS_PER_LOAD = 64 / CHUNKS;   // rows of a 1 KB wave load
    constexpr int UNITS = STEP / ROWS_PER_LOAD;  // wave loads per plane and step
    constexpr int UPW = (UNITS + NWAVES - 1) / NWAVES;   // units per wave, at most; a wave loads K and V of the same rows
    constexpr int PLANE_BYTES = STEP * D;
    // twelve waves have 168 registers each: no fragment ahead in the scores, no code of its own for the last 32 tokens
    constexpr bool K_AHEAD = NWAVES < 12, SHORT_TAIL = NWAVES < 12;
    extern __shared__ __align__(1024) unsigned char tile_smem[];   // [2][K plane, V plane]
    const uint32_t lds_address = lds_address_of(tile_smem);

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15;
    const int g = lane >> 4;

    typedef int I32x4 __attribute__((ext_vector_type(4)));

    // ---- task decode (uniform), as in tile_map_kernel ---------------------------------------------------------
    fetch_all_arguments(p);
    const WorkItem item = work_item_of_block<false>(active_kv_splits(p), p.num_kv_heads * p.num_q_head_ranges);
    if (!item.live) return;
    const ReplayValues replay = resolve_replay_values(p);
    const uint32_t head_group = item.head_group, task = item.task;
    const uint32_t range_index = load_uniform_u32(p.templates, 3 * (uint64_t)task);
    const uint32_t kv_begin = load_uniform_u32(p.templates, 3 * (uint64_t)task + 1);
    const uint32_t kv_end = load_uniform_u32(p.templates, 3 * (uint64_t)task + 2);
    if (range_index >= replay.num_active_q_token_tiles) return;
    const uint32_t flat_begin = load_uniform_u32(p.q_token_ranges, 2 * (uint64_t)range_index);
    const uint32_t flat_end = load_uniform_u32(p.q_token_ranges, 2 * (uint64_t)range_index + 1);
    const uint32_t num_active_tokens = replay.num_active_tokens;
    if (flat_begin >= num_active_tokens || flat_end > num_active_tokens || flat_end <= flat_begin) return;
    uint32_t num_q = flat_end - flat_begin;
    if (num_q > p.max_q_tokens) num_q = p.max_q_tokens;
    const uint32_t req_slot = load_uniform_u32(p.req_slots, flat_begin);
    const uint32_t layer = replay.layer;
    if constexpr (D == 128) {
        // narrow ranges share their tokens over the waves, as in tile_map_kernel
        if (num_q * p.max_q_heads <= 16) {
            const MapTask map_task{task, head_group, range_index, kv_begin, kv_end, flat_begin, num_q, req_slot, layer, replay.num_active_kv_splits};
            const bool shares = flat_begin > 0 && load_uniform_u32(p.req_slots, flat_begin - 1) == req_slot;
            if (shares) split_kv_map_block<D, 1, NWAVES, true, false, false, false>(p, map_task, tile_smem);
            else split_kv_map_block<D, 1, NWAVES, true, false, false, true>(p, map_task, tile_smem);
            return;
        }
    }
    const uint32_t head_range = head_group % p.num_q_head_ranges;
    const uint32_t kv_head = head_group / p.num_q_head_ranges;
    const uint32_t head_range_begin = head_range * p.max_q_heads;
    const uint32_t heads_left = p.q_heads_per_kv_head - head_range_begin;
    const uint32_t num_heads = heads_left < p.max_q_heads ? heads_left : p.max_q_heads;
    const uint32_t first_q_head = kv_head * p.q_heads_per_kv_head + head_range_begin;

    // ---- pages of the first step -----------------------------------------------------------------------------------
    // A wave load covers rows of one eight-token half of a row tile: its page is wave-uniform, and its id a scalar load one
    // step earlier.  Those of the first step are requested before the block's range is known, for the template's range: almost
    // always they are the same, and a round trip to memory less stands in front of the first K/V request.
    const uint32_t* table = p.page_ids + ((uint64_t)req_slot * p.num_gqa_layers + layer) * p.pages_per_request_layer;
    typedef uint32_t StepIds __attribute__((ext_vector_type(UPW < 2 ? 2 : UPW)));
    auto unit_of = [&](int i) -> uint32_t { return (uint32_t)(wave + i * NWAVES); };
    auto ids_of_step = [&](uint32_t step_token, uint32_t lo, uint32_t hi) __attribute__((always_inline)) -> StepIds {
        StepIds ids;
#pragma unroll
        for (int i = 0; i < UPW; ++i) {
            uint32_t token = step_token + unit_of(i) * ROWS_PER_LOAD;
            token = token < lo ? lo : token;
            token = token >= hi ? hi - 1 : token;
            const uint32_t page = token >> p.tokens_per_page_shift, last_page = p.pages_per_request_layer - 1;
            ids[i] = unit_of(i) < (uint32_t)UNITS ? load_uniform_u32(table, page < last_page ? page : last_page) : 0u;
        }
        return ids;
    };
    const uint32_t expected_hi = kv_end > kv_begin ? kv_end : kv_begin + 1;
    StepIds ids = ids_of_step(kv_begin & ~15u, kv_begin, expected_hi);

    // ---- Q rows of the wave's columns and what the columns see ---------------------------------------------------
    auto column_token = [&](int nt) { return token_of_column(p, (wave * NTW + nt) * 16 + r16); };
    auto column_head = [&](int nt) { return (wave * NTW + nt) * 16 + r16 - column_token(nt) * p.max_q_heads; };
    uint4 q_bits[NTW][KD][2][2];   // dims kd*128 + (half*4 + g)*16 .. +15
    uint32_t col_lo[NTW], col_hi[NTW];
    bool col_active[NTW];
    uint32_t wave_lo = 0u, wave_hi = 0xffffffffu, wave_last = 0u;
    bool lane_has_column = false;
#pragma unroll
    for (int nt = 0; nt < NTW; ++nt) {
        const uint32_t token_offset = column_token(nt);
        col_active[nt] = token_offset < num_q && column_head(nt) < num_heads;
        lane_has_column = lane_has_column | col_active[nt];
        // a padding column takes the block's first row: it is never stored, and no other column depends on it
        const uint64_t token = flat_begin + (col_active[nt] ? token_offset : 0u);
        const uint32_t vis_lo = p.visible_ranges[2 * token];
        const uint32_t vis_hi = p.visible_ranges[2 * token + 1];
        const uint16_t* row = p.q + (token * p.num_q_heads + first_q_head + (col_active[nt] ? column_head(nt) : 0u)) * D + g * 16;
#pragma unroll
        for (int kd = 0; kd < KD; ++kd)
#pragma unroll
            for (int i = 0; i < 4; ++i) q_bits[nt][kd][i >> 1][i & 1] = *reinterpret_cast<const uint4*>(row + kd * 128 + (i >> 1) * 64 + (i & 1) * 8);
        col_lo[nt] = vis_lo > kv_begin ? vis_lo : kv_begin;
        col_hi[nt] = vis_hi < kv_end ? vis_hi : kv_end;
    }
    // the block's range and shortest span from the visible ranges of its tokens, one per lane: every wave finds them by itself
    uint32_t blk_lo = 0xffffffffu, blk_hi = 0u, min_span = 0xffffffffu;
    for (uint32_t t = lane; t < num_q; t += 64) {
        const uint64_t token = flat_begin + t;
        const uint32_t vis_lo = p.visible_ranges[2 * token], vis_hi = p.visible_ranges[2 * token + 1];
        const uint32_t lo = vis_lo > kv_begin ? vis_lo : kv_begin, hi = vis_hi < kv_end ? vis_hi : kv_end;
        const uint32_t span = hi > lo ? hi - lo : 0u;
        if (span > 0u) {
            blk_lo = lo < blk_lo ? lo : blk_lo;
            blk_hi = hi > blk_hi ? hi : blk_hi;
        }
        min_span = span < min_span ? span : min_span;
    }
    blk_lo = __builtin_amdgcn_readfirstlane(min_over_rows(min_within_row(blk_lo)));
    blk_hi = __builtin_amdgcn_readfirstlane(~min_over_rows(min_within_row(~blk_hi)));
    min_span = __builtin_amdgcn_readfirstlane(min_over_rows(min_within_row(min_span)));
    {
        const uint64_t table_tokens = (uint64_t)p.pages_per_request_layer << p.tokens_per_page_shift;
        if (blk_hi > table_tokens) blk_hi = (uint32_t)table_tokens;
    }
    constexpr uint32_t kPreciseSpan = 1024;   // as in tile_map_kernel
    const bool precise = min_span <= kPreciseSpan;
    // [wave_lo, wave_hi): tokens that every active column of the wave sees; none of them sees a token from wave_last on
#pragma unroll
    for (int nt = 0; nt < NTW; ++nt) {
        if (col_hi[nt] > blk_hi) col_hi[nt] = blk_hi;
        if (col_hi[nt] < col_lo[nt]) col_hi[nt] = col_lo[nt];
        if (col_active[nt]) {
            wave_lo = col_lo[nt] > wave_lo ? col_lo[nt] : wave_lo;
            wave_hi = col_hi[nt] < wave_hi ? col_hi[nt] : wave_hi;
            wave_last = col_hi[nt] > wave_last ? col_hi[nt] : wave_last;
        }
    }
    wave_lo = __builtin_amdgcn_readfirstlane(max_within_row(wave_lo));
    wave_hi = __builtin_amdgcn_readfirstlane(min_within_row(wave_hi));
    wave_last = __builtin_amdgcn_readfirstlane(max_within_row(wave_last));
    uint32_t col_span[NTW];
#pragma unroll
    for (int nt = 0; nt < NTW; ++nt) col_span[nt] = col_hi[nt] - col_lo[nt];
    const bool wave_idle = __builtin_amdgcn_ballot_w64(lane_has_column) == 0;

    // ---- step schedule and loads ---------------------------------------------------------------------------------
    const uint32_t first_token = blk_lo & ~15u;
    const uint32_t num_steps = blk_hi > blk_lo ? (blk_hi - first_token + STEP - 1) / STEP : 0;
    const uint32_t tpp_mask = p.tokens_per_page - 1;
    const unsigned char* const k_plane = p.kv_pages + (uint64_t)kv_head * p.tokens_per_page * D;
    const uint64_t v_distance = (uint64_t)p.num_kv_heads * p.tokens_per_page * D;
    // Tokens outside [blk_lo, blk_hi) are redirected to the nearest one inside: their slots may hold anything.
    auto visible_token = [&](uint32_t token) -> uint32_t {
        token = token < blk_lo ? blk_lo : token;
        return token >= blk_hi ? blk_hi - 1 : token;
    };
    // Chunk c of row r sits at position c ^ swizzle(r) of the row.  K: a ds_read_b128 touches sixteen rows; V: a ds_read_b64_tr_b8
    // eight rows and the eight rows sixteen further on; both find them on different banks (rows of 128 bytes alias in pairs).
    auto k_swizzle = [](uint32_t row) -> uint32_t { return D == 128 ? (row >> 1) & 7u : row & 15u; };
    auto v_swizzle = [](uint32_t row) -> uint32_t { return D == 128 ? ((row >> 1) & 3u) | ((row >> 2) & 4u) : (row & 7u) | ((row >> 1) & 8u); };
    constexpr uint32_t kVSwizzleOfRow16 = D == 128 ? 4u << 4 : 8u << 4;   // ... in bytes; the K swizzle does not see row bit 4
    auto fetch_ids = [&](uint32_t step) __attribute__((always_inline)) -> StepIds { return ids_of_step(first_token + step * STEP, blk_lo, blk_hi); };
    auto request_step = [&](uint32_t step, const StepIds ids) __attribute__((always_inline)) {
        const uint32_t target = lds_address + (step & 1) * 2 * PLANE_BYTES;
        // the lane number is found anew: what follows from it must not live in registers from step to step
        uint32_t l = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
        asm volatile("" : "+v"(l));
        const uint32_t first_row = wave * ROWS_PER_LOAD + l / CHUNKS, position = l % CHUNKS;
        const uint32_t step_token = first_token + step * STEP;
        if (step_token >= blk_lo && step_token + STEP <= blk_hi) {
            // no clamps; the units of a wave lie whole multiples of 16 rows apart, which changes no more than one bit of the place in a
            // page of 32 tokens and one of the V swizzle
            const uint32_t in_page = ((step_token + first_row) & tpp_mask) * D;
            const uint32_t k_offset = in_page + ((position ^ k_swizzle(first_row)) << 4), v_offset = in_page + ((position ^ v_swizzle(first_row)) << 4);
            const uint32_t page_bit = p.tokens_per_page == 32 ? 16 * D : 0;
#pragma unroll
            for (int i = 0; i < UPW; ++i) {
                if (unit_of(i) >= (uint32_t)UNITS) continue;
                constexpr int ROW_STRIDE = NWAVES * ROWS_PER_LOAD;
                static_assert(ROW_STRIDE % 16 == 0, "whole row tiles");
                const bool odd = (ROW_STRIDE * i / 16) % 2 != 0;
                const unsigned char* page = k_plane + (uint64_t)__builtin_amdgcn_readfirstlane(ids[i]) * p.page_bytes;
                load_to_lds_b128<false>(page, odd ? k_offset ^ page_bit : k_offset, target + unit_of(i) * 1024);
                load_to_lds_b128<false>(page + v_distance, odd ? v_offset ^ page_bit ^ kVSwizzleOfRow16 : v_offset, target + PLANE_BYTES + unit_of(i) * 1024);
            }
            return;
        }
#pragma unroll
        for (int i = 0; i < UPW; ++i) {
            if (unit_of(i) >= (uint32_t)UNITS) continue;
            // rows behind the range are not read from K (their scores are masked) and are zeros in V (zero weights must meet finite values)
            if (step_token + unit_of(i) * ROWS_PER_LOAD >= blk_hi) {
                *(I32x4 __attribute__((address_space(3)))*)(target + PLANE_BYTES + unit_of(i) * 1024 + l * 16) = I32x4{0, 0, 0, 0};
                continue;
            }
            const uint32_t row = first_row + i * NWAVES * ROWS_PER_LOAD;
            const uint32_t offset = (visible_token(step_token + row) & tpp_mask) * D;
            const unsigned char* page = k_plane + (uint64_t)__builtin_amdgcn_readfirstlane(ids[i]) * p.page_bytes;
            load_to_lds_b128<false>(page, offset + ((position ^ k_swizzle(row)) << 4), target + unit_of(i) * 1024);
            load_to_lds_b128<false>(page + v_distance, offset + ((position ^ v_swizzle(row)) << 4), target + PLANE_BYTES + unit_of(i) * 1024);
        }
    };
    if (num_steps > 0) {
        if (blk_lo != kv_begin || blk_hi != expected_hi) ids = fetch_ids(0);
        request_step(0, ids);
        if (num_steps > 1) ids = fetch_ids(1);
    }

    // ---- Q as two E4M3 pieces in B operand order ------------------------------------------------------------------
    i32x8 q_high[NTW][KD], q_low[NTW][KD];
    float scale[NTW];
#pragma unroll
    for (int nt = 0; nt < NTW; ++nt) {
        uint32_t largest = 0;
#pragma unroll
        for (int kd = 0; kd < KD; ++kd)
#pragma unroll
            for (int i = 0; i < 4; ++i) largest = largest_magnitudes(q_bits[nt][kd][i >> 1][i & 1], largest);
        largest = ~min_over_rows(~larger_half(largest));
        const SplitScale split = split_scale_of(largest);
        scale[nt] = p.scale_log2e * split.column_scale();
#pragma unroll
        for (int kd = 0; kd < KD; ++kd)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const SplitCodes codes = split_bf16x8(q_bits[nt][kd][i >> 1][i & 1], split);
                q_high[nt][kd][2 * i] = (int)codes.high.x;
                q_high[nt][kd][2 * i + 1] = (int)codes.high.y;
                q_low[nt][kd][2 * i] = (int)codes.low.x;
                q_low[nt][kd][2 * i + 1] = (int)codes.low.y;
            }
    }

    // ---- online softmax ---------------------------------------------------------------------------------------------
    // Weights are exp2(score - ref) for a reference per column that moves when a score lies more than 8 above it, to 4 below
    // the largest score then: weights stay at most 2^8 (E4M3 ends at 448) and a column's largest at 2^4 or more, far above the
    // pieces' fixed steps (2^-9, 2^-13, 2^-17).
    constexpr float kTop = 8.0f, kMoveTo = 4.0f;
    f32x4 acc[NTW][MT];
    float ref[NTW], lane_top[NTW], run_sum[NTW];
    bool anchored[NTW];
#pragma unroll
    for (int nt = 0; nt < NTW; ++nt) {
        ref[nt] = 0.0f;
        lane_top[nt] = -INFINITY;
        run_sum[nt] = 0.0f;
        anchored[nt] = false;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[nt][mt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    // LDS read addresses.  K: row r16 of a row tile, chunk g of the first four; V: this lane's row (lanes 2j + h of a 16-lane group
    // pass half h of the sixteen dims of the j-th of the lane group's eight tokens: four of a row tile and four of the next).
    // Rows are whole powers of two, so another chunk is the address with the chunk's bits toggled.
    const uint32_t v_row = (r16 >> 1) < 4 ? g * 4 + (r16 >> 1) : 16 + g * 4 + (r16 >> 1) - 4;
    const uint32_t k_address = lds_address + r16 * D + ((g ^ k_swizzle(r16)) << 4);
    const uint32_t v_address = lds_address + PLANE_BYTES + v_row * D + (v_swizzle(v_row) << 4) + (r16 & 1) * 8;
    typedef const I32x4 __attribute__((address_space(3)))* LdsU128;
    typedef int CodeWords __attribute__((ext_vector_type(2)));
    typedef CodeWords __attribute__((address_space(3)))* LdsCodes;

    // One step of a wave: the first TILES row tiles of the 128 tokens (eight, or four or two where no column sees more)
    auto process_step = [&](auto num_pieces, auto row_tiles, uint32_t step) __attribute__((always_inline)) {
        constexpr int PIECES = decltype(num_pieces)::value;
        constexpr int TILES = decltype(row_tiles)::value;
        const uint32_t step_token = first_token + step * STEP;
        const uint32_t ring = (step & 1) * 2 * PLANE_BYTES;
        const uint32_t k_step = k_address + ring, v_step = v_address + ring;
        // scores of the step in the log2 domain, relative to the reference
        f32x4 v[NTW][TILES];
#pragma unroll
        for (int nt = 0; nt < NTW; ++nt)
#pragma unroll
            for (int t = 0; t < TILES; ++t) v[nt][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        auto k_fragment = [&](int index) __attribute__((always_inline)) -> i32x8 {   // row tile index / KD, dims (index % KD) * 128 ..
            const uint32_t row = (index / KD) * 16 * D, dims = (index % KD) * 128;
            return __builtin_shufflevector(*(LdsU128)((k_step ^ dims) + row), *(LdsU128)((k_step ^ (dims + 64)) + row), 0, 1, 2, 3, 4, 5, 6, 7);
        };
        // a fragment is read while the products of the one in front of it run, where the wave has the registers
        i32x8 a = k_fragment(0);
#pragma unroll
        for (int index = 0; index < TILES * KD; ++index) {
            if (K_AHEAD || index % (2 * KD) == 0) __builtin_amdgcn_sched_barrier(0);
            if (!K_AHEAD) a = k_fragment(index);
            const i32x8 ahead = K_AHEAD && index + 1 < TILES * KD ? k_fragment(index + 1) : a;
#pragma unroll
            for (int nt = 0; nt < NTW; ++nt) v[nt][index / KD] = mfma_fp8_k128(a, q_high[nt][index % KD], v[nt][index / KD], kPieceScale0);
#pragma unroll
            for (int nt = 0; nt < NTW; ++nt) v[nt][index / KD] = mfma_fp8_k128(a, q_low[nt][index % KD], v[nt][index / KD], kPieceScale1);
            a = ahead;
        }
        __builtin_amdgcn_sched_barrier(0);
        float step_top[NTW];
        bool wants_move = false;
#pragma unroll
        for (int nt = 0; nt < NTW; ++nt) {
#pragma unroll
            for (int t = 0; t < TILES; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) v[nt][t][i] = __builtin_fmaf(v[nt][t][i], scale[nt], -ref[nt]);
        }
        if (step_token < wave_lo || step_token + TILES * 16 > wave_hi) {
#pragma unroll
            for (int nt = 0; nt < NTW; ++nt) {
                const uint32_t behind_lo = step_token + g * 4 - col_lo[nt];
#pragma unroll
                for (int t = 0; t < TILES; ++t)
#pragma unroll
                    for (int i = 0; i < 4; ++i) v[nt][t][i] = behind_lo + t * 16 + i < col_span[nt] ? v[nt][t][i] : -INFINITY;
            }
        }
#pragma unroll
        for (int nt = 0; nt < NTW; ++nt) {
            step_top[nt] = -INFINITY;
#pragma unroll
            for (int t = 0; t < TILES; ++t) step_top[nt] = max_of_three(max_of_three(step_top[nt], v[nt][t][0], v[nt][t][1]), v[nt][t][2], v[nt][t][3]);
            wants_move = wants_move | (step_top[nt] > kTop) | (!anchored[nt] & (step_top[nt] > -INFINITY));
        }
        if (__builtin_amdgcn_ballot_w64(wants_move) != 0) {
            // rare: the four lanes of a column agree on the step's largest score, the reference moves
#pragma unroll
            for (int nt = 0; nt < NTW; ++nt) {
                const float column_top = max_over_rows(step_top[nt]);
                const bool move = column_top > kTop || (!anchored[nt] && column_top > -INFINITY);
                const float shift = move ? column_top - kMoveTo : 0.0f;
                const float alpha = anchored[nt] ? fast_exp2(-shift) : 0.0f;   // nothing is accumulated before the first key
                anchored[nt] = anchored[nt] | move;
                ref[nt] += shift;
                lane_top[nt] -= shift;
                step_top[nt] -= shift;
                run_sum[nt] *= alpha;
#pragma unroll
                for (int t = 0; t < TILES; ++t) v[nt][t] -= shift;
                if (step > 0) {
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) acc[nt][mt] *= alpha;
                }
            }
        }
        i32x8 weights[NTW][PIECES];
#pragma unroll
        for (int nt = 0; nt < NTW; ++nt) {
            float step_sum = 0.0f;
#pragma unroll
            for (int t = 0; t < TILES; ++t) {
                if (t % 2 == 0) __builtin_amdgcn_sched_barrier(0);
                float e[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) e[i] = fast_exp2(v[nt][t][i]);
                step_sum += (e[0] + e[1]) + (e[2] + e[3]);
                const uint32_t first = f32x4_to_fp8x4(e[0], e[1], e[2], e[3]);
                subtract_fp8x4(e, first);
                const uint32_t second = f32x4_to_scaled_fp8x4(e[0], e[1], e[2], e[3], kPieceStep);
                weights[nt][0][t] = (int)first;
                weights[nt][1][t] = (int)second;
                if constexpr (PIECES == 3) {
                    subtract_scaled_fp8x4(e, second, kPieceStep);
                    weights[nt][2][t] = (int)f32x4_to_scaled_fp8x4(e[0], e[1], e[2], e[3], kPieceStep * kPieceStep);
                }
            }
            lane_top[nt] = max_of_three(lane_top[nt], step_top[nt], step_top[nt]);
            run_sum[nt] += step_sum;
#pragma unroll
            for (int t = TILES; t < 8; ++t)
#pragma unroll
                for (int piece = 0; piece < PIECES; ++piece) weights[nt][piece][t] = 0;
        }
        // O^T += V^T . P^T over the 128 tokens: byte 4 t + i of a lane's fragment is token 16 t + 4 g + i of the step
        // one address register, changed in place from fragment to fragment: a new one would often be a register that a product still reads
        uint32_t v_place = v_step;
        auto v_fragment = [&](int mt) __attribute__((always_inline)) -> i32x8 {
            if (mt > 0) v_place ^= (mt ^ (mt - 1)) * 16;
            asm volatile("" : "+v"(v_place));
            i32x8 fragment;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const CodeWords codes = __builtin_amdgcn_ds_read_tr8_b64_v2i32((LdsCodes)(v_place + q * 32 * D));
                fragment[2 * q] = codes[0];
                fragment[2 * q + 1] = codes[1];
            }
            return fragment;
        };
        if constexpr (TILES == 2) {
            // thirty-two tokens: the product of that depth, which knows no scales, so the second and third pieces go apart
            typedef int CodeLong __attribute__((ext_vector_type(2)));
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                if (mt > 0) v_place ^= (mt ^ (mt - 1)) * 16;
                const long codes = __builtin_bit_cast(long, __builtin_amdgcn_ds_read_tr8_b64_v2i32((LdsCodes)v_place));
#pragma unroll
                for (int nt = 0; nt < NTW; ++nt) {
                    auto piece_of = [&](int piece) __attribute__((always_inline)) -> long { return __builtin_bit_cast(long, CodeLong{weights[nt][piece][0], weights[nt][piece][1]}); };
                    const f32x4 none = {0.0f, 0.0f, 0.0f, 0.0f};
                    f32x4 rest = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(codes, piece_of(1), none, 0, 0, 0);
                    if constexpr (PIECES == 3) {
                        const f32x4 last = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(codes, piece_of(2), none, 0, 0, 0);
#pragma unroll
                        for (int i = 0; i < 4; ++i) rest[i] = __builtin_fmaf(last[i], kPieceStep, rest[i]);
                    }
                    acc[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(codes, piece_of(0), acc[nt][mt], 0, 0, 0);
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[nt][mt][i] = __builtin_fmaf(rest[i], kPieceStep, acc[nt][mt][i]);
                }
            }
            return;
        }
        a = v_fragment(0);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            __builtin_amdgcn_sched_barrier(0);
            const i32x8 ahead = mt + 1 < MT ? v_fragment(mt + 1) : a;
#pragma unroll
            for (int piece = 0; piece < PIECES; ++piece)
#pragma unroll
                for (int nt = 0; nt < NTW; ++nt)
                    acc[nt][mt] = mfma_fp8_k128(a, weights[nt][piece], acc[nt][mt], piece == 0 ? kPieceScale0 : piece == 1 ? kPieceScale1 : kPieceScale2);
            a = ahead;
        }
    };
    // steps with more than half their tokens in the block's range, and the rest
    const uint32_t long_steps = num_steps > 0 && blk_hi - first_token - (num_steps - 1) * STEP <= STEP / 2 ? num_steps - 1 : num_steps;
    auto begin_step = [&](uint32_t step) __attribute__((always_inline)) -> bool {   // whether the wave has work in it
        wait_vmem_outstanding<0>();            // this wave's part of the step has landed
        barrier_keeping_loads_in_flight();     // everyone's has, and everyone is done with the other half of the ring
        if (step + 1 < num_steps) {
            request_step(step + 1, ids);
            if (step + 2 < num_steps) ids = fetch_ids(step + 2);
        }
        return !wave_idle && first_token + step * STEP < wave_last;
    };
    auto walk = [&](auto num_pieces) __attribute__((always_inline)) {
        asm volatile(".p2align 6");   // as the interior loop of tile_map_kernel
        for (uint32_t step = 0; step < long_steps; ++step)
            if (begin_step(step)) process_step(num_pieces, std::integral_constant<int, 8>{}, step);
        if (long_steps < num_steps && begin_step(long_steps)) {
            if (!SHORT_TAIL || blk_hi - first_token - long_steps * STEP > 32) process_step(num_pieces, std::integral_constant<int, 4>{}, long_steps);
            else process_step(num_pieces, std::integral_constant<int, SHORT_TAIL ? 2 : 4>{}, long_steps);
        }
    };
    if (precise) walk(std::integral_constant<int, 3>{});
    else walk(std::integral_constant<int, 2>{});

    // ---- epilogue: every wave owns its columns, no cross-wave merge ------------------------------------------------
    const uint32_t mode = p.output_mode;
#pragma unroll
    for (int nt = 0; nt < NTW; ++nt) {
        const float total = sum_over_rows(run_sum[nt]);         // the lanes of a column each hold the sum over their tokens
        const float column_top = max_over_rows(lane_top[nt]);   // the column's largest score, relative to ref[nt]
        if (!col_active[nt]) continue;
        const float inverse = total > 0.0f ? 1.0f / total : 0.0f;
        const uint32_t q_head = first_q_head + column_head(nt);
        uint64_t row;
        if (mode == kMapDirectBf16) {
            row = (uint64_t)(flat_begin + column_token(nt)) * p.num_q_heads + q_head;
        } else {
            row = ((uint64_t)task * p.num_q_heads + q_head) * p.max_q_tokens + column_token(nt);
            if (g == 0) {
                p.exp_sums[row] = total > 0.0f ? total * fast_exp2(-column_top) : 0.0f;
                p.max_logits[row] = total > 0.0f ? (ref[nt] + column_top) * 0.6931471805599453f : -INFINITY;
            }
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            f32x4 value = acc[nt][mt] * inverse;
            const uint32_t d = mt * 16 + g * 4;
            if (mode == kMapDirectBf16 && p.gates != nullptr) value = gate_bf16x4(value, p.gates + row * D + d);
            if (mode == kMapPartialF32) {
                *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(p.out) + row * D + d) = value;
            } else {
                const uint2 packed = make_uint2(pack_bf16x2(value[0], value[1]), pack_bf16x2(value[2], value[3]));
                *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(p.out) + row * D + d) = packed;
            }
        }
    }
}

}  // namespace khm
