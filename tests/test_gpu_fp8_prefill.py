"""Prefill tiles on FP8 pages (80..256 columns): contexts on both sides of a 128-token span and of its 64- and 32-token remainders, slices
off every boundary, head ranges and Q ranges that leave columns and waves idle, all page sizes, NaN in unused slots, Q rows of any
magnitude, dominant keys, and the bits that weights and scores keep."""
import numpy as np
import pytest

from khalamari_amd import sdpa
from khalamari_amd._lib import DTYPE_BF16, DTYPE_F32
from oracle import gqa_oracle as oracle

from . import gpu_runner, helpers

pytestmark = pytest.mark.gpu

# (Q heads, KV heads, head dim, tokens per page, Q tokens of a tile): 192, 128, 256 and 160 columns at head dim 256, 128 and 80 at 128
TILES = [(12, 2, 256, 16, 32), (16, 2, 256, 32, 16), (16, 1, 256, 8, 16), (10, 2, 256, 8, 32), (8, 2, 128, 8, 32), (10, 2, 128, 16, 16)]


@pytest.mark.parametrize("hq,hkv,d,tpp,tile", TILES)
def test_steps_and_their_remainders(device, hq, hkv, d, tpp, tile):
    histories, q_lens = [0, 15, 0, 63, 90, 127, 200, 1400, 700], [17, 17, 64, 65, 38, 1, 57, 33, 5]
    w = helpers.make_workload(num_q_heads=hq, num_kv_heads=hkv, head_dim=d, tokens_per_page=tpp, histories=histories, q_lens=q_lens,
                              seed=d + tpp + tile, fp8_pages=True, garbage_bits=0x7F)
    expected = helpers.expected_output(w)
    for kv_slice, direct, partial in [(1 << 20, True, DTYPE_BF16), (1100, False, DTYPE_BF16), (77, False, DTYPE_F32)]:
        ranges, templates, cu = helpers.fixed_slice_plan(histories, q_lens, tile, kv_slice)
        print(f"fp8 prefill Hq{hq}/Hkv{hkv}/D{d} tpp={tpp} tile={tile} slice={kv_slice} direct={direct}", flush=True)
        actual = gpu_runner.run_sliced_q(w, ranges, templates, cu, device, kind=sdpa.MAP_Q_TOKENS_AND_HEADS, max_q_tokens=tile,
                                         max_q_heads=hq // hkv, stage=64, direct=direct, partial_dtype=partial)
        helpers.assert_parity(actual, expected, f"fp8 prefill slice={kv_slice} direct={direct}")


@pytest.mark.parametrize("hq,hkv,d,tpp,tile", TILES)
def test_q_rows_of_any_magnitude(device, hq, hkv, d, tpp, tile):
    """Rows whose values span many powers of two, tiny rows and zero rows keep the general tolerance; a NaN or an infinity stays within its own row."""
    histories, q_lens = [40, 300], [33, 40]
    w = helpers.make_workload(num_q_heads=hq, num_kv_heads=hkv, head_dim=d, tokens_per_page=tpp, histories=histories, q_lens=q_lens,
                              seed=d + tile, fp8_pages=True, garbage_bits=0x7F)
    q = oracle.bf16_bits_to_f32(w.q_bits).reshape(w.num_tokens, hq, d)
    rng = np.random.default_rng(tile)
    q[1] *= np.exp2(rng.integers(-30, 1, size=q[1].shape)).astype(np.float32)
    q[2] *= np.float32(1e-30)
    q[3] = 0.0
    q[4, :, 5:] = np.float32(1e-39)
    q[5, :, 7] = np.float32(-48.0)
    w.q_bits[...] = oracle.f32_to_bf16_bits(q).reshape(w.q_bits.shape)
    expected = helpers.expected_output(w).reshape(w.num_tokens, hq, d)
    # the oracle takes finite rows only: two rows become unsound after it
    q[6, 0, 3] = np.nan
    q[7, hq - 1, 9] = np.inf
    w.q_bits[...] = oracle.f32_to_bf16_bits(q).reshape(w.q_bits.shape)
    sound = np.ones((w.num_tokens, hq), dtype=bool)
    sound[6, 0] = sound[7, hq - 1] = False
    for kv_slice, direct in [(1 << 20, True), (200, False)]:
        ranges, templates, cu = helpers.fixed_slice_plan(histories, q_lens, tile, kv_slice)
        print(f"fp8 prefill magnitudes Hq{hq}/Hkv{hkv}/D{d} tpp={tpp} direct={direct}", flush=True)
        actual = gpu_runner.run_sliced_q(w, ranges, templates, cu, device, kind=sdpa.MAP_Q_TOKENS_AND_HEADS, max_q_tokens=tile,
                                         max_q_heads=hq // hkv, stage=64, direct=direct).reshape(expected.shape)
        helpers.assert_parity(actual[sound], expected[sound], f"fp8 prefill magnitudes direct={direct}")
        if direct:   # partial states of NaN scores have no sum, and the Reduce counts such a partial as empty
            assert not np.isfinite(actual[~sound]).any()


def _one_request(hq, hkv, d, tpp, q, k, v):
    """A request whose keys, values and Q rows are given (k and v [context][hkv][d], q the last rows of the context), and what float64
    attention over the stored codes and the bf16 Q rows gives, [T][Hq][D]."""
    context, tokens = k.shape[0], q.shape[0]
    w = helpers.make_workload(num_q_heads=hq, num_kv_heads=hkv, head_dim=d, tokens_per_page=tpp, histories=[context - tokens], q_lens=[tokens],
                              seed=d + tpp, fp8_pages=True)
    k, v = oracle.fp8_round_trip(oracle.bf16_round(k)), oracle.fp8_round_trip(oracle.bf16_round(v))
    w.kv_pages[...] = oracle.pack_pages(w.geom, w.kv_pages.shape[0], [(k, v)], [w.page_ids[:-(-context // tpp)]], fill_bits=0x7F)
    w.q_bits[...] = oracle.f32_to_bf16_bits(q).reshape(w.q_bits.shape)
    rows = oracle.bf16_bits_to_f32(w.q_bits).reshape(tokens, hkv, hq // hkv, d).astype(np.float64)
    expected = np.empty((tokens, hkv, hq // hkv, d))
    hidden = np.arange(context)[None, :] > (context - tokens + np.arange(tokens))[:, None]
    for head in range(hkv):
        scores = rows[:, head].reshape(-1, d) @ k[:, head].astype(np.float64).T * w.geom.scale
        scores = np.where(hidden[:, None, :], -np.inf, scores.reshape(tokens, -1, context)).reshape(-1, context)
        weights = np.exp(scores - scores.max(axis=1, keepdims=True))
        expected[:, head] = (weights @ v[:, head].astype(np.float64) / weights.sum(axis=1, keepdims=True)).reshape(tokens, -1, d)
    return w, expected.reshape(tokens, hq, d)


def _relative_error(actual, expected):
    return float(np.linalg.norm(actual.astype(np.float64) - expected) / np.linalg.norm(expected))


@pytest.mark.parametrize("sink", [0, 9000])
@pytest.mark.parametrize("hq,hkv,d,tpp,tile", TILES)
def test_one_dominant_key_leaves_the_others_their_weight(device, hq, hkv, d, tpp, tile, sink):
    """An attention sink: one key 12.5 nats above 20000 others, each of whose weights is 4e-6 of its own while together they hold a
    twelfth of the sum, and nearly all of the output, since the sink's value is small and theirs have a mean of one.  Bound: weights, partial
    states and output rows are rounded to bf16 once each."""
    context, tokens = 20000, 2 * tile
    rng = np.random.default_rng(sink + tile)
    k = rng.standard_normal((context, hkv, d)).astype(np.float32)
    v = 1.0 + rng.standard_normal((context, hkv, d)).astype(np.float32)
    q = 0.5 * rng.standard_normal((tokens, hq, d)).astype(np.float32)
    k[:, :, 0] = 0.0
    k[sink], v[sink] = 0.0, 0.015625
    k[sink, :, 0] = 16.0
    q[:, :, 0] = 12.5 / 16.0 * d ** 0.5
    w, expected = _one_request(hq, hkv, d, tpp, q, k, v)
    for kv_slice, direct in [(1 << 20, True), (1 << 20, False), (8192, False)]:
        ranges, templates, cu = helpers.fixed_slice_plan([context - tokens], [tokens], tile, kv_slice)
        print(f"fp8 sink at {sink} Hq{hq}/Hkv{hkv}/D{d} tile={tile} slice={kv_slice} direct={direct}", flush=True)
        actual = gpu_runner.run_sliced_q(w, ranges, templates, cu, device, kind=sdpa.MAP_Q_TOKENS_AND_HEADS, max_q_tokens=tile,
                                         max_q_heads=hq // hkv, stage=64, direct=direct).reshape(expected.shape)
        error = _relative_error(actual, expected)
        print(f"relative error {error:.2e}", flush=True)
        assert error <= 3 * 2.0 ** -9


@pytest.mark.parametrize("offset", [0.0, 120.0])
@pytest.mark.parametrize("hq,hkv,d,tpp,tile", TILES)
def test_few_keys_keep_sixteen_bits_of_their_weights(device, hq, hkv, d, tpp, tile, offset):
    """float32 states over a few hundred keys, with and without a key channel that lifts every score by `offset` nats (it cancels in the
    softmax).  Bound: a weight of hi + lo bf16 pieces is off by 2^-18 at most; a score is a chain of at most eight float32 sums of 32
    products, each rounded to 2^-24 of a magnitude of up to offset + 10 nats; twice that for the exponential and the weighted sum."""
    context, tokens = 500, 2 * tile
    rng = np.random.default_rng(tile)
    k, v = (rng.standard_normal((context, hkv, d)).astype(np.float32) for _ in range(2))
    q = rng.standard_normal((tokens, hq, d)).astype(np.float32)
    if offset:
        k[:, :, 0] = 240.0
        q[:, :, 0] = offset / 240.0 * d ** 0.5
    w, expected = _one_request(hq, hkv, d, tpp, q, k, v)
    ranges, templates, _ = helpers.fixed_slice_plan([context - tokens], [tokens], tile, 1 << 20)
    print(f"fp8 few keys Hq{hq}/Hkv{hkv}/D{d} tile={tile} offset={offset}", flush=True)
    states = gpu_runner.run_sliced_q_map(w, ranges, templates, device, kind=sdpa.MAP_Q_TOKENS_AND_HEADS, max_q_tokens=tile, max_q_heads=hq // hkv)
    error = _relative_error(states.swapaxes(1, 2).reshape(expected.shape), expected)
    print(f"relative error {error:.2e}", flush=True)
    assert error <= 2 * (2.0 ** -18 + 8 * 2.0 ** -24 * (offset + 10.0))


@pytest.mark.parametrize("hq,hkv,d,tpp,tile", TILES)
def test_scores_that_fall_along_the_context(device, hq, hkv, d, tpp, tile):
    """The first keys hold the weight; later ones lie further and further below the reference."""
    histories, q_lens = [0, 700, 2500], [96, 64, 40]
    w = helpers.make_workload(num_q_heads=hq, num_kv_heads=hkv, head_dim=d, tokens_per_page=tpp, histories=histories, q_lens=q_lens,
                              seed=tile, key_drift=-0.04, fp8_pages=True)
    expected = helpers.expected_output(w)
    for kv_slice, direct in [(1 << 20, True), (1024, False)]:
        ranges, templates, cu = helpers.fixed_slice_plan(histories, q_lens, tile, kv_slice)
        print(f"fp8 falling scores Hq{hq}/Hkv{hkv}/D{d} tile={tile} slice={kv_slice} direct={direct}", flush=True)
        actual = gpu_runner.run_sliced_q(w, ranges, templates, cu, device, kind=sdpa.MAP_Q_TOKENS_AND_HEADS, max_q_tokens=tile,
                                         max_q_heads=hq // hkv, stage=64, direct=direct)
        # the drifting key dimension has FP8 steps, so few keys hold the weight (as in the test of rising scores)
        helpers.assert_parity(actual, expected, f"fp8 falling scores direct={direct}", abs_tol=5.0e-3)
