"""Prefill tiles whose products take the FP8 page codes as they are (Q and the weights split into E4M3 pieces): contexts on both sides of
the 128-token step and of its 64- and 32-token remainders, slices off every boundary, head ranges and Q ranges that leave columns and
waves idle, all page sizes, NaN in unused slots, Q rows of any magnitude."""
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
    """Rows whose values span many powers of two, tiny rows and zero rows keep the general tolerance (the row's scale is a power of two);
    a NaN or an infinity stays within its own row."""
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
