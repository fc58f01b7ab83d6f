"""Q ranges that fill at most one 16-column tile beside wide ones in the same launch (requests that decode beside a chunk): the waves
of a block share such a range's tokens.  Requests of their own and the last token of a chunk (its K/V are kept in the caches), ranges
on both sides of the line, slices off every boundary, NaN in unused slots."""
import numpy as np
import pytest

from khalamari_amd import sdpa
from khalamari_amd._lib import DTYPE_BF16, DTYPE_F32
from oracle import gqa_oracle as oracle

from . import gpu_runner, helpers

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("hq,hkv,tpp", [(64, 8, 16), (10, 2, 8), (16, 1, 16), (8, 2, 16)])
def test_narrow_ranges_beside_wide_ones(device, hq, hkv, tpp, fp8):
    histories, q_lens = [0, 2100, 5, 700, 130, 16, 64, 1023], [1, 1, 2, 33, 3, 4, 5, 1]
    ratio, tile = hq // hkv, 32 if hq // hkv <= 8 else 16
    w = helpers.make_workload(num_q_heads=hq, num_kv_heads=hkv, head_dim=128, tokens_per_page=tpp, histories=histories, q_lens=q_lens,
                              seed=hq + tpp, fp8_pages=fp8, garbage_bits=0x7F if fp8 else 0x7FC0)
    expected = helpers.expected_output(w)
    for kv_slice, direct, partial in [(1 << 20, True, DTYPE_BF16), (333, False, DTYPE_BF16), (64, False, DTYPE_F32)]:
        ranges, templates, cu = helpers.fixed_slice_plan(histories, q_lens, tile, kv_slice)
        print(f"narrow ranges Hq{hq}/Hkv{hkv} tpp={tpp} fp8={fp8} slice={kv_slice} direct={direct}", flush=True)
        common = dict(kind=sdpa.MAP_Q_TOKENS_AND_HEADS, max_q_tokens=tile, max_q_heads=ratio, stage=64, direct=direct, partial_dtype=partial)
        actual = gpu_runner.run_sliced_q(w, ranges, templates, cu, device, **common)
        helpers.assert_parity(actual, expected, f"narrow ranges slice={kv_slice} direct={direct}")


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("hq,hkv,heads", [(64, 8, 8), (22, 2, 8), (14, 2, 4)])   # eleven heads in ranges of 8 and 3, seven in 4 and 3
def test_narrow_ranges_gated_and_with_fewer_heads_than_the_tile(device, hq, hkv, heads, fp8):
    histories, q_lens, tile = [0, 2100, 700, 130, 63], [1, 1, 33, 3, 5], 32
    w = helpers.make_workload(num_q_heads=hq, num_kv_heads=hkv, head_dim=128, tokens_per_page=16, histories=histories, q_lens=q_lens,
                              seed=hq + heads, fp8_pages=fp8, garbage_bits=0x7F if fp8 else 0x7FC0)
    rng = np.random.default_rng(hq)
    gate_bits = oracle.f32_to_bf16_bits((rng.standard_normal((w.num_tokens, hq, 128)) * 2).astype(np.float32))
    for kv_slice, direct in [(1 << 20, True), (333, False)]:
        ranges, templates, cu = helpers.fixed_slice_plan(histories, q_lens, tile, kv_slice)
        print(f"gated narrow ranges Hq{hq}/Hkv{hkv} heads={heads} fp8={fp8} direct={direct}", flush=True)
        plain, gated = (gpu_runner.run_sliced_q(w, ranges, templates, cu, device, kind=sdpa.MAP_Q_TOKENS_AND_HEADS, max_q_tokens=tile,
                                                max_q_heads=heads, stage=64, direct=direct, gates=gates) for gates in (None, gate_bits))
        helpers.assert_parity(plain, helpers.expected_output(w), f"narrow ranges heads={heads} direct={direct}")
        # the fused gate is the standalone one on the bf16 output, bit for bit
        want = oracle.bf16_bits_to_f32(oracle.gate_bf16(oracle.f32_to_bf16_bits(plain), gate_bits))
        assert np.array_equal(gated, want.reshape(gated.shape))
