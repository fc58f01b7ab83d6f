"""The Reduce kernels against the merge in float64: every number of partials around their batches of 4, 8, 16 and 64, ranges with one, some, all and no live token, Q-head counts that fill no block, bf16 and float32 partials."""
import numpy as np
import pytest

from khalamari_amd import sdpa, sliced_q
from khalamari_amd._lib import DTYPE_BF16, DTYPE_F32, ReplayU32

pytestmark = pytest.mark.gpu
POISON = 0x4228


@pytest.mark.parametrize("partial_dtype", [DTYPE_BF16, DTYPE_F32])
@pytest.mark.parametrize("hq,hkv,d,tile,counts", [
    (8, 1, 128, 32, [1, 2, 4, 5, 3, 1]),
    (12, 2, 256, 8, [4, 8, 9, 7, 16, 3]),
    (40, 8, 128, 1, [15, 16, 17, 1, 8, 31]),
    (12, 2, 256, 2, [40, 64, 65, 17, 100, 3]),     # more than sixteen on average: the list split over a block's threads
    (5, 1, 128, 4, [1, 15, 64, 129, 16, 2]),
])
@pytest.mark.parametrize("replayed", [False, True])
def test_reduce_against_the_merge_in_float64(device, hq, hkv, d, tile, counts, partial_dtype, replayed):
    import torch

    rng = np.random.default_rng(d + tile)
    live = [tile, 1, max(1, tile // 2), max(1, tile - 1), tile, 0]   # the last range is empty: nothing of it is written
    begins = np.concatenate([[0], np.cumsum(live)])
    ranges = np.array([(begins[i], begins[i + 1]) for i in range(len(live))], dtype=np.uint32)
    cu = np.concatenate([[0], np.cumsum(counts)]).astype(np.uint32)
    tokens, templates, tiles = int(begins[-1]) + 1, int(cu[-1]), len(live)   # one token that no range holds
    layout = sliced_q.Layout(1, 1, 4, 1)
    config = sliced_q.Config(hq, hkv, d, d ** -0.5, 2 * 2 * hkv * 16 * d, layout, partial_dtype=partial_dtype)
    variant = sdpa.ExecutionVariant.sliced_q(config.sdpa_config(), sdpa.MAP_Q_TOKENS_AND_HEADS, tile, 64, hq // hkv)
    shape = sliced_q.Shape(tokens, tiles, templates)
    compute = sliced_q.Compute(config, variant, shape)

    values = rng.standard_normal((templates, hq, tile, d)).astype(np.float32)
    maxima = (3.0 * rng.standard_normal((templates, hq, tile))).astype(np.float32)
    sums = rng.uniform(0.5, 40.0, (templates, hq, tile)).astype(np.float32)
    empty = rng.random((templates, hq, tile)) < 0.15
    maxima[empty], sums[empty] = -np.inf, 0.0
    stored = torch.from_numpy(values).to(torch.bfloat16 if partial_dtype == DTYPE_BF16 else torch.float32)
    exact = stored.to(torch.float64).numpy()
    gates = torch.from_numpy(rng.standard_normal((tokens, hq, d)).astype(np.float32)).to(torch.bfloat16)

    expected = np.zeros((tokens, hq, d))
    for r in range(tiles):
        for t in range(live[r]):
            m, s, v = (a[cu[r]:cu[r + 1], :, t].astype(np.float64) for a in (maxima, sums, exact))
            top = m.max(axis=0)
            weight = np.where(s > 0, np.exp(np.where(s > 0, m, 0.0) - np.where(np.isfinite(top), top, 0.0)) * s, 0.0)
            total = weight.sum(axis=0)
            merged = (weight[..., None] * v).sum(axis=0)
            expected[begins[r] + t] = np.where(total[:, None] > 0, merged / np.where(total > 0, total, 1.0)[:, None], 0.0)

    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(device)  # noqa: E731
    params = torch.tensor([tiles, 0, 0, 0], dtype=torch.int32, device=device) if replayed else None
    common = dict(partial_output=stored.to(device), partial_exp_sums=dev(sums), partial_max_logits=dev(maxima), q_token_ranges=dev(ranges.view(np.int32)),
                  cu_sdpa_partial_outputs=dev(cu.view(np.int32)), replay_parameters=params,
                  num_active_q_token_tiles=ReplayU32.parameter(0) if replayed else ReplayU32.fixed(tiles))
    out = torch.full((tokens, hq, d), POISON, dtype=torch.int16, device=device)
    gated = torch.full_like(out, POISON)
    print(f"reduce rows Hq{hq} D{d} tile={tile} counts={counts} f32={partial_dtype == DTYPE_F32} replayed={replayed}", flush=True)
    compute.invoke_reduce(output=out, **common)
    compute.invoke_reduce(output=gated, gates=gates.to(device), **common)
    torch.cuda.synchronize()
    assert bool((out[-1] == POISON).all()) and bool((gated[-1] == POISON).all())
    out, gated, expected, gates = out[:-1], gated[:-1], expected[:-1], gates[:-1]
    actual = out.view(torch.bfloat16).to(torch.float64).cpu().numpy()
    # one rounding to bf16 (eight significant bits: 2^-8 of the value at most) and float32 sums of terms of order one
    assert np.all(np.abs(actual - expected) <= np.abs(expected) * 2.0 ** -8 + max(counts) * 2.0 ** -23)
    # the gate multiplies the rounded value with a sigmoid computed in bf16 steps, u = 2^-8 each: the exponential (half of its
    # error reaches the quotient), the denominator, the quotient and, below zero, one minus it, 3.5 u in all of a value up to
    # one; the product is rounded once more
    sigmoid = 1.0 / (1.0 + np.exp(-gates.to(torch.float64).numpy()))
    actual_gated = gated.view(torch.bfloat16).to(torch.float64).cpu().numpy()
    assert np.all(np.abs(actual_gated - actual * sigmoid) <= np.abs(actual) * (4.0 + sigmoid) * 2.0 ** -8)


@pytest.mark.parametrize("partial_dtype", [DTYPE_BF16, DTYPE_F32])
@pytest.mark.parametrize("hq,hkv,d,tile,partials", [(12, 2, 256, 8, 3), (12, 2, 256, 8, 9), (40, 8, 128, 2, 16), (12, 2, 128, 2, 40), (6, 1, 256, 1, 70)])
def test_reduce_of_buffers_aligned_to_four_bytes(device, hq, hkv, d, tile, partials, partial_dtype):
    """Every buffer a view that starts four bytes behind a 256-byte boundary: the same bytes as from whole allocations."""
    import torch

    units, dtype = 5, torch.bfloat16 if partial_dtype == DTYPE_BF16 else torch.float32
    tokens, templates = units * tile, units * partials
    generator = torch.Generator(device=device)
    generator.manual_seed(d + partials)
    randn = lambda n: torch.randn(n, device=device, generator=generator)  # noqa: E731
    rows = templates * hq * tile
    buffers = dict(partial_output=randn(rows * d).to(dtype), partial_exp_sums=randn(rows).abs() + 0.5, partial_max_logits=3.0 * randn(rows),
                   q_token_ranges=torch.tensor([(i * tile, (i + 1) * tile) for i in range(units)], dtype=torch.int32, device=device).flatten(),
                   cu_sdpa_partial_outputs=torch.arange(units + 1, dtype=torch.int32, device=device) * partials, gates=randn(tokens * hq * d).to(torch.bfloat16))
    config = sliced_q.Config(hq, hkv, d, d ** -0.5, 2 * 2 * hkv * 16 * d, sliced_q.Layout(1, 1, 4, 1), partial_dtype=partial_dtype)
    variant = sdpa.ExecutionVariant.sliced_q(config.sdpa_config(), sdpa.MAP_Q_TOKENS_AND_HEADS, tile, 64, hq // hkv)
    compute = sliced_q.Compute(config, variant, sliced_q.Shape(tokens, units, templates))

    def shifted(whole):
        lead = 4 // whole.element_size()
        view = torch.empty(whole.numel() + lead, dtype=whole.dtype, device=device)[lead:]
        assert view.data_ptr() % 8 == 4
        return view.copy_(whole)

    def run(place):
        output = place(torch.zeros(tokens * hq * d, dtype=torch.bfloat16, device=device))
        compute.invoke_reduce(output=output, num_active_q_token_tiles=ReplayU32.fixed(units), **{name: place(whole) for name, whole in buffers.items()})
        torch.cuda.synchronize()
        return output

    print(f"reduce of shifted buffers Hq{hq} D{d} tile={tile} partials={partials} f32={partial_dtype == DTYPE_F32}", flush=True)
    whole = run(lambda buffer: buffer)
    assert bool(whole.any()) and torch.equal(run(shifted).view(torch.int16), whole.view(torch.int16))
