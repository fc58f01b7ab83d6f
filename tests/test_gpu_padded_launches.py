"""Launches over padded domains: with a fixed active count the padding gets no blocks, with a replay parameter the launch covers
the whole domain and the kernel finds its work item from the active count.  Both must give the same bytes for every number of KV
heads (work items are dealt to the XCDs heads first), match the oracle on the active rows and leave the others alone."""
import numpy as np
import pytest

from khalamari_amd import sdpa, sliced_q
from khalamari_amd._lib import ReplayU32

from . import gpu_runner, helpers

pytestmark = pytest.mark.gpu
POISON = 0x4228


@pytest.mark.parametrize("hq,hkv,d,fp8,tile", [(8, 1, 128, False, 8), (16, 2, 128, True, 8), (12, 3, 128, False, 8), (24, 4, 256, True, 8),
                                                (40, 8, 128, False, 8), (36, 9, 128, True, 8), (64, 16, 128, False, 8), (60, 20, 128, True, 8),
                                                (32, 16, 256, False, 8), (64, 8, 128, False, 32), (64, 8, 128, True, 32), (36, 9, 128, True, 32),
                                                (12, 3, 256, True, 32), (24, 4, 256, True, 32)])
@pytest.mark.parametrize("direct", [False, True])
def test_fixed_and_replayed_counts_give_the_same_bytes(device, hq, hkv, d, fp8, tile, direct):
    import torch

    histories, q_lens = [5, 700, 0, 130, 64], [40, 3, 17, 1, 33]
    heads = hq // hkv
    w = helpers.make_workload(num_q_heads=hq, num_kv_heads=hkv, head_dim=d, tokens_per_page=16, histories=histories, q_lens=q_lens, seed=hq + d,
                              fp8_pages=fp8)
    ranges, templates, cu = helpers.fixed_slice_plan(histories, q_lens, tile, 4096 if direct else 200)
    pad = 9
    total = len(templates) + pad
    padded_templates = np.full((total, 3), 0xFFFFFFFF, dtype=np.uint32)
    padded_templates[:len(templates)] = templates
    total_ranges = total if direct else len(ranges) + pad
    padded_ranges = np.zeros((total_ranges, 2), dtype=np.uint32)
    padded_ranges[:len(ranges)] = ranges
    padded_cu = np.full(total_ranges + 1, cu[-1], dtype=np.uint32)
    padded_cu[:len(cu)] = cu
    config = gpu_runner.component_config(w, sliced_q.Config)
    variant = sdpa.ExecutionVariant.sliced_q(config.sdpa_config(), sdpa.MAP_Q_TOKENS_AND_HEADS, tile, 64, heads)
    shape = sliced_q.Shape(w.num_tokens, total_ranges, total)
    compute = sliced_q.Compute(config, variant, shape, direct=direct)
    dev = lambda a: gpu_runner.to_device(a, device)  # noqa: E731
    q, pages, slots, table, vis = map(dev, (w.q_bits, w.kv_pages, w.req_slots, w.page_ids, w.visible))
    ranges_d, templates_d, cu_d = map(dev, (padded_ranges, padded_templates, padded_cu))
    partial = torch.zeros(config.partial_output_bytes(variant, shape), dtype=torch.uint8, device=device)
    sums = torch.zeros(config.partial_output_stats_bytes(variant, shape), dtype=torch.uint8, device=device)
    maxs = torch.zeros_like(sums)
    expected = helpers.expected_output(w)

    def run(tokens, tiles, splits, params):
        out = torch.full((w.num_tokens, hq, d), POISON, dtype=torch.int16, device=device)
        common = dict(q=q, kv_pages=pages, req_slots=slots, page_ids=table, visible_kv_token_ranges=vis, q_token_ranges=ranges_d,
                      sdpa_map_task_templates=templates_d, page_table_index=ReplayU32.fixed(w.layer), num_active_tokens=tokens,
                      num_active_q_token_tiles=tiles, replay_parameters=params)
        if direct:
            compute.invoke_direct(output=out, **common)
        else:
            compute.invoke_map(partial_output=partial, partial_exp_sums=sums, partial_max_logits=maxs, num_active_kv_splits=splits, **common)
            compute.invoke_reduce(partial_output=partial, partial_exp_sums=sums, partial_max_logits=maxs, q_token_ranges=ranges_d,
                                  cu_sdpa_partial_outputs=cu_d, output=out, num_active_q_token_tiles=tiles, replay_parameters=params)
        torch.cuda.synchronize()
        return out

    for active_requests in (5, 3, 1):
        tokens = int(sum(q_lens[:active_requests]))
        tiles = int(sum(-(-n // tile) for n in q_lens[:active_requests]))
        splits = int(cu[tiles])
        print(f"padded launch Hq{hq}/Hkv{hkv}/D{d} fp8={fp8} tile={tile} direct={direct} requests={active_requests}", flush=True)
        params = torch.tensor([tokens, tiles, splits, 0], dtype=torch.int32, device=device)
        fixed = run(*(ReplayU32.fixed(x) for x in (tokens, tiles, splits)), None)
        replayed = run(*(ReplayU32.parameter(i) for i in range(3)), params)
        assert torch.equal(fixed, replayed)
        helpers.assert_parity(gpu_runner.bf16_tensor_to_f32(fixed)[:tokens], expected[:tokens], f"{active_requests} requests")
        assert np.all(fixed[tokens:].cpu().numpy() == POISON)
        if active_requests == 5 and not direct:
            # a replayed count beyond the shape stands for the whole table: no template is read behind it, padding has no Q range
            beyond = torch.tensor([tokens, tiles, total + 7, 0], dtype=torch.int32, device=device)
            assert torch.equal(fixed, run(*(ReplayU32.parameter(i) for i in range(3)), beyond))
