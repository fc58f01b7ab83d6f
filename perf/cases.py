"""The attention work a serving program hands to this library, as cases that can be timed.

A case is one pass of a GQA layer between its input and its output projection (or of several layers of one step): the
projection rows of a batch of requests become Q rows, gate rows and K/V rows in the paged cache, and the batch attends over
the cache.  A batch is what the executor schedules: requests that decode one token, verify a few drafted ones, or run a
chunk of a prompt, in any mixture, each with its own history.  The lengths come from the case alone, the values and the
page permutation from the seed.

Fields of a case
  hq, hkv, d            head geometry
  page, fp8             tokens per page; FP8 E4M3FN or bf16 pages
  gated                 projection rows carry a gate half per Q head; the attention output is multiplied with its sigmoid
  rope, yarn, w32       rotary dims, Yarn scaling, float32 norm weights
  requests, q_lo, q_hi  requests and their new tokens (uniform)
  chunks, chunk         how many of the requests run a chunk of `chunk` tokens instead
  hist_lo, hist_hi      tokens already cached per request (uniform)
  lengths               seed of the lengths
  slice                 KV tokens per partition; 0 leaves the partition to the selector
  separate              the layer recorded operator by operator (split, Q norm + RoPE, K norm + RoPE, page write, Map, Reduce,
                        gate) instead of in its shortest form
  layers, step          layers of the pass; a whole step also plans the batch (selector, metadata) and replays the recorded
                        layers from a HIP graph
  block                 > 0: a proposal block of that many tokens per request (history Map, dense block partial, Reduce)
"""
import gc
from types import SimpleNamespace

import numpy as np
import torch

from khalamari_amd import (activation_gate, batch_metadata, bidi_block_metadata, bidi_block_sdpa, k_norm_rope_page_write, kv_page_write,
                           projection_norm_rope_page_write, qgkv_split, qkv_split, rms_norm_rope, sdpa, sliced_kv, sliced_q)
from khalamari_amd._lib import DTYPE_BF16, DTYPE_F32, DTYPE_FP8_E4M3FN, ReplayU32
from khalamari_amd.replay import ReplayBucketPolicy
from khalamari_amd.selector import GQAReplayBucketPolicy, RequestShape, Selector

DEVICE = "cuda:0"
GEOMETRIES = ((32, 8, 128), (64, 8, 128), (24, 4, 256), (16, 2, 256), (40, 8, 128), (32, 4, 128))
DEFAULTS = dict(hq=64, hkv=8, d=128, page=16, fp8=False, gated=False, rope=128, yarn=False, w32=False, requests=1, q_lo=1, q_hi=1, chunks=0,
                chunk=0, hist_lo=0, hist_hi=0, lengths=1, slice=0, separate=False, layers=1, step=False, block=0)
# The most one drawn case may read from the cache and compute: below the largest listed cases.
MOST_CACHE_BYTES = 1.2e9
MOST_FLOPS = 3.0e12
# One launch merges its own partial states where the step is bound by launches; above this many bytes of K/V the Map and the
# Reduce are two launches (the rule the benchmark uses).
ONE_LAUNCH_KV_BYTES = 64 << 20


def _case(**fields):
    return {**DEFAULTS, **fields}


def listed():
    return [
        # one user's conversation, decoded token by token: latency and launches are everything
        _case(name="decode_single", hq=32, hkv=8, d=128, rope=128, requests=1, hist_lo=1023, hist_hi=1023),
        # a small server's decode step, planned and replayed from a graph for several layers
        _case(name="decode_step", hq=24, hkv=4, d=256, rope=64, fp8=True, gated=True, requests=12, hist_lo=200, hist_hi=3000, layers=4, step=True),
        # the benchmark's decode batch: 32 ragged contexts in partitions of 512 tokens, bf16 pages
        _case(name="decode_batch", requests=32, hist_lo=511, hist_hi=8191, lengths=2, slice=512),
        # a fuller batch on FP8 pages, partitioned by the selector
        _case(name="decode_batch_fp8", fp8=True, gated=True, requests=45, hist_lo=300, hist_hi=12000, lengths=3),
        # long documents: four contexts of 131072 tokens, partitions of 2048, gated
        _case(name="decode_long_fp8", hq=24, hkv=4, d=256, rope=256, fp8=True, gated=True, requests=4, hist_lo=131071, hist_hi=131071, slice=2048),
        # speculative decoding: 2 to 5 tokens a request are verified
        _case(name="verify", requests=16, q_lo=2, q_hi=5, hist_lo=4096, hist_hi=32768, lengths=4),
        _case(name="verify_d256_fp8", hq=24, hkv=4, d=256, rope=64, fp8=True, gated=True, requests=23, q_lo=2, q_hi=5, hist_lo=1000, hist_hi=20000, lengths=5),
        # chunked prefill of long prompts: the largest compute
        _case(name="prefill_chunks", requests=8, q_lo=2048, q_hi=2048, hist_lo=0, hist_hi=16384, lengths=5),
        # short chunks far into long documents (a few hundred new tokens over a long prefix)
        _case(name="chunk_on_long_fp8", hq=24, hkv=4, d=256, rope=256, fp8=True, gated=True, requests=3, q_lo=64, q_hi=256, hist_lo=10000, hist_hi=66000, lengths=6),
        # fresh prompts of chat length, nothing cached, recorded operator by operator
        _case(name="prompts", hq=32, hkv=8, d=128, gated=True, requests=9, q_lo=20, q_hi=900, lengths=7, separate=True),
        # continuous batching: a chunk of a new prompt beside requests that decode
        _case(name="mixed_fp8", fp8=True, gated=True, requests=27, q_lo=1, q_hi=1, chunks=2, chunk=500, hist_lo=100, hist_hi=6000, lengths=8),
        # block drafting: sixteen proposed tokens a request attend to their block and to the history
        _case(name="proposal", hq=32, hkv=8, d=128, fp8=True, requests=40, block=16, hist_lo=200, hist_hi=5000, lengths=9),
    ]


def _log_uniform(rng, low, high):
    return int(round(low * (high / low) ** rng.random()))


def draw(rng):
    while True:
        hq, hkv, d = rng.choice(GEOMETRIES)
        case = _case(hq=hq, hkv=hkv, d=d, page=rng.choice((8, 16, 16, 16)), fp8=rng.random() < 0.5, gated=rng.random() < 0.5,
                     rope=rng.choice((d, d, 64)), yarn=rng.random() < 0.2, w32=rng.random() < 0.2, lengths=rng.randrange(1 << 20),
                     separate=rng.random() < 0.25)
        family = rng.choice(("decode", "decode", "step", "verify", "verify", "prefill", "prefill", "mixed", "proposal"))
        if family in ("decode", "step"):
            longest = _log_uniform(rng, 100, 100000 if family == "decode" else 8000)
            case.update(requests=_log_uniform(rng, 1, 96 if family == "decode" else 32), hist_lo=longest // rng.choice((1, 4, 20)), hist_hi=longest,
                        slice=rng.choice((0, 0, 512, 2048)))
            if family == "step":
                case.update(step=True, layers=rng.choice((2, 4, 6)), slice=0)
        elif family == "verify":
            longest = _log_uniform(rng, 200, 60000)
            case.update(requests=_log_uniform(rng, 1, 48), q_lo=2, q_hi=rng.choice((3, 5, 8)), hist_lo=longest // rng.choice((1, 4, 20)), hist_hi=longest)
        elif family == "prefill":
            new = _log_uniform(rng, 24, 2048)
            prefix = rng.choice((0, _log_uniform(rng, 100, 30000)))
            case.update(requests=_log_uniform(rng, 1, 12), q_lo=max(1, new // rng.choice((1, 8))), q_hi=new, hist_lo=prefix // 4, hist_hi=prefix)
        elif family == "mixed":
            longest = _log_uniform(rng, 200, 20000)
            requests = _log_uniform(rng, 3, 64)
            case.update(requests=requests, q_hi=rng.choice((1, 1, 4)), chunks=rng.choice((1, 1, 2)), chunk=_log_uniform(rng, 60, 1500), hist_lo=longest // 20,
                        hist_hi=longest)
        else:
            longest = _log_uniform(rng, 50, 20000)
            case.update(requests=_log_uniform(rng, 2, 64), block=rng.choice((4, 7, 8, 16)), hist_lo=max(1, longest // 10), hist_hi=longest, gated=False,
                        separate=False, yarn=False, w32=False, rope=d)
        if _cache_bytes(case) <= MOST_CACHE_BYTES and _flops(case) <= MOST_FLOPS:
            return case


# ---- lengths and work ------------------------------------------------------------------------------------------------------


def _lengths(case):
    """(histories, new tokens) of the requests."""
    rng = np.random.default_rng(case["lengths"])
    histories = rng.integers(case["hist_lo"], case["hist_hi"] + 1, size=case["requests"])
    new = rng.integers(case["q_lo"], case["q_hi"] + 1, size=case["requests"])
    if case["chunks"]:
        new[rng.permutation(case["requests"])[:case["chunks"]]] = case["chunk"]
    if case["block"]:
        new[:] = case["block"]
    return [int(x) for x in histories], [int(x) for x in new]


def _cache_bytes(case):
    """K and V bytes of every token the requests see, once."""
    histories, new = _lengths(case)
    visible = sum(histories) + (0 if case["block"] else sum(new))
    return case["layers"] * visible * 2 * case["hkv"] * case["d"] * (1 if case["fp8"] else 2)


def _flops(case):
    histories, new = _lengths(case)
    if case["block"]:
        pairs = sum(n * (h + n) for h, n in zip(histories, new))
    else:
        pairs = sum(n * h + n * (n + 1) // 2 for h, n in zip(histories, new))
    return case["layers"] * 4 * case["hq"] * case["d"] * pairs


def work(case):
    histories, new = _lengths(case)
    tokens, hq, hkv, d = sum(new), case["hq"], case["hkv"], case["d"]
    output = tokens * hq * d * 2
    table = sum(-(-(h + n) // case["page"]) for h, n in zip(histories, new)) * 4
    if case["block"]:
        rows = tokens * (hq + 2 * hkv) * d * 2     # Q rows and the block's own K and V rows
        return {"bytes": _cache_bytes(case) + rows + output + table, "flops": _flops(case)}
    rows = tokens * ((2 if case["gated"] else 1) * hq + 2 * hkv) * d * 2
    written = tokens * 2 * hkv * d * (1 if case["fp8"] else 2)
    return {"bytes": _cache_bytes(case) + case["layers"] * (rows + written + output + table), "flops": _flops(case)}


def tolerance(case):
    # bf16 results with float32 sums.  Against the same layers in float64 on the same projection rows and cache, the outputs of
    # seven of the listed cases are off by 3.8e-3 to 5.5e-3 in the 2-norm and by up to 0.05 at their worst value (Q rows, partial states,
    # softmax weights and the gate's steps are bf16 on the way).  Cache bytes are the same to the bit.
    return {"rel": 1.6e-2, "max": 0.2}


# ---- states ------------------------------------------------------------------------------------------------------------------


def _randn(shape, generator):
    return torch.randn(shape, device=DEVICE, dtype=torch.float32, generator=generator).to(torch.bfloat16)


def _cache(case, histories, new, seed, generator):
    """(pool, page table, blocks per request): pages permuted over the pool, every layer with pages of its own."""
    layers, tpp = case["layers"], case["page"]
    pages = [-(-(h + n) // tpp) for h, n in zip(histories, new)]
    blocks = max(pages)
    order = np.random.default_rng(seed).permutation(layers * sum(pages)).astype(np.int32)
    table = np.zeros((len(pages), layers, blocks), dtype=np.int32)
    at = 0
    for r, count in enumerate(pages):
        for layer in range(layers):
            table[r, layer, :count] = order[at:at + count]
            at += count
    values = order.size * 2 * case["hkv"] * tpp * case["d"]
    if case["fp8"]:
        pool = torch.empty(values, dtype=torch.uint8, device=DEVICE)
        step = 1 << 28
        for first in range(0, values, step):
            part = pool[first:first + step]
            kv_page_write.fp8_encode_device(_randn((part.numel(),), generator), part, part.numel())
    else:
        pool = _randn((values,), generator)
    return pool, torch.from_numpy(table).to(DEVICE), blocks


def prepare(case, seed):
    torch.cuda.set_device(DEVICE)
    generator = torch.Generator(device=DEVICE)
    generator.manual_seed(seed)
    return _prepare_block(case, seed, generator) if case["block"] else _prepare_layers(case, seed, generator)


def _prepare_layers(case, seed, generator):
    hq, hkv, d, tpp, gated, layers = (case[k] for k in ("hq", "hkv", "d", "page", "gated", "layers"))
    histories, new = _lengths(case)
    requests, tokens = len(new), sum(new)
    s = SimpleNamespace(case=case, histories=histories, requests=requests, cu=[0], graph=None)
    for n in new:
        s.cu.append(s.cu[-1] + n)
    s.pool, s.page_ids, blocks = _cache(case, histories, new, seed, generator)
    kv_dtype = DTYPE_FP8_E4M3FN if case["fp8"] else DTYPE_BF16
    page_bytes = 2 * hkv * tpp * d * (1 if case["fp8"] else 2)

    # the plan of the batch: selector and metadata
    sconfig = sdpa.Config(DTYPE_BF16, hq, hkv, d, tpp)
    layout = sliced_kv.Layout(requests, layers, blocks, 1)
    s.total = ReplayBucketPolicy(max(tokens, 1)).capacity(tokens) if case["step"] else tokens
    s.variant = None
    if case["slice"] and max(new) == 1 and hq // hkv <= 8:
        s.variant = sdpa.ExecutionVariant.sliced_kv(sconfig, d, 128, min(hq // hkv, 8))
        most = max(-(-(h + 1) // case["slice"]) for h in histories)
        s.selector = Selector.for_partitions(sdpa.Registry.from_variants(sconfig, [s.variant]), s.total, requests, lambda v: most)
    else:
        s.selector = Selector.for_lookup(sconfig, s.total, layout)
    limits = s.selector.limits()
    s.policy = GQAReplayBucketPolicy(limits.max_tokens, limits.max_map_task_templates)
    s.metadata = batch_metadata.GQAMetadataBuffers(limits.max_tokens, limits.max_map_task_templates)
    selection, shape = _plan(s)
    variant, direct = selection.variant(), selection.direct_output()

    # rows, weights, outputs and scratch
    rows = lambda heads: torch.zeros((s.total, heads, d), dtype=torch.bfloat16, device=DEVICE)  # noqa: E731
    width = ((2 if gated else 1) * hq + 2 * hkv) * d
    s.projection = [_randn((s.total, width), generator) for _ in range(layers)]
    weight = lambda: (0.75 + 0.5 * torch.rand(d, device=DEVICE, generator=generator)).to(torch.float32 if case["w32"] else torch.bfloat16)  # noqa: E731
    q_weights, k_weights = [weight() for _ in range(layers)], [weight() for _ in range(layers)]
    s.out = [rows(hq) for _ in range(layers)]
    q, gate = rows(hq), rows(hq) if gated else None

    def norm(heads):
        config = rms_norm_rope.Config.bf16(heads, d, case["rope"], 1e-6, 1_000_000.0).with_norm_weight_dtype(DTYPE_F32 if case["w32"] else DTYPE_BF16)
        return config.with_rope_scaling(rms_norm_rope.Yarn(8.0, 1.2, 32.0, 1.0, 8192, True)) if case["yarn"] else config

    page_config = kv_page_write.Config(hkv, d, page_bytes, kv_dtype=kv_dtype)
    page_shape = kv_page_write.Shape(s.total, kv_page_write.PageTableLayout(requests, layers, blocks, 1))
    md = s.metadata
    req_slots, positions, visible, q_ranges = md.req_slots(), md.flat_token_indices(), md.visible_kv_token_ranges(), md.q_token_ranges()
    templates, cu_partial = md.sdpa_map_task_templates(), md.cu_sdpa_partial_outputs()
    if case["step"]:
        s.params = torch.zeros(4, dtype=torch.int32, device=DEVICE)
        _upload(s, shape)
        count, tiles, splits, params = ReplayU32.parameter(0), ReplayU32.parameter(1), ReplayU32.parameter(2), s.params
    else:
        fixed = ReplayU32.fixed
        count, tiles, splits, params = fixed(shape.num_tokens), fixed(shape.num_q_token_tiles), fixed(shape.num_sdpa_map_task_templates), None

    if case["separate"]:
        k, v, k_normed, attended = rows(hkv), rows(hkv), rows(hkv), rows(hq)
        split_config = (qgkv_split if gated else qkv_split).Config.bf16(hq, hkv, d)
        split, split_shape = (qgkv_split if gated else qkv_split).Compute(split_config), qgkv_split.Shape(s.total)
        q_rows = rows(hq)
        q_norm, k_norm, writer = rms_norm_rope.Compute(norm(hq)), rms_norm_rope.Compute(norm(hkv)), kv_page_write.Compute(page_config)
        row_shape = rms_norm_rope.Shape(s.total)

        def produce(layer):
            if gated:
                split.invoke(split_shape, qgkv=s.projection[layer], q=q_rows, g=gate, k=k, v=v, num_active_tokens=count, replay_parameters=params)
            else:
                split.invoke(split_shape, qkv=s.projection[layer], q=q_rows, k=k, v=v, num_active_tokens=count, replay_parameters=params)
            q_norm.invoke(row_shape, input=q_rows, norm_weight=q_weights[layer], flat_token_indices=positions, output=q,
                          num_active_tokens=count, replay_parameters=params)
            k_norm.invoke(row_shape, input=k, norm_weight=k_weights[layer], flat_token_indices=positions, output=k_normed,
                          num_active_tokens=count, replay_parameters=params)
            writer.invoke(page_shape, pages=s.pool, flat_k=k_normed, flat_v=v, req_slots=req_slots, flat_token_indices=positions,
                          page_ids=s.page_ids, num_active_token_writes=count, page_table_index=ReplayU32.fixed(layer), replay_parameters=params)
    else:
        prologue = projection_norm_rope_page_write.Compute(norm(hq), norm(hkv), page_config, gated=gated)

        def produce(layer):
            prologue.invoke(page_shape, projection=s.projection[layer], q_norm_weight=q_weights[layer], k_norm_weight=k_weights[layer], q_output=q,
                            gate_output=gate, pages=s.pool, req_slots=req_slots, flat_token_indices=positions, page_ids=s.page_ids,
                            num_active_tokens=count, page_table_index=ReplayU32.fixed(layer), replay_parameters=params)

    fused_gate = gate if gated and not case["separate"] else None
    if variant.map_kind == sdpa.MAP_SLICED_KV:
        config = sliced_kv.Config(hq, hkv, d, d ** -0.5, page_bytes, layout, DTYPE_BF16, kv_dtype)
        kshape = sliced_kv.Shape(shape.num_total_tokens, shape.num_total_sdpa_map_task_templates)
        compute, scratch = sliced_kv.Compute(config, variant, kshape), sliced_kv.Scratch(DEVICE, config, kshape)
        one_launch = not case["separate"] and _cache_bytes(case) // layers < ONE_LAUNCH_KV_BYTES
        counters = torch.zeros(compute.arrival_counters_bytes(), dtype=torch.uint8, device=DEVICE)
        partial = dict(partial_exp_sums=scratch.partial_exp_sums, partial_max_logits=scratch.partial_max_logits, partial_output=scratch.partial_output)

        def attend(layer, output):
            batch = dict(q=q, kv_pages=s.pool, req_slots=req_slots, page_ids=s.page_ids, sdpa_map_task_templates=templates,
                         page_table_index=ReplayU32.fixed(layer), num_active_tokens=count, num_active_kv_splits=splits, replay_parameters=params, **partial)
            if one_launch:
                compute.invoke_map_reduce(cu_sdpa_partial_outputs=cu_partial, output=output, arrival_counters=counters, gates=fused_gate, **batch)
                return
            compute.invoke_map(**batch)
            compute.invoke_reduce(cu_sdpa_partial_outputs=cu_partial, output=output, num_active_tokens=count, gates=fused_gate,
                                  replay_parameters=params, **partial)
    else:
        config = sliced_q.Config(hq, hkv, d, d ** -0.5, page_bytes, layout, DTYPE_BF16, kv_dtype)
        qshape = sliced_q.Shape(shape.num_total_tokens, shape.num_total_q_token_tiles, shape.num_total_sdpa_map_task_templates)
        compute = sliced_q.Compute.new_direct(config, variant, qshape) if direct else sliced_q.Compute.new(config, variant, qshape)
        if not direct:
            zeros = lambda count_: torch.zeros(count_, dtype=torch.uint8, device=DEVICE)  # noqa: E731
            partial = dict(partial_output=zeros(config.partial_output_bytes(variant, qshape)), partial_exp_sums=zeros(config.partial_output_stats_bytes(variant, qshape)),
                           partial_max_logits=zeros(config.partial_output_stats_bytes(variant, qshape)))

        def attend(layer, output):
            batch = dict(q=q, kv_pages=s.pool, req_slots=req_slots, page_ids=s.page_ids, visible_kv_token_ranges=visible,
                         q_token_ranges=q_ranges, sdpa_map_task_templates=templates, page_table_index=ReplayU32.fixed(layer),
                         num_active_tokens=count, num_active_q_token_tiles=tiles, replay_parameters=params)
            if direct:
                compute.invoke_direct(output=output, gates=fused_gate, **batch)
                return
            compute.invoke_map(num_active_kv_splits=splits, **batch, **partial)
            compute.invoke_reduce(q_token_ranges=q_ranges, cu_sdpa_partial_outputs=cu_partial, output=output,
                                  num_active_q_token_tiles=tiles, gates=fused_gate, replay_parameters=params, **partial)

    def record():
        for layer in range(layers):
            produce(layer)
            if gated and case["separate"]:
                attend(layer, attended)
                activation_gate.invoke(DTYPE_BF16, hq, d, s.total, attended, gate, s.out[layer], count, replay_parameters=params)
            else:
                attend(layer, s.out[layer])

    s.record = record
    if case["step"]:
        record()
        torch.cuda.synchronize()
        gc.collect()
        gc.disable()   # a collector run could free device memory, which ends the capture
        try:
            s.graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(s.graph):
                record()
        finally:
            gc.enable()
    return s


def _plan(s):
    shapes = RequestShape.from_batch(s.histories, s.cu)
    if s.variant is not None:
        selection = s.selector.select_partitioned(s.variant, s.case["slice"], False, shapes, s.policy, s.total)
    else:
        selection = s.selector.select(shapes, s.policy, s.total)
    return selection, s.metadata.update(list(range(s.requests)), s.histories, s.cu, selection)


def _upload(s, shape):
    counts = torch.tensor([shape.num_tokens, shape.num_q_token_tiles, shape.num_sdpa_map_task_templates, 0], dtype=torch.int32, pin_memory=True)
    s.params.copy_(counts, non_blocking=True)


def _prepare_block(case, seed, generator):
    hq, hkv, d, tpp, block = (case[k] for k in ("hq", "hkv", "d", "page", "block"))
    histories, new = _lengths(case)
    requests, tokens = len(new), sum(new)
    s = SimpleNamespace(case=case, graph=None)
    s.pool, s.page_ids, blocks = _cache(case, histories, [0] * requests, seed, generator)
    kv_dtype = DTYPE_FP8_E4M3FN if case["fp8"] else DTYPE_BF16
    page_bytes = 2 * hkv * tpp * d * (1 if case["fp8"] else 2)
    variant, capacity = bidi_block_metadata.select(sdpa.Config(DTYPE_BF16, hq, hkv, d, tpp), requests, block)
    indices = [h + i for h in histories for i in range(block)]
    ranges = [(0, h) for h in histories for _ in range(block)]
    meta = bidi_block_metadata.build(list(range(requests)), indices, ranges, block, variant, capacity.max_sdpa_map_task_templates)
    shape = meta.replay_shape
    device = lambda a: torch.from_numpy(np.ascontiguousarray(a).view(np.int32)).to(DEVICE)  # noqa: E731
    req_slots, visible, q_ranges = device(meta.req_slots), device(meta.visible_kv_token_ranges), device(meta.q_token_ranges)
    templates, cu = device(meta.sdpa_map_task_templates), device(meta.cu_sdpa_partial_outputs)
    q, local_k, local_v = _randn((tokens, hq, d), generator), _randn((tokens, hkv, d), generator), _randn((tokens, hkv, d), generator)
    s.out = [torch.zeros((tokens, hq, d), dtype=torch.bfloat16, device=DEVICE)]
    config = sliced_q.Config(hq, hkv, d, d ** -0.5, page_bytes, sliced_kv.Layout(requests, 1, blocks, 1), DTYPE_BF16, kv_dtype)
    qshape = sliced_q.Shape(shape.num_total_tokens, shape.num_total_q_token_tiles, shape.num_total_sdpa_map_task_templates)
    compute = sliced_q.Compute.new(config, variant, qshape)
    zeros = lambda count: torch.zeros(count, dtype=torch.uint8, device=DEVICE)  # noqa: E731
    partial = dict(partial_output=zeros(config.partial_output_bytes(variant, qshape)), partial_exp_sums=zeros(config.partial_output_stats_bytes(variant, qshape)),
                   partial_max_logits=zeros(config.partial_output_stats_bytes(variant, qshape)))
    block_sdpa = bidi_block_sdpa.Compute(bidi_block_sdpa.Config(block, int(variant.map_max_q_tokens), hq, hkv, d, d ** -0.5, DTYPE_BF16))
    block_shape = bidi_block_sdpa.Shape(shape.num_total_tokens, shape.num_total_q_token_tiles, shape.num_total_sdpa_map_task_templates)
    fixed = ReplayU32.fixed
    count, tiles, splits = fixed(shape.num_tokens), fixed(shape.num_q_token_tiles), fixed(shape.num_sdpa_map_task_templates)

    def record():
        compute.invoke_map(q=q, kv_pages=s.pool, req_slots=req_slots, page_ids=s.page_ids, visible_kv_token_ranges=visible, q_token_ranges=q_ranges,
                           sdpa_map_task_templates=templates, page_table_index=fixed(0), num_active_tokens=count, num_active_q_token_tiles=tiles,
                           num_active_kv_splits=splits, **partial)
        block_sdpa.invoke(block_shape, tiles, q=q, local_k=local_k, local_v=local_v, q_token_ranges=q_ranges, cu_sdpa_partial_outputs=cu, **partial)
        compute.invoke_reduce(q_token_ranges=q_ranges, cu_sdpa_partial_outputs=cu, output=s.out[0], num_active_q_token_tiles=tiles, **partial)

    s.record = record
    return s


def run(state):
    if state.case["step"]:
        _, shape = _plan(state)
        _upload(state, shape)
        state.graph.replay()
    else:
        state.record()
    # the block drafting pass leaves the cache as it was
    return {"attention": state.out} if state.case["block"] else {"attention": state.out, "cache": state.pool}
