"""The work that a serving program has this library do, as cases that can be
timed and checked: the KV-cache transfer of prefill/decode disaggregation
(pack, unpack, pool to pool, the forward pass's K/V row writes) and the paged
attention that reads the same pools (decode, prefill, chunked prefill, the
verification of drafted tokens), each through the public Python binding.

A case is a dict of plain values. ``op`` names the path:

  write      the forward pass's drop-in scatter of new K/V rows into their
             slots, one synchronous call a layer
  relay      pack of every layer into transfer rows, unpack into the decode
             pool (one launch for all layers, or one a layer)
  transfer   pool to pool over all layers in one launch
  attend     paged attention over bf16 pages, one asynchronous call a layer

The byte and flop counts of ``work`` are what the path cannot do without:
each payload byte, K/V row, query and output moved once per direction.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sglang-rs_amd"))
import sgl_rocm_kv as kv  # noqa: E402

_GOLDEN = 0.6180339887498949
_context = None


def _kernels():
    """One context a process, as a serving program keeps it."""
    global _context
    if _context is None:
        _context = kv.RocmKvPairCopyKernels(0)
    return _context


def _buffer(t):
    return kv.device_buffer(t.data_ptr(), t.numel() * t.element_size())


def _ragged(count, low, high):
    """`count` lengths spread evenly over [low, high], in a scattered order;
    the first is `high`."""
    return [low + round((high - low) * (1.0 - (i * _GOLDEN) % 1.0)) for i in range(count)]


# ---- the listed cases -----------------------------------------------------------------------


def listed():
    return [
        # One decode step's new K/V rows of 64 requests (Llama-3-8B rows, 8 KV heads x 128):
        # the smallest call, all launch and synchronisation.
        dict(name="write_llama8b_64", op="write", rows=64, layers=8, heads=8, dim=128, page=64),
        # A handful of short requests of a small model (Qwen2-0.5B: 24 layers, 2 KV heads x 64),
        # token-paged prefill pool to 16-token decode pages: the small transfer.
        dict(name="relay_qwen_4978", op="relay", rows=4978, layers=24, heads=2, dim=64, elt=2, src_page=1,
             dst_page=16, hnd=False, per_layer=False, packed=False),
        # The headline transfer's layers: 64 requests x 2,048 tokens of Llama-3-8B rows, layer by layer.
        dict(name="relay_llama8b_131072", op="relay", rows=131072, layers=4, heads=8, dim=128, elt=2, src_page=1,
             dst_page=64, hnd=False, per_layer=True, packed=False),
        # DeepSeek's packed MLA rows of 649 bytes: no row starts on a vector.
        dict(name="relay_mla649_30011", op="relay", rows=30011, layers=16, heads=1, dim=649, elt=1, src_page=64,
             dst_page=64, hnd=False, per_layer=True, packed=True),
        # Co-resident pools, fp8 Llama-3.2-1B rows into head-major pages (64-byte head chunks).
        dict(name="transfer_fp8_hnd_40000", op="transfer", rows=40000, layers=16, heads=8, dim=64, elt=1,
             src_page=1, dst_page=64, hnd=True),
        # One user's decode step over 4,096 tokens (Llama-3-8B): latency.
        dict(name="decode_llama8b_1", op="attend", queries=1, per_request=1, low=4096, high=4096, layers=8,
             qheads=32, heads=8, dk=128, dv=128, page=64, hnd=False),
        # A full decode batch, ragged up to 4,096 tokens.
        dict(name="decode_llama8b_64", op="attend", queries=64, per_request=1, low=100, high=4096, layers=4,
             qheads=32, heads=8, dk=128, dv=128, page=64, hnd=False),
        # Llama-3.2-1B (64-wide heads) on the head-major pages that the transfer can write.
        dict(name="decode_llama1b_hnd_16", op="attend", queries=16, per_request=1, low=300, high=3001, layers=4,
             qheads=32, heads=8, dk=64, dv=64, page=64, hnd=True),
        # DeepSeek-V3's latent decode: 128 query heads over one 576/512-wide latent head.
        dict(name="decode_mla_32", op="attend", queries=32, per_request=1, low=1000, high=8192, layers=2,
             qheads=128, heads=1, dk=576, dv=512, page=64, hnd=False),
        # Causal prefill of four ragged prompts (one query per prompt token, as the reference's
        # scheduler metadata has it).
        dict(name="prefill_llama8b_4", op="attend", queries=0, per_request=0, requests=4, low=300, high=2048,
             layers=1, qheads=32, heads=8, dk=128, dv=128, page=64, hnd=False),
        # The last 384 tokens of a 6,144-token prompt whose prefix is cached (Qwen2-0.5B: 7 query
        # heads per KV head, 16-token pages).
        dict(name="chunk_qwen_384", op="attend", queries=384, per_request=384, low=6144, high=6144, layers=2,
             qheads=14, heads=2, dk=64, dv=64, page=16, hnd=False),
        # Verification of drafted tokens: five positions of each of 24 requests (dims 256, 8 query
        # heads over 2 KV heads, Qwen3.5's full-attention layers).
        dict(name="verify_qwen256_24x5", op="attend", queries=120, per_request=5, low=200, high=3000, layers=2,
             qheads=8, heads=2, dk=256, dv=256, page=64, hnd=False),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    """One more case: a path, a model's shape and sizes over the range that
    the listed cases span (the largest never above the largest listed one)."""
    kind = rng.choice(["write", "relay", "relay", "transfer", "decode", "decode", "decode", "mla", "prefill",
                       "prefill", "chunk", "verify"])
    heads, dim = rng.choice([(8, 128), (2, 64), (8, 64), (1, 128), (4, 128)])
    if kind == "write":
        return dict(op="write", rows=_log(rng, 1, 1024), layers=8, heads=heads, dim=dim,
                    page=rng.choice([1, 16, 64]))
    if kind in ("relay", "transfer"):
        packed = kind == "relay" and rng.random() < 0.25
        elt = 1 if packed else rng.choice([1, 2])
        if packed:
            heads, dim = 1, 649
        layers = rng.choice([4, 16, 24])
        most = min(131072, (1 << 31) // (layers * (1 if packed else 2) * heads * dim * elt))
        rows = _log(rng, 300, most)
        hnd = not packed and rng.random() < 0.4
        case = dict(op=kind, rows=rows, layers=layers, heads=heads, dim=dim, elt=elt,
                    src_page=64 if packed else rng.choice([1, 16]), dst_page=rng.choice([16, 64]), hnd=hnd)
        if kind == "relay":
            case.update(per_layer=rows * heads * dim * elt > (1 << 24), packed=packed)
        return case
    if kind == "mla":
        high = _log(rng, 500, 8192)
        return dict(op="attend", queries=rng.randint(1, 32), per_request=1, low=max(1, high // 8), high=high,
                    layers=2, qheads=128, heads=1, dk=576, dv=512, page=64, hnd=False)
    qheads, heads, dim = rng.choice([(32, 8, 128), (14, 2, 64), (32, 8, 64), (8, 2, 256), (8, 1, 128)])
    page, hnd = rng.choice([16, 64]), rng.random() < 0.3
    if kind == "decode":
        high = _log(rng, 64, 4096)
        return dict(op="attend", queries=_log(rng, 1, 64), per_request=1, low=max(1, high // rng.choice([1, 4, 16])),
                    high=high, layers=4, qheads=qheads, heads=heads, dk=dim, dv=dim, page=page, hnd=hnd)
    if kind == "prefill":
        high = _log(rng, 40, 2048)
        return dict(op="attend", queries=0, per_request=0, requests=rng.randint(1, 6), low=max(1, high // 8),
                    high=high, layers=1, qheads=qheads, heads=heads, dk=dim, dv=dim, page=page, hnd=hnd)
    if kind == "chunk":
        high = _log(rng, 600, 6144)
        per = rng.randint(48, 512)
        return dict(op="attend", queries=per, per_request=per, low=high, high=high, layers=2, qheads=qheads,
                    heads=heads, dk=dim, dv=dim, page=page, hnd=hnd)
    high = _log(rng, 200, 3000)
    per, requests = rng.randint(2, 8), rng.randint(1, 24)
    return dict(op="attend", queries=per * requests, per_request=per, low=max(per, high // 8), high=high, layers=2,
                qheads=qheads, heads=heads, dk=dim, dv=dim, page=page, hnd=hnd)


# ---- inputs ---------------------------------------------------------------------------------


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _random_bytes(g, count):
    """`count` random bytes (whole 8-byte words) on the GPU."""
    words = torch.randint(-(1 << 63), (1 << 63) - 1, (-(-count // 8),), generator=g, device="cuda")
    return words.view(torch.uint8)[:count]


def _page_slots(g, lengths, page):
    """Slots of requests of `lengths` tokens on random pages of a pool with a
    quarter more pages than they need: (int64 slots, page count)."""
    pages = [-(-n // page) for n in lengths]
    count = sum(pages) + sum(pages) // 4 + 1
    table = torch.randperm(count, generator=g, device="cuda")
    at, got = 0, []
    for n, used in zip(lengths, pages):
        got.append((table[at:at + used, None] * page + torch.arange(page, device="cuda")).reshape(-1)[:n])
        at += used
    return torch.cat(got).contiguous(), count


def _lengths_of(rows):
    """Request lengths that add up to `rows` (about 1,000 tokens each, ragged)."""
    got, left = [], rows
    while left:
        n = min(left, 200 + (len(got) * 617) % 1700)
        got.append(n)
        left -= n
    return got


def _layout(case, page, pages):
    if case.get("packed"):
        model = kv.KvCacheModelLayout.packed_bytes_per_layer(case["layers"], case["dim"])
        return kv.PagedKvCacheLayout.for_model(model, "fp8_e4m3", page, page * pages)
    runtime = kv.KvCacheRuntimeLayout.for_model("bf16" if case.get("elt", 2) == 2 else "fp8_e4m3", page,
                                                case["layers"], case["heads"], case["dim"])
    return kv.PagedKvCacheLayout.new(runtime, pages)


def _row_bytes(case):
    return case["heads"] * case["dim"] * case.get("elt", 2)


def _prepare_write(case, seed):
    g = _generator(seed)
    n, row = case["rows"], _row_bytes(case)
    slots, pages = _page_slots(g, [max(1, 4 * n)], case["page"])
    slots = slots[torch.randperm(slots.numel(), generator=g, device="cuda")[:n]].contiguous()
    layout = _layout(case, case["page"], pages)
    pool = _random_bytes(g, layout.total_byte_len)
    rows = [(_random_bytes(g, n * row), _random_bytes(g, n * row)) for _ in range(case["layers"])]
    plans = [kv.KvPairCopyPlan.new(n, layout.slot_count, layout.kv_pair_copy_geometry(i), row, row)
             for i in range(case["layers"])]
    return dict(pool=pool, keep=(slots, rows), plans=plans, slots=_buffer(slots), pool_buffer=_buffer(pool),
                rows=[(_buffer(k), _buffer(v)) for k, v in rows])


def _run_write(case, s):
    k, stream = _kernels(), torch.cuda.current_stream().cuda_stream
    for plan, (keys, values) in zip(s["plans"], s["rows"]):
        k.scatter(plan, keys=keys, values=values, slot_indices=s["slots"], pool=s["pool_buffer"], stream=stream)
    return s["pool"]


def _prepare_copy(case, seed):
    g = _generator(seed)
    n, layers, row = case["rows"], case["layers"], _row_bytes(case)
    lengths = _lengths_of(n)
    src_slots, src_pages = _page_slots(g, lengths, case["src_page"])
    dst_slots, dst_pages = _page_slots(g, lengths, case["dst_page"])
    src_layout, dst_layout = _layout(case, case["src_page"], src_pages), _layout(case, case["dst_page"], dst_pages)
    src = _random_bytes(g, src_layout.total_byte_len)
    dst = torch.zeros(dst_layout.total_byte_len, dtype=torch.uint8, device="cuda")
    s = dict(n=n, keep=(src, src_slots, dst_slots), dst=dst, src_slots=_buffer(src_slots),
             dst_slots=_buffer(dst_slots), src_stride=src_layout.bytes_per_layer_page,
             dst_stride=dst_layout.bytes_per_layer_page)
    at = dict(heads=case["heads"])
    head_layout = kv.HND if case["hnd"] else kv.NHD
    s["src_views"] = [src_layout.pool_view(src.data_ptr(), src.numel(), i, **at) for i in range(layers)]
    s["dst_views"] = [dst_layout.pool_view(dst.data_ptr(), dst.numel(), i, head_layout, **at) for i in range(layers)]
    if case["op"] == "relay":
        planes = 1 if case["packed"] else 2
        s["plane"] = n * row
        s["rows"] = torch.empty(layers * planes * n * row, dtype=torch.uint8, device="cuda")
        base = s["rows"].data_ptr()
        s["row_views"] = [kv.rows_view([base + (planes * i + t) * n * row for t in range(planes)],
                                       [s["rows"].numel() - (planes * i + t) * n * row for t in range(planes)],
                                       [row] * planes) for i in range(layers)]
        s["row_stride"] = planes * n * row
    return s


def _run_relay(case, s):
    k, stream, n, layers = _kernels(), torch.cuda.current_stream().cuda_stream, s["n"], case["layers"]
    if case["per_layer"]:
        for src, rows, dst in zip(s["src_views"], s["row_views"], s["dst_views"]):
            k.pack_layer(src, s["src_slots"], n, rows, stream=stream)
            k.unpack_layer(rows, n, dst, s["dst_slots"], stream=stream)
    else:
        k.pack_layers(s["src_views"][0], s["src_stride"], layers, s["src_slots"], n, s["row_views"][0],
                      s["row_stride"], stream=stream)
        k.unpack_layers(s["row_views"][0], s["row_stride"], layers, n, s["dst_views"][0], s["dst_stride"],
                        s["dst_slots"], stream=stream)
    return [_words(s["rows"]), _words(s["dst"])]


def _run_transfer(case, s):
    _kernels().transfer_layers(s["src_views"][0], s["src_stride"], case["layers"], s["src_slots"], s["n"],
                               s["dst_views"][0], s["dst_stride"], s["dst_slots"],
                               stream=torch.cuda.current_stream().cuda_stream)
    return _words(s["dst"])


def _words(t):
    """A byte buffer as 8-byte words where it holds whole ones."""
    return t.view(torch.int64) if t.numel() % 8 == 0 else t


def _sequences(case):
    """(tokens of each request, queries of each request, length of each query)."""
    per = case["per_request"]
    if per == 0:  # causal prefill: every token of a prompt is a query
        lengths = _ragged(case["requests"], case["low"], case["high"])
        counts = list(lengths)
    else:
        lengths = _ragged(case["queries"] // per, case["low"], case["high"])
        counts = [per] * len(lengths)
    return lengths, counts, [n - c + 1 + i for n, c in zip(lengths, counts) for i in range(c)]


def _attend_inputs(case, seed):
    """Pool, slots and queries of an attention case, as torch tensors."""
    g = _generator(seed)
    lengths, counts, query_lengths = _sequences(case)
    h, dk, dv, page, layers = case["heads"], case["dk"], case["dv"], case["page"], case["layers"]
    slots, pages = _page_slots(g, lengths, page)
    pool = torch.empty(pages * page * layers * h * (dk + dv), dtype=torch.bfloat16, device="cuda")
    pool.normal_(generator=g)
    queries = torch.empty(layers, len(query_lengths), case["qheads"], dk, dtype=torch.bfloat16, device="cuda")
    queries.normal_(generator=g)
    return lengths, counts, query_lengths, slots, pages, pool, queries


def _prepare_attend(case, seed):
    lengths, counts, query_lengths, slots, pages, pool, queries = _attend_inputs(case, seed)
    h, dk, dv, page, layers, n = (case[x] for x in ("heads", "dk", "dv", "page", "layers", "qheads"))
    key, value = h * dk * 2, h * dv * 2
    runtime = kv.KvCacheRuntimeLayout("bf16", page, layers, h, dk, 2, layers * (key + value),
                                      layers * (key + value) * page)
    layout = (kv.PagedKvCacheLayout.new(runtime, pages) if dk == dv
              else kv.PagedKvCacheLayout.new_with_tensor_pair(runtime, pages, key, value))
    assert layout.total_byte_len == pool.numel() * 2
    requests = torch.repeat_interleave(torch.arange(len(counts), dtype=torch.int32),
                                       torch.tensor(counts)).to("cuda")
    query_lengths = torch.tensor(query_lengths, dtype=torch.int64).to("cuda")
    offsets = torch.tensor([0] + lengths, dtype=torch.int64).cumsum(0).to("cuda")
    output = torch.zeros(layers, queries.shape[1], n, dv, dtype=torch.bfloat16, device="cuda")
    plans = [kv.PagedAttentionPlan.for_layer(layout, i, queries.shape[1], len(counts), slots.numel(), n,
                                             dk ** -0.5, kv.HND if case["hnd"] else kv.NHD) for i in range(layers)]
    common = dict(query_request_indices=_buffer(requests), query_sequence_lengths=_buffer(query_lengths),
                  request_slot_offsets=_buffer(offsets), sequence_slots=_buffer(slots), pool=_buffer(pool))
    calls = [(plan, dict(common, queries=_buffer(queries[i]), output=_buffer(output[i])))
             for i, plan in enumerate(plans)]
    return dict(keep=(pool, queries, slots, requests, query_lengths, offsets), output=output, calls=calls,
                longest=max(lengths))


def _run_attend(case, s):
    k, stream = _kernels(), torch.cuda.current_stream().cuda_stream
    for plan, buffers in s["calls"]:
        k.paged_attention_async(plan, max_sequence_length=s["longest"], stream=stream, **buffers)
    return s["output"]


_PREPARE = {"write": _prepare_write, "relay": _prepare_copy, "transfer": _prepare_copy, "attend": _prepare_attend}
_RUN = {"write": _run_write, "relay": _run_relay, "transfer": _run_transfer, "attend": _run_attend}


def prepare(case, seed):
    state = _PREPARE[case["op"]](case, seed)
    state["case"] = case
    return state


def run(state):
    return _RUN[state["case"]["op"]](state["case"], state)


# ---- what a pass cannot do without ----------------------------------------------------------


def work(case):
    if case["op"] != "attend":
        payload = case["rows"] * case["layers"] * _row_bytes(case) * (1 if case.get("packed") else 2)
        return dict(bytes=payload * (4 if case["op"] == "relay" else 2), flops=0)
    lengths, _, query_lengths = _sequences(case)
    width = case["dk"] + case["dv"]
    moved = 2 * case["heads"] * width * sum(lengths) + 2 * case["qheads"] * width * len(query_lengths)
    return dict(bytes=case["layers"] * moved, flops=case["layers"] * 2 * case["qheads"] * width * sum(query_lengths))


def tolerance(case):
    """Copies move bytes. Attention returns bf16 from fp32 sums: two
    implementations differ by roundings of the last bit of some outputs."""
    return "exact" if case["op"] != "attend" else dict(rel=4e-3, max=4e-2)


def exact(case, seed):
    """Softmax attention in 64 bits, request by request and KV head by KV head."""
    if case["op"] != "attend":
        return None
    lengths, counts, query_lengths, slots, pages, pool, queries = _attend_inputs(case, seed)
    h, dk, dv, page, layers, n = (case[x] for x in ("heads", "dk", "dv", "page", "layers", "qheads"))
    group, per_layer = n // h, page * h * (dk + dv)
    by_page = pool.view(pages, layers, per_layer)
    out = torch.empty(layers, queries.shape[1], n, dv, dtype=torch.float64, device="cuda")
    for layer in range(layers):
        keys, values = by_page[:, layer, :page * h * dk], by_page[:, layer, page * h * dk:]
        if case["hnd"]:
            keys = keys.reshape(pages, h, page, dk).transpose(1, 2)
            values = values.reshape(pages, h, page, dv).transpose(1, 2)
        keys, values = keys.reshape(pages * page, h, dk), values.reshape(pages * page, h, dv)
        first, q0 = 0, 0
        for length, count in zip(lengths, counts):
            own = slots[first:first + length]
            limits = torch.tensor(query_lengths[q0:q0 + count], device="cuda").repeat_interleave(group)
            dead = torch.arange(length, device="cuda")[None, :] >= limits[:, None]
            k64, v64 = keys[own].double(), values[own].double()
            for head in range(h):
                q64 = queries[layer, q0:q0 + count, head * group:(head + 1) * group].double().reshape(-1, dk)
                scores = (q64 @ k64[:, head].t().contiguous()) * dk ** -0.5
                weights = torch.softmax(scores.masked_fill_(dead, -math.inf), dim=1)
                out[layer, q0:q0 + count, head * group:(head + 1) * group] = \
                    (weights @ v64[:, head].contiguous()).reshape(count, group, dv)
            first, q0 = first + length, q0 + count
    return out
