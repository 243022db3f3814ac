"""GPU tests of the paged attention's tile bodies (launches with several
queries per request on average: prefill, chunked prefill, drafted tokens)
against the float64 oracle, under the bound that tests/test_gpu_attention.py
derives: the outputs' own bf16 rounding plus 2^-12 sum_i w_i |v_i| for the
fp32 sums (the tile bodies keep hi + lo weights and fp32 split records).

A tile holds up to 128 (query, query head) rows of one request (64 at dims
256), its tokens come in blocks of 64 (32), the slot table covers 2,048 (dims
64) or 4,096 tokens, and the search looks at 2,048 queries at a time, so the
sizes below sit at those edges. Whether a call takes the tile bodies is the
host's estimate; every test asks which body its call takes.
"""
import ctypes
import math

import numpy as np
import pytest

import oracle
import sgl_rocm_kv as kv
from sgl_rocm_kv import hip
from test_gpu_attention import _bf16_normal, _Case, _check, _say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def k():
    if hip.device_count() == 0:
        pytest.fail("no GPU visible: the gpu tests need an MI355X")
    ctx = kv.RocmKvPairCopyKernels(0)
    yield ctx
    ctx.close()


def _requests(rng, spans, slot_count):
    """Metadata of requests given as (cached tokens, queries): query j of a
    request attends cached + j + 1 tokens."""
    lens = np.array([c + n for c, n in spans])
    rso = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
    slots = rng.choice(slot_count, size=int(rso[-1]), replace=False).astype(np.uint64)
    qri = np.repeat(np.arange(len(spans)), [n for _, n in spans])
    qsl = np.concatenate([c + 1 + np.arange(n) for c, n in spans])
    return qri, qsl, rso, slots


class _Call:
    """Device buffers of one call, for launches into outputs of their own."""

    def __init__(self, c, q, qri, qsl, rso, slots, max_len):
        self.plan = kv.PagedAttentionPlan.for_layer(c.layout, c.layer, len(qri), len(rso) - 1, len(slots), c.qh,
                                                    1.0 / math.sqrt(c.dk), kv.HND if c.hnd else kv.NHD)
        arrays = dict(queries=q, query_request_indices=np.asarray(qri, np.uint32),
                      query_sequence_lengths=np.asarray(qsl, np.uint64),
                      request_slot_offsets=np.asarray(rso, np.uint64), sequence_slots=np.asarray(slots, np.uint64))
        self.bufs = {n: hip.DeviceBuffer.from_array(a) for n, a in arrays.items()}
        self.bufs["pool"], self.max_len = c.pool, max_len

    def output(self):
        out = hip.DeviceBuffer(self.plan.output_required_bytes)
        out.fill(0xFF)
        return out

    def run(self, k, out, stream=None):
        k.paged_attention_async(self.plan, max_sequence_length=self.max_len, stream=stream, output=out, **self.bufs)

    def route(self, k):
        out = self.output()
        return k.attention_route(self.plan, max_sequence_length=self.max_len, output=out, **self.bufs)


@pytest.mark.parametrize("body,H,qh,d,P,hnd,spans", [
    # too few or too short for tiles: the per-query bodies, several queries per request
    ("staged128", 2, 8, 128, 16, False, [(0, 1), (0, 2), (0, 31), (0, 32), (0, 33), (0, 63), (0, 64), (0, 65)]),
    ("staged128k", 2, 8, 128, 64, True, [(0, 300), (127, 3), (64, 64), (63, 66)]),
    ("staged64", 2, 14, 64, 1, True, [(0, 40), (0, 18), (0, 19), (1, 1)]),
    ("staged64", 4, 4, 64, 64, False, [(0, 200), (0, 128), (77, 127)]),
    ("staged256", 2, 8, 256, 64, False, [(0, 70), (500, 5), (31, 33)]),
    ("staged256", 1, 16, 256, 16, True, [(100, 40), (0, 9)]),
    ("wide128", 1, 64, 128, 64, False, [(4090, 9), (0, 3)]),
    ("wide128", 1, 48, 128, 1, False, [(0, 21), (64, 2)]),
    # tiles
    ("tile128", 8, 32, 128, 16, False, [(0, 1), (0, 2), (0, 31), (0, 32), (0, 33), (0, 63), (0, 64), (0, 65)]),
    ("tile128", 8, 32, 128, 64, True, [(0, 300), (127, 3), (64, 64), (63, 66)]),
    ("tile128", 8, 32, 128, 64, False, [(700, 5), (40, 5), (1999, 5), (3, 5)]),    # drafted tokens, split
    ("tile64", 2, 14, 64, 16, False, [(0, 129), (2000, 150), (5, 2)]),              # groups of 7, split
    ("tile64", 8, 56, 64, 1, True, [(0, 140), (0, 118), (0, 119), (1, 1)]),
    ("tile64", 16, 16, 64, 64, False, [(0, 200), (0, 128), (77, 127)]),             # one head a group: 128 queries a tile
    ("tile128", 1, 64, 128, 64, False, [(90, 200)]),                                # groups of 64: two queries a tile
    ("tile128", 1, 48, 128, 1, False, [(90, 200)]),                                 # two queries a tile, 32 idle rows
    ("tile256", 4, 16, 256, 64, False, [(0, 70), (500, 5), (31, 33)]),
    ("tile256", 2, 32, 256, 16, True, [(1000, 70), (0, 39)]),                       # groups of 16, split
    ("tile256", 1, 32, 256, 64, False, [(300, 60), (0, 39)]),                       # groups of 32: two queries a tile
    ("tile64", 2, 14, 64, 16, False, [(0, 1500), (0, 900), (0, 2)]),                # a run cut at the search's step
    ("tile128", 2, 8, 128, 16, True, [(0, 700)] * 2 + [(300, 2)] * 400),            # both ways of the search, two steps
    ("tile64", 48, 96, 64, 16, False, [(0, 511)]),                                  # 384 whole tiles: folded over 256 CUs
])
def test_causal_queries(k, body, H, qh, d, P, hnd, spans):
    rng = np.random.default_rng(d + qh + len(spans))
    pages = -(-sum(c + n for c, n in spans) // P) + 3
    c = _Case(rng, P=P, L=2, H=H, dk=d, dv=d, qh=qh, pages=pages, layer=1, hnd=hnd)
    qri, qsl, rso, slots = _requests(rng, spans, c.layout.slot_count)
    q = _bf16_normal(rng, len(qri) * qh * d).reshape(len(qri), qh, d)
    _say(f"{body} H={H} qh={qh} d={d} P={P} hnd={hnd} queries={len(qri)}")
    assert c.route(k, q, qri, qsl, rso, slots, int(qsl.max())).body == body
    got, want = c.run(k, q, qri, qsl, rso, slots, 1.0 / math.sqrt(d), max_len=int(qsl.max()))
    _check(got, want, c)


@pytest.mark.parametrize("d,length", [(64, 2152), (128, 4202), (256, 4152)])
def test_splits_longer_than_the_slot_table(k, d, length):
    """60 requests of two queries each over the same slots: enough tiles that
    none is split, so each fills its slot table again on the way."""
    rng = np.random.default_rng(d + 7)
    c = _Case(rng, P=16, L=1, H=8, dk=d, dv=d, qh=8, pages=length // 16 + 2, layer=0)
    own = rng.choice(c.layout.slot_count, size=length, replace=False).astype(np.uint64)
    qri, qsl = np.repeat(np.arange(60), 2), np.tile([length - 1, length], 60)
    qsl[8:24] -= 3 * np.arange(16)
    rso, slots = np.arange(61, dtype=np.uint64) * np.uint64(length), np.tile(own, 60)
    q = _bf16_normal(rng, 120 * 8 * d).reshape(120, 8, d)
    route = c.route(k, q, qri, qsl, rso, slots, length)
    assert route.body == f"tile{d}" and route.splits == 1 and route.chunk_tokens > (2048 if d == 64 else 4096)
    _say(f"tiles past the slot table, d={d}, {length} tokens")
    got, want = c.run(k, q, qri, qsl, rso, slots, 1.0 / math.sqrt(d), max_len=length)
    _check(got, want, c)


@pytest.mark.parametrize("d", [64, 128, 256])
def test_queries_in_any_order(k, d):
    """Runs of one request cut by others, decreasing and repeated lengths,
    and far more tiles than queries that come request by request make."""
    rng = np.random.default_rng(d)
    H = 4 if d == 256 else 8
    c = _Case(rng, P=16, L=1, H=H, dk=d, dv=d, qh=4 * H, pages=120, layer=0)
    lens = np.array([900, 333, 64])
    rso = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
    slots = rng.choice(c.layout.slot_count, size=int(rso[-1]), replace=False).astype(np.uint64)
    qri = np.concatenate([np.arange(90) % 3, np.zeros(70, int), rng.integers(0, 3, 64), np.full(3, 2)])
    qsl = np.array([rng.integers(1, lens[r] + 1) for r in qri])
    qsl[90:160] = np.sort(qsl[90:160])[::-1]
    q = _bf16_normal(rng, len(qri) * 4 * H * d).reshape(len(qri), 4 * H, d)
    _say(f"tiles in any order, d={d}, {len(qri)} queries")
    assert c.route(k, q, qri, qsl, rso, slots, 900).body == f"tile{d}"
    got, want = c.run(k, q, qri, qsl, rso, slots, 1.0 / math.sqrt(d), max_len=900)
    _check(got, want, c)


@pytest.mark.parametrize("H,qh,d,spans,shuffle", [
    (8, 32, 64, [(0, 200)] * 4, False),          # four prompts in turn: gathered tiles of 32
    (8, 32, 128, [(0, 64)] * 8, False),
    (1, 8, 128, [(30, 300), (0, 700), (5, 1300), (0, 3)], True),   # over the search's step of 2,048 queries
    (2, 8, 256, [(1500, 5)] * 24, False),         # drafts, position by position
    (1, 4, 64, [(600, 40 + i % 7) for i in range(60)], True),
    (4, 4, 64, [(0, 2500), (0, 90), (0, 20)], False),  # 128 a tile; a step of one request alone
])
def test_interleaved_queries(k, H, qh, d, spans, shuffle):
    """Queries of several requests in turn (query j of every request before
    query j + 1 of any), or in a random order: every step of the search then
    has more runs than there are requests, and its tiles gather a request's
    queries."""
    rng = np.random.default_rng(d + qh + len(spans))
    c = _Case(rng, P=16, L=1, H=H, dk=d, dv=d, qh=qh, pages=sum(c + n for c, n in spans) // 16 + 3, layer=0)
    qri, qsl, rso, slots = _requests(rng, spans, c.layout.slot_count)
    turn = np.concatenate([np.arange(n) for _, n in spans])
    order = rng.permutation(len(qri)) if shuffle else np.argsort(turn, kind="stable")
    qri, qsl = qri[order], qsl[order]
    q = _bf16_normal(rng, len(qri) * qh * d).reshape(len(qri), qh, d)
    call = _Call(c, q, qri, qsl, rso, slots, int(qsl.max()))
    assert call.route(k).body == f"tile{d}"
    _say(f"tiles of gathered queries H={H} qh={qh} d={d} queries={len(qri)} shuffle={shuffle}")
    got, want = c.run(k, q, qri, qsl, rso, slots, 1.0 / math.sqrt(d), max_len=int(qsl.max()))
    _check(got, want, c)


def test_gathered_tiles_report_bad_requests(k):
    """A bad request index among interleaved queries raises the reference's
    request bit and leaves every other query's result as it is."""
    rng = np.random.default_rng(8)
    c = _Case(rng, P=16, L=1, H=8, dk=64, dv=64, qh=32, pages=60, layer=0)
    qri, qsl, rso, slots = _requests(rng, [(0, 200)] * 4, c.layout.slot_count)
    order = np.argsort(np.tile(np.arange(200), 4), kind="stable")
    qri, qsl = qri[order], qsl[order]
    q = _bf16_normal(rng, 800 * 32 * 64).reshape(800, 32, 64)
    outs = []
    for bad in (False, True):
        index = qri.copy()
        if bad:
            index[[5, 300]] = [4, 1 << 30]
        call = _Call(c, q, index, qsl, rso, slots, 200)
        assert call.route(k).body == "tile64"
        outs.append(call.output())
        _say(f"tiles of gathered queries, two bad indices: {bad}")
        call.run(k, outs[-1])
        if bad:
            with pytest.raises(kv.KvError) as e:
                k.check_errors()
            assert e.value.variant == "DeviceMetadataInvalid" and e.value.fields[0] == 1
        else:
            k.check_errors()
    good, got = (o.download(dtype=np.uint16).reshape(800, 32, 64) for o in outs)
    keep = np.delete(np.arange(800), [5, 300])
    # (A tile that loses a query passes the maxima of the others alone, so
    # last bits may differ: two results within the bound of _check of one value.)
    a, b = (oracle.bf16_to_f32(x[keep]).astype(np.float64) for x in (good, got))
    assert (np.abs(a - b) <= 2 * (2.0 ** -8 * np.abs(a) + 5.5 * 2.0 ** -12)).all()
    assert (got[[5, 300]] == 0xFFFF).all()


@pytest.mark.parametrize("bits", [0x7F80, 0xFF80, 0x7FC0])  # inf, -inf, NaN
@pytest.mark.parametrize("d", [64, 128, 256])
def test_values_past_a_query_are_not_seen(k, d, bits):
    """Tokens 50 and 180 of a causal prompt hold infinite or NaN keys and
    values: queries that do not attend them are as without them."""
    rng = np.random.default_rng(d + bits)
    H = 4 if d == 256 else 8
    c = _Case(rng, P=16, L=1, H=H, dk=d, dv=d, qh=4 * H, pages=20, layer=0)
    qri, qsl, rso, slots = _requests(rng, [(0, 200)], c.layout.slot_count)
    pool16 = c.pool_h.view(np.uint16)
    for token in (50, 180):
        for tensor in (0, 1):
            page, pos = divmod(int(slots[token]), 16)
            at, end = c.layout.tensor_token_byte_range(page, 0, tensor, pos)
            pool16[at // 2 + (token % 7):end // 2:5] = bits
    c.pool.upload(c.pool_h)
    q = _bf16_normal(rng, 200 * 4 * H * d).reshape(200, 4 * H, d)
    _say(f"tiles with values of 0x{bits:x} past some queries, d={d}")
    assert c.route(k, q, qri, qsl, rso, slots, 200).body == f"tile{d}"
    with np.errstate(all="ignore"):
        got, want = c.run(k, q, qri, qsl, rso, slots, 1.0 / math.sqrt(d), max_len=200)
    c.absw = c.absw[:50]
    assert np.isfinite(got[:50]).all()
    _check(got[:50], want[:50], c)


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("what,flag", [("index", 1), ("empty", 2), ("long", 2), ("slot", 4)])
def test_bad_metadata_is_reported(k, d, what, flag):
    """A request index past the requests, lengths of 0 or past the request's
    slots, and a slot past the pool raise the reference's flag bits from
    inside a tile; the other queries' outputs are written (all but those
    that attend the bad slot)."""
    rng = np.random.default_rng(9)
    H = 4 if d == 256 else 8
    c = _Case(rng, P=16, L=1, H=H, dk=d, dv=d, qh=4 * H, pages=50, layer=0)
    slots = rng.choice(c.layout.slot_count, size=600, replace=False).astype(np.uint64)
    index, lengths = np.repeat([0, 1], 130), np.full(260, 160)
    keep = np.ones(260, bool)
    if what == "index":
        index[50] = 7
    elif what == "slot":
        slots[70] = c.layout.slot_count
        keep[:130] = False
    else:
        lengths[50] = 0 if what == "empty" else 301
    if what != "slot":
        keep[50] = False
    q = _bf16_normal(rng, 260 * 4 * H * d).reshape(260, 4 * H, d)
    call = _Call(c, q, index, lengths, [0, 300, 600], slots, 600)
    assert call.route(k).body == f"tile{d}"
    out = call.output()
    _say(f"tiles with a bad {what}, d={d}")
    call.run(k, out)
    with pytest.raises(kv.KvError) as e:
        k.check_errors()
    assert e.value.variant == "DeviceMetadataInvalid" and e.value.fields[0] == flag
    written = (out.download(dtype=np.uint16).reshape(260, -1) != 0xFFFF).all(axis=1)
    assert written[keep].all() and (what == "slot" or not written[50])


def _chunk_call(seed, H, qh, d, cached, queries):
    rng = np.random.default_rng(seed)
    c = _Case(rng, P=16, L=1, H=H, dk=d, dv=d, qh=qh, pages=(cached + queries) // 16 + 3, layer=0)
    qri, qsl, rso, slots = _requests(rng, [(cached, queries)], c.layout.slot_count)
    q = _bf16_normal(rng, queries * qh * d).reshape(queries, qh, d)
    return _Call(c, q, qri, qsl, rso, slots, cached + queries)


def test_calls_on_several_streams_keep_their_records_apart(k):
    """Chunks of prompts that are split only because their tiles are few, on
    two streams, beside a decode call on a third whose records are in the
    context's shared buffer: each result equals that of the call alone."""
    first, second = _chunk_call(1, 8, 32, 128, 600, 384), _chunk_call(2, 8, 32, 64, 700, 300)
    for call, body in ((first, "tile128"), (second, "tile64")):
        route = call.route(k)
        assert route.body == body and route.splits > 1 and route.records_apart
    rng = np.random.default_rng(3)
    c = _Case(rng, P=16, L=1, H=8, dk=128, dv=128, qh=32, pages=600, layer=0)
    decode = _Call(c, _bf16_normal(rng, 2 * 32 * 128).reshape(2, 32, 128), [0, 1], [4000, 3000], [0, 4000, 7000],
                   rng.choice(c.layout.slot_count, size=7000, replace=False), 4000)
    route = decode.route(k)
    assert route.body == "staged128" and route.splits > 1 and not route.records_apart
    calls = (first, second, decode)
    want = []
    for call in calls:
        out = call.output()
        call.run(k, out)
        hip.synchronize()
        want.append(out.download(dtype=np.uint16))
        assert not np.all(want[-1] == 0xFFFF)
    streams = [hip.Stream() for _ in calls]
    outs = [[call.output() for call in calls] for _ in range(20)]
    hip.synchronize()
    _say("tiles: 60 calls on three streams")
    for row in outs:
        for call, out, stream in zip(calls, row, streams):
            call.run(k, out, stream)
    for stream in streams:
        stream.synchronize()
    k.check_errors()
    for i, row in enumerate(outs):
        for out, w in zip(row, want):
            np.testing.assert_array_equal(out.download(dtype=np.uint16), w, err_msg=f"round {i}")
    for stream in streams:
        stream.destroy()


def test_captured_call_is_not_split(k):
    """The same chunk under graph capture, in a context that has split
    nothing yet: it is captured (nothing is allocated, no event waited for),
    and every replay matches the eager result up to the splits' rounding."""
    call = _chunk_call(4, 8, 32, 128, 600, 384)
    ctx = kv.RocmKvPairCopyKernels(0)
    assert call.route(ctx).records_apart
    out, stream = call.output(), hip.Stream()
    h, vp = hip.lib(), ctypes.c_void_p
    h.hipStreamBeginCapture.argtypes = [vp, ctypes.c_int]
    h.hipStreamEndCapture.argtypes = [vp, ctypes.POINTER(vp)]
    h.hipGraphInstantiate.argtypes = [ctypes.POINTER(vp), vp, vp, vp, ctypes.c_size_t]
    h.hipGraphLaunch.argtypes = [vp, vp]
    h.hipGraphExecDestroy.argtypes = [vp]
    h.hipGraphDestroy.argtypes = [vp]
    hip.synchronize()
    graph, execution = vp(), vp()
    _say("tiles: a chunk under graph capture")
    hip.check(h.hipStreamBeginCapture(stream.handle, 0), "hipStreamBeginCapture")
    call.run(ctx, out, stream)
    hip.check(h.hipStreamEndCapture(stream.handle, ctypes.byref(graph)), "hipStreamEndCapture")
    hip.check(h.hipGraphInstantiate(ctypes.byref(execution), graph, None, None, 0), "hipGraphInstantiate")
    eager = call.output()
    call.run(ctx, eager)
    hip.synchronize()
    want = eager.download(dtype=np.uint16)
    replays = []
    for i in range(3):
        out.fill(0xFF)
        hip.synchronize()
        hip.check(h.hipGraphLaunch(execution, stream.handle), "hipGraphLaunch")
        stream.synchronize()
        replays.append(out.download(dtype=np.uint16))
        call.run(ctx, eager)  # eager work between the replays
        hip.synchronize()
        np.testing.assert_array_equal(eager.download(dtype=np.uint16), want)
    ctx.check_errors()
    a, b = (oracle.bf16_to_f32(x).astype(np.float64) for x in (replays[0], want))
    # Both are within the bound of _check of one exact value: a bf16 rounding
    # each and 2^-12 of sum w|v| (|v| <= 5.5 here) each.
    assert (np.abs(a - b) <= 2 * (2.0 ** -8 * np.abs(a) + 5.5 * 2.0 ** -12)).all()
    for r in replays[1:]:
        np.testing.assert_array_equal(r, replays[0])
    hip.check(h.hipGraphExecDestroy(execution), "hipGraphExecDestroy")
    hip.check(h.hipGraphDestroy(graph), "hipGraphDestroy")
    stream.destroy()
    ctx.close()


def test_no_allocation_entry_point_splits_alike(k):
    """Tiles through the no-allocation entry point: the same splits, bit for
    bit the same result, for a chunk whose queries alone would not be split
    and for one whose queries would."""
    for call in (_chunk_call(5, 8, 32, 128, 600, 384), _chunk_call(6, 2, 14, 64, 3000, 100),
                 _chunk_call(7, 2, 8, 256, 2000, 60)):
        route = call.route(k)
        assert route.body.startswith("tile") and route.splits > 1
        outs = [call.output() for _ in range(2)]
        _say(f"tiles through the no-allocation entry point: {route}")
        call.run(k, outs[0])
        k.paged_attention_async_noalloc(call.plan, max_sequence_length=call.max_len, output=outs[1], **call.bufs)
        k.check_errors()
        a, b = (o.download(dtype=np.uint16) for o in outs)
        assert not np.all(a == 0xFFFF)
        np.testing.assert_array_equal(a, b)
