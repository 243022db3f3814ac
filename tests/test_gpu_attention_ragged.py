"""GPU tests of paged attention over ragged decode batches (the average
request below two thirds of the longest, enough work to number the splits
that have tokens first) against the float64 oracle, under the bound that
tests/test_gpu_attention.py derives. The query counts sit at the edges of the
64-query steps of the search and of the most queries it takes (256). Whether
a batch is numbered is the host's rule; every test asks."""
import math

import numpy as np
import pytest

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


def _ragged(rng, queries, longest, mean):
    """Lengths of 1 to `longest`, one of each, about `mean` on average."""
    lens = np.minimum(1 + rng.exponential(mean, queries).astype(np.int64), longest)
    lens[rng.integers(queries)] = longest
    lens[0] = 1 if queries > 1 else longest
    return lens


@pytest.mark.parametrize("body,live,queries,H,qh,dk,dv,hnd,longest,mean", [
    ("staged128", True, 256, 1, 4, 128, 128, False, 2600, 700),
    ("staged128", False, 257, 1, 4, 128, 128, False, 2600, 700),  # past the most that is numbered
    ("staged128", False, 256, 1, 4, 128, 128, False, 1500, 450),  # too little work
    ("staged128k", True, 65, 8, 8, 128, 128, True, 2500, 900),    # head-major, K in registers
    ("staged128k", False, 65, 2, 8, 128, 128, True, 2500, 900),
    ("staged128", True, 64, 4, 28, 128, 128, False, 3000, 1000),
    ("staged64", True, 129, 4, 16, 64, 64, False, 2000, 500),
    ("staged64", True, 256, 2, 4, 64, 64, False, 2000, 500),
    ("staged128", True, 3, 8, 32, 128, 128, False, 20000, 9000),
    ("staged256", True, 63, 4, 4, 256, 256, True, 1500, 600),
    ("staged256", False, 63, 2, 8, 256, 256, True, 1500, 500),
    ("latent_exact", True, 21, 1, 128, 576, 512, False, 5000, 1500),
    ("latent_exact", False, 1, 1, 128, 576, 512, False, 700, 700),
    ("latent_exact", True, 9, 1, 100, 576, 512, False, 400, 90),     # short MLA batch: 64-token splits
    ("staged128", True, 70, 8, 32, 128, 128, False, 40000, 300),  # one sequence of far more splits than the others
    ("staged64", True, 64, 4, 8, 64, 64, True, 60000, 400),
])
def test_ragged_decode(k, body, live, queries, H, qh, dk, dv, hnd, longest, mean):
    rng = np.random.default_rng(queries + dk)
    lens = _ragged(rng, queries, longest, mean)
    rso = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
    P = 16
    c = _Case(rng, P=P, L=1, H=H, dk=dk, dv=dv, qh=qh, pages=-(-int(rso[-1]) // P) + 3, layer=0, hnd=hnd)
    slots = rng.choice(c.layout.slot_count, size=int(rso[-1]), replace=False).astype(np.uint64)
    q = _bf16_normal(rng, queries * qh * dk).reshape(queries, qh, dk)
    _say(f"ragged decode: {queries} queries, {int(rso[-1])} tokens, longest {longest}, dims {dk}/{dv} hnd={hnd}")
    route = c.route(k, q, np.arange(queries), lens, rso, slots, longest)
    assert route.body == body and route.live_splits_first == live
    got, want = c.run(k, q, np.arange(queries), lens, rso, slots, 1.0 / math.sqrt(dk), max_len=longest)
    _check(got, want, c)


@pytest.mark.parametrize("length", [0, 1 << 40])
def test_refused_length_is_reported_once_and_alone(k, length):
    """A length that the metadata checks refuse takes no other query's place:
    it raises the reference's sequence bit, and the rest is computed."""
    rng = np.random.default_rng(3)
    lens = _ragged(rng, 64, 3000, 1000)
    rso = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
    c = _Case(rng, P=16, L=1, H=4, dk=128, dv=128, qh=8, pages=-(-int(rso[-1]) // 16) + 3, layer=0)
    slots = rng.choice(c.layout.slot_count, size=int(rso[-1]), replace=False).astype(np.uint64)
    q = _bf16_normal(rng, 64 * 8 * 128).reshape(64, 8, 128)
    asked = lens.astype(np.uint64)
    asked[10] = length
    plan = kv.PagedAttentionPlan.for_layer(c.layout, 0, 64, 64, len(slots), 8, 0.1)
    out = hip.DeviceBuffer.from_array(np.full(plan.output_required_bytes // 2, 0x7FC0, np.uint16))
    bufs = dict(queries=q, query_request_indices=np.arange(64, dtype=np.uint32), query_sequence_lengths=asked,
                request_slot_offsets=rso, sequence_slots=slots)
    bufs = {n: hip.DeviceBuffer.from_array(a) for n, a in bufs.items()}
    assert k.attention_route(plan, max_sequence_length=3000, pool=c.pool, output=out, **bufs).live_splits_first
    with pytest.raises(kv.KvError) as e:
        k.paged_attention(plan, max_sequence_length=3000, pool=c.pool, output=out, **bufs)
    assert e.value.variant == "DeviceMetadataInvalid" and e.value.fields[0] == 2
    got = out.download().view(np.uint16).reshape(64, -1)
    written = (got != 0x7FC0).all(axis=1)
    assert not written[10] and written[np.arange(64) != 10].all()
