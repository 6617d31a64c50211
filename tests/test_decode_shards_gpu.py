"""Decode of pools with token rows below 2 KiB (tensor-parallel shards of the Qwen3 shapes, 8 x 64).

They run on the whole-row kernel with 2 or 4 token rows per wave.  Vs the oracle, and planned,
planning and fused-append calls against the unplanned ones bit for bit, at lengths around the
wave's rows (2, 4), the workgroup's (16, 32), the page, the burst and the range sizes.
"""
import numpy as np
import pytest
import torch

import oracle
from gpu_util import assert_attn_close, say, to_dev
from infurnace_amd import _capi
from infurnace_amd.kernels import (PagedAttentionError, decode_plan, paged_attention, qk_norm_rope_store_and_decode,
                                   rope_table, store_kv_and_decode)
from infurnace_amd.kernels.paged_attention import workspace_for
from test_decode_planning_gpu import _case, _check

pytestmark = pytest.mark.gpu

SHAPES = [(8, 4, 128), (16, 4, 128), (4, 2, 128), (8, 2, 128), (16, 8, 64)]
EDGES = [1, 2, 3, 4, 5, 15, 16, 17, 18, 31, 32, 33, 47, 63, 64, 65, 127, 128, 129, 255, 257, 1000, 1023, 4096]


@pytest.mark.parametrize("hq,hkv,d", SHAPES)
def test_shard_decode_edges(dev, hq, hkv, d):
    say(f"shard decode hq={hq} hkv={hkv} d={d}")
    rng = np.random.default_rng(hq * 11 + hkv + d)
    pool, table, lens, q = _case(rng, EDGES, hq, hkv, d)
    got = paged_attention(*(to_dev(x, dev) for x in (q, pool, table, lens)))
    assert_attn_close(got, oracle.paged_attention(q, pool, table, lens), f"hq={hq} hkv={hkv} d={d}")
    for append in (False, True):
        _check(dev, pool, table, lens, q, append=append, what=f"hq={hq} hkv={hkv} d={d} append={append}")


@pytest.mark.parametrize("hq,hkv,d", SHAPES)
@pytest.mark.parametrize("length", [1, 3, 31, 33, 130, 512, 6000])
def test_shard_decode_one_row(dev, hq, hkv, d, length):
    """One row (its keys split over up to 256 ranges, fp32 split states), with the fused append."""
    say(f"shard one row hq={hq} hkv={hkv} d={d} length={length}")
    rng = np.random.default_rng(length + hq + hkv)
    pool, table, lens, q = _case(rng, [length], hq, hkv, d)
    k, v = (rng.standard_normal((1, hkv, d), dtype=np.float32).astype(np.float16) for _ in range(2))
    slots = np.asarray([table[0, (length - 1) // 16] * 16 + (length - 1) % 16], np.int32)
    p = to_dev(pool, dev)
    got = store_kv_and_decode(to_dev(q, dev), p, to_dev(table, dev), to_dev(lens, dev), None, to_dev(slots, dev),
                              to_dev(k, dev), to_dev(v, dev))
    oracle.store_kv(pool, slots, None, k, v)
    assert np.array_equal(p.cpu().numpy().view(np.uint16), pool.view(np.uint16))
    assert_attn_close(got, oracle.paged_attention(q, pool, table, lens), f"length {length}")


@pytest.mark.parametrize("hq,hkv,d", [(16, 4, 128), (8, 2, 128)])
def test_shard_decode_inactive_empty_bad_pages(dev, hq, hkv, d):
    """Inactive rows write nothing, empty ones zeros, pages outside the pool contribute no key --
    also where one wave load spans a bad page and a good one -- and shared pages (cached loads) agree."""
    say(f"shard bad pages hq={hq} hkv={hkv}")
    rng = np.random.default_rng(hq)
    pool, table, lens, q = _case(rng, [50, 700, 33, 90, 0, 301, 2000], hq, hkv, d)
    used = {int(x) for b in range(len(lens)) for x in table[b, :-(-int(lens[b]) // 16)]}
    pool[:, [p for p in range(pool.shape[1]) if p not in used]] = np.float16(np.nan)  # (pages no row holds)
    active = np.asarray([1, 0, 1, 1, 1, 1, 1], np.uint8)
    table[5, 1], table[5, 3], table[6, 0] = pool.shape[1] + 1000, -7, 1 << 30
    a = [to_dev(x, dev) for x in (q, pool, table, lens)]
    out = torch.full(q.shape, 7.0, dtype=torch.float16, device=dev)
    paged_attention(*a, to_dev(active, dev), out=out)
    cached = paged_attention(*a, shared_prefix_pages=torch.zeros(0, dtype=torch.int32, device=dev))
    good = np.flatnonzero((active != 0) & (lens > 0))
    assert torch.all(out[1] == 7.0) and torch.all(out[4] == 0.0)
    t2, l2 = table[good].copy(), lens[good].copy()
    for i, b in enumerate(good):  # the rows' keys without the bad pages
        n = -(-int(lens[b]) // 16)
        ok = [int(x) for x in table[b, :n] if 0 <= x < pool.shape[1]]
        l2[i] -= 16 * (n - len(ok))
        t2[i, :len(ok)] = ok
    ref = oracle.paged_attention(q[good], pool, t2, l2)
    idx = torch.as_tensor(good, device=dev)
    assert_attn_close(out[idx], ref, "bad pages")
    assert_attn_close(cached[idx], ref, "cached loads")
    _check(dev, pool, table, lens, q, active=active, what="bad pages")


def test_shard_many_short_rows(dev):
    """700 rows of a few keys: ranges with more pieces than a plan record holds."""
    say("shard many short rows")
    rng = np.random.default_rng(700)
    pool, table, lens, q = _case(rng, rng.integers(1, 40, size=700), 16, 4, 128)
    got = paged_attention(*(to_dev(x, dev) for x in (q, pool, table, lens)))
    assert_attn_close(got, oracle.paged_attention(q, pool, table, lens), "short rows")
    _check(dev, pool, table, lens, q, what="short rows")
    _check(dev, pool, table, lens, q, append=True, what="short rows append")


def test_shard_calls_without_a_plan_buffer(dev):
    """Callers from when these shapes had no plan: a missing or short plan buffer means no plan."""
    say("shard without a plan buffer")
    rng = np.random.default_rng(4)
    pool, table, lens, q = _case(rng, [300, 40], 16, 4, 128)
    qd, p, bt, sl = (to_dev(x, dev) for x in (q, pool, table, lens))
    ref = paged_attention(qd, p, bt, sl)
    L = _capi.lib()
    st = torch.cuda.current_stream(dev).cuda_stream
    ws = workspace_for(dev, st, L.ifn_paged_decode_workspace_bytes(2, 16, 4, 128, 16, 400))
    buf = torch.zeros(64, dtype=torch.uint8, device=dev)
    args = (bt.data_ptr(), table.shape[1], sl.data_ptr(), None)
    for plan, nbytes in ((None, 0), (buf.data_ptr(), 64), (buf.data_ptr() + 4, 60)):
        assert L.ifn_paged_decode_plan(plan, nbytes, *args, None, p.shape[1], 2, 16, 4, 128, 16, 400, st) == 0
        for fn in (L.ifn_paged_decode_planned, L.ifn_paged_decode_planning):
            out = torch.empty_like(qd)
            assert fn(out.data_ptr(), qd.data_ptr(), p.data_ptr(), p.shape[1], *args, 2, 16, 4, 128, 16, 400, 0.0, plan,
                      nbytes, ws.data_ptr(), ws.numel(), st) == 0
            assert torch.equal(out.view(torch.int16), ref.view(torch.int16))
    assert int(buf.sum()) == 0


@pytest.mark.parametrize("hq,hkv,d", [(16, 4, 128), (8, 2, 128), (16, 8, 128)])
@pytest.mark.parametrize("first", ["prep", "plain"])
def test_lazy_plan_with_slots_across_call_forms(dev, hq, hkv, d, first):
    """A lazy plan with slots whose first call takes none (the pre-append step of these rows attends after a
    separate append): it stays valid for every later call, and is stale only once its tensors change."""
    say(f"lazy plan across forms hq={hq} hkv={hkv} first={first}")
    rng = np.random.default_rng(hq + hkv)
    pool, table, lens, q = _case(rng, [300, 1, 33, 700], hq, hkv, d)
    qd, p, bt, sl = (to_dev(x, dev) for x in (q, pool, table, lens))
    pos = lens - 1
    sm = to_dev((table[np.arange(4), pos // 16] * 16 + pos % 16).astype(np.int32), dev)
    f = lambda *s: torch.randn(s, device=dev)
    qf, kf, vf, w = f(4, hq, d), f(4, hkv, d), f(4, hkv, d), f(d)
    rope, pd = rope_table(700, d, 1e6, device=dev), to_dev(pos.astype(np.int32), dev)
    plan = decode_plan(qd.shape, p, bt, sl, None, sm, lazy=True)
    assert plan.pending
    prep = lambda pl: qk_norm_rope_store_and_decode(qf, kf, vf, w, w, rope, pd, sm, None, p, bt, sl, plan=pl)
    plain = lambda pl, **o: paged_attention(qd, p, bt, sl, plan=pl, **o)
    append = lambda pl, **o: store_kv_and_decode(qd, p, bt, sl, None, sm, kf.half(), vf.half(), plan=pl, **o)
    same = lambda a, b: torch.equal(a.view(torch.int16), b.view(torch.int16))
    (prep if first == "prep" else plain)(plan)
    assert not plan.pending
    assert same(prep(plan), prep(None))
    for o in ({}, dict(validate=True)):
        assert same(plain(plan, **o), plain(None))
        assert same(append(plan, **o), append(None))
    sl[0] -= 17
    for call in (plain, append):
        with pytest.raises(PagedAttentionError, match="stale"):
            call(plan, validate=True)
