"""Chunks large enough for the 128-row prefill kernel (paged_prefill_block.hip), vs the oracle.

Every row is checked: row r of a chunk at ``start`` is the single query of a sequence of
start + r + 1 keys.  Tolerance atol 2e-3 / rtol 1e-2 in fp16, as for the other prefill kernel.
"""
import numpy as np
import pytest
import torch

import oracle
from gpu_util import assert_attn_close, say, to_dev
from infurnace_amd.kernels import (paged_attention, qk_norm_rope_append, qk_norm_rope_append_and_prefill, rope_table,
                                   store_kv, store_kv_and_prefill)

pytestmark = pytest.mark.gpu


def _case(hq, hkv, start, T, bad=()):
    d = 128
    rng = np.random.default_rng(start * 3 + T + hq)
    pages = -(-(start + T) // 16)
    P = pages + 5
    table = rng.permutation(P)[:pages].astype(np.int32)
    for i, v in bad:
        table[i] = v
    f = lambda *s: rng.standard_normal(s, dtype=np.float32).astype(np.float16)
    return f(2, P, 16, hkv, d), table, f(T, hq, d), f(T, hkv, d), f(T, hkv, d)


# One group (two workgroups per CU) from 512 workgroups of 128 rows, or from 257 when the chunk is no
# longer than what precedes it; two groups below.  Starts off the page (the store is its own launch), on
# the page but off the tile, chunk ends inside a page and a tile, every group size.
@pytest.mark.parametrize("hq,hkv,start,T", [
    (64, 8, 0, 1024), (64, 8, 37, 1030), (32, 8, 16, 2049), (8, 8, 0, 8192),  # one group
    (64, 8, 600, 517), (32, 8, 1072, 1050),                                   # one group, 257 .. 511
    (64, 8, 0, 530), (32, 8, 720, 1100), (16, 8, 5, 2065), (16, 4, 48, 2070), # two groups, 257 .. 511
    (64, 8, 288, 272), (32, 8, 531, 529), (16, 8, 2064, 1041),                # two groups, 129 .. 256
])
def test_block_prefill_matches_oracle(dev, hq, hkv, start, T):
    say(f"block prefill hq={hq} hkv={hkv} start={start} T={T}")
    pool, table, q, k, v = _case(hq, hkv, start, T)
    pos = np.arange(start, start + T)
    slots = (table[pos // 16].astype(np.int64) * 16 + pos % 16).astype(np.int32)
    p1, p2, tb, qd, kd, vd = (to_dev(x, dev) for x in (pool, pool, table, q, k, v))
    store_kv(p1, to_dev(slots, dev), None, kd, vd)
    o1 = paged_attention(qd, p1, tb, None, None, query_start=start)
    o2 = store_kv_and_prefill(qd, p2, tb, kd, vd, query_start=start)
    assert torch.equal(p1.view(torch.int16), p2.view(torch.int16)), "pool differs from store_kv's"
    assert torch.equal(o1.view(torch.int16), o2.view(torch.int16)), "output differs from the two-launch chunk"
    oracle.store_kv(pool, slots, None, k, v)
    # (a sample of rows from every 128-row block where the chunk is long: about 300 rows)
    rows = np.unique(np.concatenate([np.arange(0, T, max(1, T // 280)), np.arange(max(0, T - 20), T)]))
    ref = oracle.paged_attention_rows(q[rows], pool, np.repeat(table[None], len(rows), axis=0),
                                      (start + 1 + rows).astype(np.int32))
    assert_attn_close(o2[torch.as_tensor(rows, device=dev)], ref, f"start={start} T={T}")


@pytest.mark.parametrize("hq,start,T", [(64, 0, 1030), (64, 64, 560), (64, 320, 300)])
def test_block_prefill_bad_pages(dev, hq, start, T):
    """Pages outside the pool, before the chunk and in it: nothing stored, their keys not attended."""
    say(f"block prefill bad pages start={start} T={T}")
    bad = [(start // 16 + 3, 1 << 20), (start // 16 + 17, -1)] + ([(1, -7), (start // 16 - 1, 1 << 30)] if start else [])
    pool, table, q, k, v = _case(hq, 8, start, T, bad)
    ok = (table >= 0) & (table < pool.shape[1])
    pos = np.arange(start, start + T)
    slots = np.where(ok[pos // 16], table[pos // 16].astype(np.int64) * 16 + pos % 16, -1).astype(np.int32)
    p2 = to_dev(pool, dev)
    o2 = store_kv_and_prefill(to_dev(q, dev), p2, to_dev(table, dev), to_dev(k, dev), to_dev(v, dev), query_start=start)
    oracle.store_kv(pool, slots, None, k, v)
    assert np.array_equal(p2.cpu().numpy().view(np.uint16), pool.view(np.uint16))
    # the same attention over the valid pages alone (softmax does not depend on the keys' order)
    rows = np.arange(0, T, 7)
    lens, tabs = [], []
    for r in rows:
        n = start + r + 1
        last = (n - 1) // 16
        full = [int(table[i]) for i in range(last) if ok[i]]
        tail = n - 16 * last if ok[last] else 0
        tabs.append(full + ([int(table[last])] if tail else []))
        lens.append(16 * len(full) + tail)
    t2 = np.zeros((len(rows), table.shape[0]), np.int32)
    for i, t in enumerate(tabs):
        t2[i, :len(t)] = t
    ref = oracle.paged_attention_rows(q[rows], pool, t2, np.asarray(lens, np.int32))
    assert_attn_close(o2[torch.as_tensor(rows, device=dev)], ref, f"bad pages start={start} T={T}")


# one group from 512 workgroups and in 257 .. 511, two groups in 257 .. 511 and 129 .. 256
@pytest.mark.parametrize("hq,start,T", [(64, 0, 1031), (64, 608, 517), (32, 736, 1100), (64, 288, 272)])
def test_block_prefill_in_place(dev, hq, start, T):
    """The pre-append chunk as one call attends in place (its queries lie in the output): equal to the two calls."""
    say(f"block prefill in place hq={hq} start={start} T={T}")
    pool, table, q, k, v = _case(hq, 8, start, T)
    p1, p2, tb, qd, kd, vd = (to_dev(x, dev) for x in (pool, pool, table, q, k, v))
    g = torch.Generator(device=dev).manual_seed(T)
    qf, kf, vf = (x.float() + 1e-3 * torch.randn(x.shape, generator=g, device=dev) for x in (qd, kd, vd))
    w = 1 + 0.1 * torch.randn((2, 128), generator=g, device=dev)
    rope = rope_table(start + T, 128, 1e6, device=dev)
    pos = np.arange(start, start + T, dtype=np.int32)
    slots = (table[pos // 16].astype(np.int64) * 16 + pos % 16).astype(np.int32)
    q16 = qk_norm_rope_append(qf, kf, vf, w[0], w[1], rope, to_dev(pos, dev), to_dev(slots, dev), None, p1)
    o1 = paged_attention(q16, p1, tb, None, query_start=start)
    o2 = qk_norm_rope_append_and_prefill(qf, kf, vf, w[0], w[1], rope, p2, tb, query_start=start)
    assert torch.equal(p1.view(torch.int16), p2.view(torch.int16)), "pools differ"
    assert torch.equal(o1.view(torch.int16), o2.view(torch.int16)), "outputs differ"
