"""Native wrapper calls against the checked Python path: same results, same refusals."""
import ctypes
import sys

import pytest
import torch

from gpu_util import say
from infurnace_amd import _capi
from infurnace_amd.kernels import _fast, decode_plan, kv_prep, kv_store, rope_table
from infurnace_amd.kernels import KVStoreError, PagedAttentionError, DeviceArray

pytestmark = pytest.mark.gpu
att = sys.modules["infurnace_amd.kernels.paged_attention"]
H, F, I = torch.float16, torch.float32, torch.int32


class _Data:
    def __init__(self, dev, B=5, hq=16, hkv=8, d=128, layers=2):
        g = torch.Generator(device=dev).manual_seed(B + hq + d)
        r = lambda *s, t=H: torch.randn(s, generator=g, device=dev, dtype=F).to(t)
        lens = [37, 300, 1, 64, 129][:B]
        self.table = torch.randperm(B * 20, generator=g, device=dev)[:B * 20].view(B, 20).to(I)
        self.pool = r(layers, 2, B * 20, 16, hkv, d)
        self.lens = torch.tensor(lens, dtype=I, device=dev)
        pos = self.lens - 1
        self.pos = pos
        self.slots = (self.table[torch.arange(B, device=dev), (pos // 16).long()] * 16 + pos % 16).to(I)
        self.q, self.k, self.v = r(B, hq, d), r(B, hkv, d), r(B, hkv, d)
        self.qf, self.kf, self.vf = r(B, hq, d, t=F), r(B, hkv, d, t=F), r(B, hkv, d, t=F)
        self.qw, self.kw = r(d, t=F), r(d, t=F)
        self.rope = rope_table(320, d, 1e6, device=dev)
        self.act = torch.tensor([1, 0, 1, 1, 1][:B], dtype=torch.uint8, device=dev)


def _calls(t):
    """(name, native function, wrapper, checked function, arguments after the pool's, options) of every entry."""
    pa, sd, sp = att.paged_attention, att.store_kv_and_decode, att.store_kv_and_prefill
    decode = [{}, dict(layer=1), dict(scale=0.07), dict(max_seq_len=200), dict(out=1), dict(active=1), dict(active=2),
              dict(plan=1), dict(plan=2), dict(single=1)]
    for o in decode:
        yield "decode", pa, att._paged_attention, lambda p, x: ((t.q, p, t.table, t.lens, x), {}), o
        yield "decode", sd, att._store_kv_and_decode, \
            lambda p, x: ((t.q, p, t.table, t.lens, x, t.slots, t.k, t.v), {}), dict(o, slots=1)
        yield "prep_decode", kv_prep.qk_norm_rope_store_and_decode, kv_prep._qk_norm_rope_store_and_decode, \
            lambda p, x: ((t.qf, t.kf, t.vf, t.qw, t.kw, t.rope, t.pos, t.slots, x, p, t.table, t.lens), {}), \
            dict(o, slots=1)
    for o in ({}, dict(shared=0), dict(shared=2, layer=1)):
        yield "decode", pa, att._paged_attention, lambda p, x: ((t.q, p, t.table, t.lens, x), {}), o
    for o in ({}, dict(layer=1), dict(scale=0.07), dict(out=1), dict(single=1)):
        yield "prefill", pa, att._paged_attention, lambda p, x: ((t.q, p, t.table[0], None), dict(query_start=7)), o
        yield "prefill", sp, att._store_kv_and_prefill, \
            lambda p, x: ((t.q, p, t.table[:1], t.k, t.v), dict(query_start=32)), o
        yield "prep_prefill", kv_prep.qk_norm_rope_append_and_prefill, kv_prep._qk_norm_rope_append_and_prefill, \
            lambda p, x: ((t.qf, t.kf, t.vf, t.qw, t.kw, t.rope, p, t.table[0]), dict(query_start=32)), o
    for o in ({}, dict(layer=1), dict(active=1), dict(active=2), dict(single=1)):
        yield "prep_append", kv_prep.qk_norm_rope_append, kv_prep._qk_norm_rope_append, \
            lambda p, x: ((t.qf, t.kf, t.vf, t.qw, t.kw, t.rope, t.pos, t.slots, x, p), {}), o
        yield "store", kv_store.store_kv, kv_store._store_kv, lambda p, x: ((p, t.slots, x, t.k, t.v), {}), o
    yield "store_layers", kv_store.store_kv_layers, kv_store._store_kv_layers, \
        lambda p, x: ((p, t.slots, x, torch.stack([t.k] * 2), torch.stack([t.v] * 2)), {}), {}


def _options(t, o, p, args, planned):
    kw = {k: v for k, v in o.items() if k in ("layer", "scale", "max_seq_len")}
    if o.get("out"):
        kw["out"] = torch.full(t.q.shape, 7.0, dtype=H, device=t.q.device)
    if "shared" in o:
        kw["shared_prefix_pages"] = t.table[0, :0].contiguous()
        if o["shared"]:
            kw["shared_prefix_pages"] = t.common
    if o.get("plan"):
        kw["plan"] = planned
    return kw


def test_native_calls_equal_the_checked_path(dev, monkeypatch):
    t = _Data(dev)
    t.table[:, :2] = t.table[0, :2]
    t.common = t.table[0, :2].contiguous()
    t.slots = (t.table[torch.arange(5, device=dev), (t.pos // 16).long()] * 16 + t.pos % 16).to(I)
    t.slots[2] = t.table[2, 10] * 16  # (row 2's own position lies in a page that every row reads)
    taken = []
    for n in _fast._NAMES:
        fn = getattr(_fast.load(), n)
        monkeypatch.setattr(_fast, n, lambda *a, _f=fn, _n=n: taken.append((_n, r := _f(*a))) or r)
    for name, wrapper, checked, build, o in _calls(t):
        say(f"native {wrapper.__name__} {o}")
        act = None if not o.get("active") else t.act if o["active"] == 1 else t.act.bool()
        got = []
        for fn in (checked, wrapper, wrapper):  # (the checked call first: it grows the workspace)
            p = t.pool.clone()
            if o.get("single"):
                p = p[0].clone()
            args, kw = build(p, act)
            plan = None
            if o.get("plan"):
                plan = decode_plan(t.q.shape, p, t.table, t.lens, None, t.slots if o.get("slots") else None,
                                   lazy=o["plan"] == 2)
            kw = dict(kw, **_options(t, o, p, args, plan))
            del taken[:]
            r = fn(*args, **kw)
            if fn is wrapper:
                assert taken and taken[0][0] == name and taken[0][1] is not None, "the native call declined"
            if "out" in kw:
                assert r is kw["out"]
            if plan is not None:
                assert not plan.pending
            torch.cuda.synchronize()
            got.append((r, p))
        for r, p in got[1:]:
            assert torch.equal(p.view(torch.int16), got[0][1].view(torch.int16))
            if r is not None:
                assert torch.equal(r.view(torch.int16), got[0][0].view(torch.int16))


def test_native_calls_leave_refusals_to_the_checked_path(dev):
    """Errors, carriers, subclasses, modes and odd values go to the Python path, with its results."""
    say("native refusals")
    t = _Data(dev)
    ref = att._paged_attention(t.q, t.pool, t.table, t.lens)
    ok = lambda *a, **k: torch.equal(att.paged_attention(*a, **k).view(torch.int16), ref.view(torch.int16))
    da = DeviceArray(t.q.data_ptr(), t.q.shape, "float16", device=0, owner=t.q)
    assert ok(da, t.pool, t.table, t.lens)
    assert ok(torch.nn.Parameter(t.q, requires_grad=False), t.pool, t.table, t.lens)
    with dev:  # (a function mode)
        assert ok(t.q, t.pool, t.table, t.lens)
    assert ok(t.q, t.pool, t.table, t.lens, validate=True)
    for bad in (dict(layer=2), dict(scale=-1.0), dict(scale=float("nan")), dict(max_seq_len=-1), dict(block_size=32)):
        with pytest.raises(PagedAttentionError):
            att.paged_attention(t.q, t.pool, t.table, t.lens, **bad)
    with pytest.raises(PagedAttentionError):
        att.paged_attention(t.q.transpose(1, 2).contiguous().transpose(1, 2), t.pool, t.table, t.lens)
    with pytest.raises(PagedAttentionError):
        att.paged_attention(t.q, t.pool, t.table.long(), t.lens)
    with pytest.raises(KVStoreError):
        kv_store.store_kv(t.pool, t.slots[:3], None, t.k, t.v)
    plan = decode_plan(t.q.shape, t.pool, t.table, t.lens, None, t.slots)
    with pytest.raises(PagedAttentionError):  # another mask than the plan's
        att.store_kv_and_decode(t.q, t.pool.clone(), t.table, t.lens, t.act, t.slots, t.k, t.v, plan=plan)
    plain = decode_plan(t.q.shape, t.pool, t.table, t.lens)
    with pytest.raises(PagedAttentionError):  # a plan without slots
        att.store_kv_and_decode(t.q, t.pool.clone(), t.table, t.lens, None, t.slots, t.k, t.v, plan=plain)
    empty = att.paged_attention(t.q[:0], t.pool, t.table[:0], t.lens[:0])
    assert empty.shape == (0, 16, 128)


def test_native_call_uses_the_current_stream(dev):
    say("native current stream")
    t = _Data(dev)
    ref = att._paged_attention(t.q, t.pool, t.table, t.lens)
    torch.cuda.synchronize()
    s = torch.cuda.Stream(device=dev)
    with torch.cuda.stream(s):
        for _ in range(3):
            o = att.paged_attention(t.q, t.pool, t.table, t.lens)
    s.synchronize()
    assert torch.equal(o.view(torch.int16), ref.view(torch.int16))
    assert (dev.index or 0, s.cuda_stream) in att._WORKSPACES


def test_failed_launch_raises_once(dev):
    """An entry point that reports a failed launch is not called again: its error reaches the caller.  (The
    entries stand in on the host; nothing is launched.)"""
    say("native failed launch")
    t = _Data(dev)
    wrappers = [lambda: att._paged_attention(t.q, t.pool, t.table, t.lens),
                lambda: att._paged_attention(t.q, t.pool, t.table[0], None, query_start=32)]
    for w in wrappers:  # (the workspace is there)
        w()
    torch.cuda.synchronize()
    calls = []
    status = _capi.IFN_ERR_HIP

    @ctypes.CFUNCTYPE(ctypes.c_int)
    def failing():
        calls.append(1)
        return status
    lib = _capi.lib()
    at = [ctypes.cast(failing if not n.endswith("_bytes") else getattr(lib, n), ctypes.c_void_p).value
          for n in _fast._ENTRIES]
    each = [lambda: att.paged_attention(t.q, t.pool, t.table, t.lens),
            lambda: att.store_kv_and_decode(t.q, t.pool, t.table, t.lens, None, t.slots, t.k, t.v),
            lambda: kv_prep.qk_norm_rope_store_and_decode(t.qf, t.kf, t.vf, t.qw, t.kw, t.rope, t.pos, t.slots, t.act,
                                                          t.pool, t.table, t.lens),
            lambda: att.paged_attention(t.q, t.pool, t.table[0], None, query_start=32),
            lambda: att.store_kv_and_prefill(t.q, t.pool, t.table[0], t.k, t.v, query_start=32),
            lambda: kv_prep.qk_norm_rope_append_and_prefill(t.qf, t.kf, t.vf, t.qw, t.kw, t.rope, t.pool, t.table[0],
                                                            query_start=32),
            lambda: kv_prep.qk_norm_rope_append(t.qf, t.kf, t.vf, t.qw, t.kw, t.rope, t.pos, t.slots, None, t.pool),
            lambda: kv_store.store_kv(t.pool, t.slots, None, t.k, t.v),
            lambda: kv_store.store_kv_layers(t.pool, t.slots, None, torch.stack([t.k] * 2), torch.stack([t.v] * 2))]
    ext = _fast.load()
    try:
        ext.bind("".join(map(_fast._signature, _fast._ENTRIES)), *at)
        for fn in each:
            del calls[:]
            with pytest.raises(_capi.KernelLaunchError) as e:
                fn()
            assert e.value.status == status and len(calls) == 1
        status = _capi.IFN_ERR_WORKSPACE  # (a refusal: the checked path makes the call)
        ref = att._paged_attention(t.q, t.pool, t.table, t.lens)
        assert torch.equal(each[0]().view(torch.int16), ref.view(torch.int16))
    finally:
        _fast.load()


@pytest.mark.parametrize("hq,hkv,d", [(16, 4, 128), (8, 2, 128), (16, 8, 64), (8, 4, 256)])
def test_pre_append_shapes_without_a_fused_kernel_are_declined_first(dev, hq, hkv, d):
    """No output is allocated (or cleared) for a pre-append step that the fused kernel does not cover."""
    say(f"native pre-append declined hq={hq} hkv={hkv} d={d}")
    t = _Data(dev, hq=hq, hkv=hkv, d=d)
    call = lambda fn, **k: fn(t.qf, t.kf, t.vf, t.qw, t.kw, t.rope, t.pos, t.slots, t.act, t.pool, t.table, t.lens, **k)
    ref = call(kv_prep._qk_norm_rope_store_and_decode)  # (grows the workspace)
    before = torch.cuda.memory_stats(dev)["allocation.all.allocated"]
    assert _fast.prep_decode(t.qf, t.kf, t.vf, t.qw, t.kw, t.rope, t.pos, t.slots, t.act, t.pool, t.table, t.lens, 0,
                             1e-6, None, None, 16, None, None, att._WORKSPACES) is None
    assert torch.cuda.memory_stats(dev)["allocation.all.allocated"] == before
    assert torch.equal(call(kv_prep.qk_norm_rope_store_and_decode).view(torch.int16), ref.view(torch.int16))
