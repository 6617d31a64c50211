"""The wrappers' native argument checks decline what is not theirs (CPU: no call may reach a kernel)."""
import os
import re

import numpy as np
import pytest
import torch

from infurnace_amd import _capi
from infurnace_amd.build import CSRC
from infurnace_amd.kernels import (KVStoreError, PagedAttentionError, _fast, paged_attention, qk_norm_rope_append,
                                   store_kv, store_kv_and_decode)

H = torch.float16
POOL = torch.zeros((2, 4, 16, 8, 128), dtype=H)
I = torch.zeros(3, dtype=torch.int32)
Q = torch.zeros((3, 16, 128), dtype=H)
KV = torch.zeros((3, 8, 128), dtype=H)
BT = torch.zeros((3, 1), dtype=torch.int32)


def test_declines_everything_that_is_no_gpu_tensor():
    ext = _fast.load()
    decode = [Q, POOL, BT, I, None, I, KV, KV, 0, None, None, 16, None, None, None, {}]
    assert ext.decode(*decode) is None
    for i in range(len(decode)):
        for odd in (None, 1.5, "x", np.zeros(3), object(), Q.to("meta")):
            assert ext.decode(*decode[:i], odd, *decode[i + 1:]) is None
    assert ext.decode() is None and ext.decode(*decode, 1) is None  # wrong counts
    assert ext.store(POOL, I, None, KV, KV, 0) is None and ext.store_layers(POOL[None], I, None, KV[None], KV[None]) is None
    assert ext.prefill(Q, POOL, BT[0], None, None, 0, 0, None, None, 16, {}) is None
    assert ext.prep_append(Q, KV, KV, Q, Q, Q, I, I, None, POOL, 0, 1e-6, None) is None
    assert ext.prep_decode(*([None] * 20)) is None and ext.prep_prefill(*([None] * 15)) is None
    with pytest.raises(TypeError):
        ext.bind(1)


def test_errors_are_the_checked_path_s():
    with pytest.raises(KVStoreError):
        store_kv(POOL, I, None, KV, KV)
    with pytest.raises(KVStoreError):
        store_kv(POOL.float(), I, None, KV, KV)
    with pytest.raises(PagedAttentionError):
        paged_attention(Q, POOL, BT, I)
    with pytest.raises(PagedAttentionError):
        store_kv_and_decode(Q, POOL, BT, I, None, None, KV, KV)
    with pytest.raises(KVStoreError):
        qk_norm_rope_append(Q.float(), KV.float(), KV.float(), Q, Q, Q, I, I, None, POOL)
    with pytest.raises(TypeError):
        store_kv(POOL[None], I, None, KV, KV, layer=None)


def test_device_work_leaves_the_gil():
    """Whatever can wait for the device -- an entry point, an output's allocation and fill -- runs without the GIL:
    a full queue behind a host function that needs it would otherwise never drain."""
    src = open(os.path.join(CSRC, "fast_call.cpp")).read()
    work = re.findall(r"at::(?:zeros|empty)\(|\bE\.\w+(?=, )", src)
    out = re.sub(r"(?:unlocked|launch)\((?:[^()]|\((?:[^()]|\([^()]*\))*\))*\)", "", src)
    assert len(work) > 12 and re.findall(r"at::(?:zeros|empty)\(|\bE\.\w+(?=, )", out) == []


def test_extension_of_other_signatures_is_not_bound(monkeypatch):
    """The extension is bound to addresses only where the declared signatures are those it was compiled with."""
    res, args = _capi.SIGNATURES["ifn_store_kv"]
    monkeypatch.setitem(_capi.SIGNATURES, "ifn_store_kv", (res, [*args[:1], *args[2:]]))
    with pytest.raises(ImportError):
        _fast.load()


@pytest.mark.parametrize("error", [ImportError, OSError, TypeError, AttributeError])
def test_unusable_extension_leaves_the_checked_path(monkeypatch, error):
    """Missing, stale or unloadable: the wrappers say so once and take their Python path."""
    def load():
        raise error("no such extension")
    monkeypatch.setattr(_fast, "load", load)
    for n in _fast._NAMES:
        monkeypatch.setattr(_fast, n, _fast._first(n))
    with pytest.warns(RuntimeWarning, match="_fast_call"), pytest.raises(KVStoreError):
        store_kv(POOL, I, None, KV, KV)
    with pytest.raises(PagedAttentionError):
        paged_attention(Q, POOL, BT, I)
