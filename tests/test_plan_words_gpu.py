"""Every word of a step plan is written: plans built over different garbage are identical, whichever
call builds them (ifn_paged_decode_plan, ifn_paged_decode_planning), and none needs clearing first."""
import numpy as np
import pytest
import torch

from gpu_util import say, to_dev
from infurnace_amd import _capi
from infurnace_amd.kernels import decode_plan, paged_attention
from infurnace_amd.kernels.paged_attention import workspace_for
from test_decode_planning_gpu import _case

pytestmark = pytest.mark.gpu


# batches around the record area's start (header and offsets rounded up to 64 words: 47, 48), one row,
# fewer ranges than workgroups, more pieces than a record holds, rows without keys
@pytest.mark.parametrize("batch,hi", [(1, 5), (1, 900), (3, 40), (47, 300), (48, 300), (700, 30)])
def test_plan_writes_every_word(dev, batch, hi):
    say(f"plan words batch={batch} hi={hi}")
    rng = np.random.default_rng(batch + hi)
    lens = rng.integers(0 if batch > 3 else hi, hi + 1, size=batch)
    pool, table, lens, q = _case(rng, lens, 16, 8, 128)
    qd, p, bt, sl = (to_dev(x, dev) for x in (q, pool, table, lens))
    mp, msl, P = table.shape[1], int(lens.max()), pool.shape[1]
    L = _capi.lib()
    st = torch.cuda.current_stream(dev).cuda_stream
    nbytes = L.ifn_paged_decode_plan_bytes(batch, 16, 8, 128, 16, mp, msl)
    ws = workspace_for(dev, st, L.ifn_paged_decode_workspace_bytes(batch, 16, 8, 128, 16, msl))
    bufs = [torch.full((nbytes,), fill, dtype=torch.uint8, device=dev) for fill in (0xA5, 0x5A, 0xFF)]
    for b in bufs[:2]:
        assert L.ifn_paged_decode_plan(b.data_ptr(), nbytes, bt.data_ptr(), mp, sl.data_ptr(), None, None, P, batch, 16,
                                       8, 128, 16, msl, st) == 0
    out = torch.empty_like(qd)
    assert L.ifn_paged_decode_planning(out.data_ptr(), qd.data_ptr(), p.data_ptr(), P, bt.data_ptr(), mp, sl.data_ptr(),
                                       None, batch, 16, 8, 128, 16, msl, 0.0, bufs[2].data_ptr(), nbytes, ws.data_ptr(),
                                       ws.numel(), st) == 0
    torch.cuda.synchronize()
    assert torch.equal(bufs[0], bufs[1]) and torch.equal(bufs[0], bufs[2])


def test_shared_prefix_plan_words(dev):
    """The shared-prefix plan of 2 KiB token rows writes every word too; smaller rows, whose shared-prefix decode
    reads no plan, get an empty one."""
    say("shared-prefix plan words")
    rng = np.random.default_rng(6)
    for hq, hkv, d in ((16, 8, 128), (16, 4, 128), (8, 2, 128), (16, 8, 64)):
        pool, table, lens, q = _case(rng, [40, 700, 33, 90], hq, hkv, d)
        table[:, :2] = table[0, :2]
        qd, p, bt, sl = (to_dev(x, dev) for x in (q, pool, table, lens))
        pages = bt[0, :2].contiguous()
        plan = decode_plan(q.shape, p, bt, sl, shared_prefix_pages=pages)
        out = paged_attention(qd, p, bt, sl, shared_prefix_pages=pages, plan=plan, validate=True)
        ref = paged_attention(qd, p, bt, sl, shared_prefix_pages=pages)
        assert torch.equal(out.view(torch.int16), ref.view(torch.int16))
        assert (plan.buf is None) == (hkv * d < 1024)
        if plan.buf is None:
            continue
        L, st = _capi.lib(), torch.cuda.current_stream(dev).cuda_stream
        for fill in (0xA5, 0xFF):
            b = torch.full_like(plan.buf, fill)
            assert L.ifn_paged_decode_shared_prefix_plan(b.data_ptr(), b.numel(), bt.data_ptr(), table.shape[1],
                                                         sl.data_ptr(), None, 2, p.shape[1], 4, hq, hkv, d, 16,
                                                         table.shape[1] * 16, st) == 0
            assert torch.equal(b, plan.buf)
