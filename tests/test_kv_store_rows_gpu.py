"""store_kv_layers on token rows of 2 KiB, 1 KiB and 512 B, at the edges of a workgroup's tokens: bit-exact."""
import numpy as np
import pytest
import torch

import oracle
from gpu_util import say, to_dev
from infurnace_amd.kernels import store_kv_layers

pytestmark = pytest.mark.gpu


# a workgroup holds 1 or 4 tokens (four times as many in larger calls, of 2 KiB rows
# 1 again in the largest); 1 KiB rows take the general path
@pytest.mark.parametrize("hkv,d,layers,tokens",
                         [(4, 128, 1, t) for t in (1, 2, 3, 130)] + [(2, 128, 1, t) for t in (1, 4, 5, 127)]
                         + [(8, 64, 3, 17), (4, 64, 2, 18), (1, 256, 1, 3),
                            (8, 128, 4, 1025), (8, 128, 20, 1001), (4, 128, 4, 2049), (8, 64, 4, 2047),
                            (4, 128, 4, 2055), (2, 128, 8, 2049), (2, 128, 8, 2063)])
def test_rows_bit_exact(dev, hkv, d, layers, tokens):
    say(f"store rows hkv={hkv} d={d} layers={layers} tokens={tokens}")
    rng = np.random.default_rng(hkv * d + tokens)
    pages = -(-tokens // 16) + 3
    # (any bits, NaN too)
    draw = lambda *s: rng.integers(0, 1 << 16, size=s, dtype=np.uint16).view(np.float16)
    pool, k, v = draw(layers, 2, pages, 16, hkv, d), draw(layers, tokens, hkv, d), draw(layers, tokens, hkv, d)
    slots = rng.permutation(pages * 16)[:tokens].astype(np.int32)
    mask = rng.random(tokens) < 0.9
    slots[tokens // 3], slots[tokens // 2] = -1, pages * 16  # (skipped, as the inactive rows are)
    if tokens == 1:
        slots[0] = 5
    for active in (None, mask):
        p = to_dev(pool, dev)
        store_kv_layers(p, to_dev(slots, dev), None if active is None else to_dev(active, dev), to_dev(k, dev),
                        to_dev(v, dev))
        want = pool.copy()
        for i in range(layers):
            oracle.store_kv(want[i], slots, active, k[i], v[i])
        torch.cuda.synchronize()
        assert torch.equal(p.cpu().view(torch.int16), torch.from_numpy(want.view(np.int16)))
