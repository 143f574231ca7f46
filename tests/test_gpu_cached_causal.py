"""A prompt behind a cached prefix is causal for any values: where a token's V
overflows fp16, the pages of the positions before it hold the bits that they hold
with an ordinary token in its place, and those from it on are not finite.

Through two layers (the second layer's K/V carry the first's attention output), on
the flash route over pages and on the decode-row route (3 heads per KV head), with
the token at the edges of key tiles, pages, query blocks and key splits.
"""
import numpy as np
import pytest

import kvhp
from gpu_util import note

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

V = 128


def _model(hq, hkv, d, max_ctx):
    h = hq * d
    m = kvhp.LlamaModel(kvhp.LlamaConfig(V, h, 2, hq, hkv, d, 512, 1e-5, 10000.0, 0), 9, max_ctx)
    # column 0 of the hidden state is the last token's alone, and the first
    # layer's V rows 1 and 2 of the last KV head take it far past 65504
    embed = m.tensor(-1, kvhp.LLAMA_EMBED).reshape(V, h).copy()
    embed[:, 0] = 0
    embed[V - 1] = 0
    embed[V - 1, 0] = 1
    m.set_tensor(-1, kvhp.LLAMA_EMBED, embed)
    w = m.tensor(0, kvhp.LLAMA_W_QKV).reshape(-1, h).copy()
    w[-d + 1, 0], w[-d + 2, 0] = 60000, -60000
    m.set_tensor(0, kvhp.LLAMA_W_QKV, w)
    return m


@pytest.mark.parametrize("hq,hkv,d", [(16, 2, 64), (14, 2, 64), (8, 2, 64), (4, 2, 64), (2, 2, 64),
                                      (8, 1, 128), (5, 1, 128), (2, 2, 128), (3, 1, 64)])
@pytest.mark.parametrize("n,first", [(97, 33), (200, 130), (700, 512), (1290, 640)])
def test_later_position_reaches_no_earlier_row(hq, hkv, d, n, first):
    m = _model(hq, hkv, d, n)
    rng = np.random.default_rng(n + hq)
    ids = rng.integers(0, V - 1, n).astype(np.int32)
    p = (n + 15) // 16
    perm = rng.permutation(p).astype(np.int32)
    bt = torch.from_numpy(perm).cuda()
    rows = (bt.long()[:, None] * 16 + torch.arange(16, device="cuda")).reshape(-1)
    start = torch.zeros((2, 2, hkv, p, 16, d), dtype=torch.float16, device="cuda")
    m.prefill_paged(ids[:first], start, p, bt, p)
    pool = start.clone()
    m.prefill_cached(ids, first, pool, p, bt, p)
    want = pool.view(2, 2, hkv, p * 16, d)[:, :, :, rows]
    assert bool(want[..., :n, :].isfinite().all())
    at = {first, first + 1, first + 31, first + 32, n // 64 * 64 - 1, n // 64 * 64, n - 2, n - 1}
    for z in sorted(z for z in at if first <= z < n):
        note(f"cached causal {hq}/{hkv}x{d} n={n} first={first} z={z}")
        other = ids.copy()
        other[z] = V - 1
        pool = start.clone()
        m.prefill_cached(other, first, pool, p, bt, p)
        got = pool.view(2, 2, hkv, p * 16, d)[:, :, :, rows]
        assert torch.equal(got[..., :z, :], want[..., :z, :]), z
        assert bool(got[0, 1, hkv - 1, z].isinf().any())
        assert not bool(got[1, 0, 0, z:n].isfinite().any()), z     # every later row sees it
    m.close()
