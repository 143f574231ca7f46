"""Prefill attention with a KV head's query heads on two workgroups (5..8 query
heads per KV head), one block per workgroup in folded order (D = 64), and on
pages behind a cached prefix with and without a split of the keys: at the edges
of query blocks and key tiles, against attention in 64 bits, to the tolerance of
the other attention tests (2e-3 + 1e-2 |r|; the largest error 2e-3).
"""
import math

import numpy as np
import pytest

import kvhp
from gpu_util import assert_attn_close, note

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _reference(q, k, v):
    B, S, hq, d = q.shape
    g = hq // k.shape[2]
    mask = torch.ones(S, S, dtype=torch.bool, device="cuda").triu(1)
    out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    for b in range(B):
        for h in range(hq):
            kt = k[b, :, h // g].double().t().contiguous()
            s = (q[b, :, h].double() @ kt / math.sqrt(d)).masked_fill(mask, -math.inf)
            out[b, :, h] = torch.softmax(s, 1) @ v[b, :, h // g].double()
    return out


@pytest.mark.parametrize("hq,hkv,d", [(5, 1, 64), (12, 2, 64), (14, 2, 64), (8, 1, 64), (10, 2, 128),
                                      (7, 1, 128), (16, 2, 128), (8, 2, 64), (4, 4, 64)])
@pytest.mark.parametrize("s,batch", [(1, 2), (31, 1), (33, 1), (64, 3), (65, 1), (96, 1), (500, 1),
                                     (777, 2)])
def test_head_groups(hq, hkv, d, s, batch):
    _check_prefill(hq, hkv, d, s, batch)


@pytest.mark.parametrize("hq,hkv,s,batch", [(8, 4, 500, 16), (8, 4, 300, 25), (16, 2, 333, 9),
                                            (5, 1, 260, 33), (2, 2, 250, 61), (4, 2, 20, 40),
                                            (7, 1, 31, 120), (32, 8, 333, 3)])
def test_folded_batches(hq, hkv, s, batch):
    """Batches whose blocks are all resident at once, two on a CU: every block of
    every sequence once, with more and with fewer workgroups of one rank than CUs
    and a single block a sequence."""
    _check_prefill(hq, hkv, 64, s, batch)


def _check_prefill(hq, hkv, d, s, batch):
    note(f"prefill groups {hq}/{hkv}x{d} S={s} B={batch}")
    torch.manual_seed(s + hq)
    q = torch.randn(batch, s, hq, d, device="cuda").half()
    k = torch.randn(batch, s, hkv, d, device="cuda").half()
    v = torch.randn(batch, s, hkv, d, device="cuda").half()
    out = torch.full_like(q, float("nan"))
    pages = (s + 15) // 16
    bt = torch.randperm(batch * pages, device="cuda").int().view(batch, pages)
    pk = torch.zeros(hkv, batch * pages, 16, d, dtype=torch.float16, device="cuda")
    pv = torch.zeros_like(pk)
    kvhp.flash_prefill_paged(q, k, v, out, s, hq, hkv, d, batch, pk, pv, bt)
    torch.cuda.synchronize()
    assert_attn_close(out.float().cpu(), _reference(q, k, v).cpu().numpy(), "head groups")
    for b in range(batch):
        rows = (bt[b].long()[:, None] * 16 + torch.arange(16, device="cuda")).reshape(-1)[:s]
        assert torch.equal(pk.view(hkv, -1, d)[:, rows], k[b].transpose(0, 1))
        assert torch.equal(pv.view(hkv, -1, d)[:, rows], v[b].transpose(0, 1))


@pytest.mark.parametrize("hq,hkv,d", [(16, 2, 64), (14, 2, 64), (4, 1, 64), (6, 3, 64), (2, 2, 64),
                                      (5, 1, 128), (8, 1, 128), (3, 1, 64)])
def test_cached_prefix(hq, hkv, d):
    """A prompt behind its own first positions' pages: logits and pages as the
    whole prompt's (two roundings of one forward: 4e-3 relative, as the prompt
    tests assert against 64 bits).  (3 heads per KV head: the decode-row route.)"""
    cfg = kvhp.LlamaConfig(544, hq * d, 2, hq, hkv, d, 512, 1e-5, 10000.0, 0)
    m = kvhp.LlamaModel(cfg, 11, 1300)
    rng = np.random.default_rng(hq * d)
    for n, first in ((40, 1), (49, 16), (96, 32), (97, 33), (200, 150), (320, 255), (700, 512),
                     (1290, 1200), (1290, 640), (1290, 7)):
        note(f"cached prefix {hq}/{hkv}x{d} n={n} first={first}")
        ids = rng.integers(0, 544, n).astype(np.int32)
        p = (n + 15) // 16 + 1
        perm = rng.permutation(p)
        bt = torch.from_numpy(perm[:p - 1].astype(np.int32)).cuda()
        whole = torch.zeros((2, 2, hkv, p, 16, d), dtype=torch.float16, device="cuda")
        _, want = m.prefill_paged(ids, whole, p, bt, p - 1)
        pool = whole.clone()
        # what lies past the prefix is not read before it is written: poisoned
        rows = (bt.long()[:, None] * 16 + torch.arange(16, device="cuda")).reshape(-1)
        flat = pool.view(2, 2, hkv, p * 16, d)
        flat[:, :, :, rows[first:]] = float("nan")
        _, got = m.prefill_cached(ids, first, pool, p, bt, p - 1)
        rel = np.linalg.norm(got - want) / np.linalg.norm(want)
        assert rel < 4e-3, (n, first, rel)
        a, b = flat[:, :, :, rows[:n]].double(), whole.view(2, 2, hkv, p * 16, d)[:, :, :, rows[:n]].double()
        assert float((a - b).norm() / b.norm()) < 4e-3
        assert bool(flat[:, :, :, rows[n:]].isnan().all())     # nothing past the prompt
        assert not bool(pool[:, :, :, int(perm[p - 1])].any())
    m.close()
