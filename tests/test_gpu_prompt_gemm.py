"""The prompt's projections (serving-engine_amd/csrc/gemm.hip) through the model
entry points, at row counts on both sides of every tile edge and of the split
over K: logits and the K/V pages of every layer against the same forward in 64
bits on the GPU (plain torch).  The forward rounds activations to fp16 after every
operator (2^-11 relative each, independent): through two layers the relative
2-norm error stays below 2e-3, and the batched step's too; 4e-3 is asserted.  A
tile read or written in the wrong place is an error of order 1.  Dimensions that
those kernels do not take run on the library's products with the row-wise operators
between them, and are held to the same.
"""
import math

import numpy as np
import pytest

import kvhp
from gpu_util import note

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

# hidden 576 = 9 heads of 64 (tile tails in N), ffn 1472 = 23 steps of 64; heads of 128;
# ffn 4864 = 76 steps: 8 ranges of K, the last one shorter
CONFIGS = {
    "d64": (544, 576, 2, 9, 3, 64, 1472),
    "d128": (512, 1024, 2, 8, 2, 128, 2816),
    "ffn4864": (544, 576, 2, 9, 3, 64, 4864),
}
# on the library's products: heads of 32; ffn not a multiple of 64 (attention behind a
# cached prefix on the flash route); a vocabulary not a multiple of 32 (the head alone)
LIBRARY = {
    "d32": (544, 512, 2, 16, 4, 32, 1408),
    "ffn1440": (544, 512, 2, 8, 2, 64, 1440),
    "vocab550": (550, 576, 2, 9, 3, 64, 1472),
}


def _model(name, max_ctx):
    v, h, layers, hq, hkv, d, f = {**CONFIGS, **LIBRARY}[name]
    return kvhp.LlamaModel(kvhp.LlamaConfig(v, h, layers, hq, hkv, d, f, 1e-5, 10000.0, 0), 3,
                           max_ctx)


class _Ref:
    """The forward in 64 bits from the model's own weights."""

    def __init__(self, m):
        self.c, g = m.config, lambda l, w: torch.from_numpy(m.tensor(l, w)).cuda().double()
        c = self.c
        H = c.hidden_size
        self.embed, self.head = g(-1, kvhp.LLAMA_EMBED).view(-1, H), g(-1, kvhp.LLAMA_LM_HEAD).view(-1, H)
        self.w = [[g(l, w) for w in (kvhp.LLAMA_W_QKV, kvhp.LLAMA_W_O, kvhp.LLAMA_W_GATE_UP,
                                     kvhp.LLAMA_W_DOWN)] for l in range(c.num_layers)]

    def _norm(self, x):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + self.c.rms_eps)

    def _rope(self, x, pos):
        d = self.c.head_dim
        inv = self.c.rope_theta ** (-torch.arange(0, d, 2, dtype=torch.float64, device="cuda") / d)
        a = pos.double()[:, None, None] * inv
        x1, x2 = x[..., :d // 2], x[..., d // 2:]
        return torch.cat([x1 * a.cos() - x2 * a.sin(), x2 * a.cos() + x1 * a.sin()], -1)

    def prompt(self, ids):
        """(logits of the last position, [layer][k/v][hkv][n][d])."""
        c = self.c
        n, hq, hkv, d = len(ids), c.num_q_heads, c.num_kv_heads, c.head_dim
        x, pos = self.embed[torch.as_tensor(ids).cuda().long()], torch.arange(n, device="cuda")
        mask = torch.ones(n, n, dtype=torch.bool, device="cuda").triu(1)
        cache = []
        for wqkv, wo, wgu, wd in self.w:
            qkv = (self._norm(x) @ wqkv.view(-1, c.hidden_size).t()).view(n, hq + 2 * hkv, d)
            q, k, v = self._rope(qkv[:, :hq], pos), self._rope(qkv[:, hq:hq + hkv], pos), qkv[:, hq + hkv:]
            cache.append([k.transpose(0, 1), v.transpose(0, 1)])
            out = torch.empty_like(q)
            for h in range(hq):
                kh, vh = k[:, h // (hq // hkv)], v[:, h // (hq // hkv)]
                s = (q[:, h] @ kh.t().contiguous() / math.sqrt(d)).masked_fill(mask, -math.inf)
                out[:, h] = torch.softmax(s, 1) @ vh
            x = x + out.reshape(n, -1) @ wo.view(c.hidden_size, -1).t()
            g, u = (self._norm(x) @ wgu.view(-1, c.hidden_size).t()).chunk(2, -1)
            x = x + (g * torch.sigmoid(g) * u) @ wd.view(c.hidden_size, -1).t()
        return self._norm(x[-1]) @ self.head.t(), cache


def _rel(got, ref):
    got = got.double()
    return float((got - ref).norm() / ref.norm())


def _pages(m, n, extra=0):
    c, p = m.config, (n + 15) // 16 + extra
    pool = torch.zeros((c.num_layers, 2, c.num_kv_heads, p, 16, c.head_dim), dtype=torch.float16,
                       device="cuda")
    return pool, p


def _check_prompt(m, ref, rng, name, n, first=0):
    """A prompt of n ids, its positions below `first` cached by another call."""
    note(f"prompt gemm {name} n={n} first={first}")
    ids = rng.integers(0, m.config.vocab_size, n).astype(np.int32)
    want, cache = ref.prompt(ids)
    pool, p = _pages(m, n, extra=1)
    perm = rng.permutation(p - 1).astype(np.int32)
    bt = torch.from_numpy(perm).cuda()
    if first:
        m.prefill_paged(ids[:first], pool, p, bt, p - 1)
        _, logits = m.prefill_cached(ids, first, pool, p, bt, p - 1)
    else:
        _, logits = m.prefill_paged(ids, pool, p, bt, p - 1)
    assert _rel(torch.from_numpy(logits).cuda(), want) < 4e-3
    rows = (bt.long()[:, None] * 16 + torch.arange(16, device="cuda")).reshape(-1)[:n]
    for l in range(m.config.num_layers):
        for kv in range(2):
            got = pool[l, kv].reshape(m.config.num_kv_heads, -1, m.config.head_dim)[:, rows]
            assert _rel(got, cache[l][kv]) < 4e-3, (n, l, kv)
    assert not bool(pool[:, :, :, p - 1].any())        # the page outside the table


@pytest.mark.parametrize("name", sorted(CONFIGS))
def test_prompt_rows_at_tile_edges(name):
    m = _model(name, 1100)
    ref = _Ref(m)
    rng = np.random.default_rng(4)
    for n in (1, 2, 31, 33, 63, 64, 65, 127, 129, 192, 257, 500, 513, 1030):
        _check_prompt(m, ref, rng, name, n)
    m.close()


@pytest.mark.parametrize("name", sorted(LIBRARY))
def test_prompt_on_library_products(name):
    """Whole prompts and prompts behind a cached prefix."""
    m = _model(name, 300)
    ref = _Ref(m)
    rng = np.random.default_rng(6)
    for n, first in ((1, 0), (2, 0), (33, 0), (130, 0), (300, 0), (60, 20), (131, 16), (300, 200)):
        _check_prompt(m, ref, rng, name, n, first)
    m.close()


@pytest.mark.parametrize("name,shift", [("d64", 0), ("d64", 1), ("d128", 0)] +
                         [(name, 0) for name in sorted(LIBRARY)])
def test_large_batch_step(name, shift):
    """More than 32 sequences: the same projections, positions per row, and the
    LM head of 544 columns (17 groups of 32; on the library's product where the
    logits start `shift` floats past a 16-byte boundary)."""
    m = _model(name, 64)
    ref = _Ref(m)
    rng = np.random.default_rng(5)
    B, n = 41, 21
    note(f"prompt gemm: batched step of 41, {name}, logits shifted by {shift}")
    ids = rng.integers(0, m.config.vocab_size, (B, n)).astype(np.int32)
    pool, p = _pages(m, 32 * B)
    bt = torch.from_numpy(rng.permutation(p).astype(np.int32).reshape(B, 2)).cuda()
    lens = rng.integers(2, n + 1, B).astype(np.int32)
    for b in range(B):
        m.prefill_paged(ids[b, :lens[b] - 1], pool, p, bt[b].contiguous(), 2)
    tok = torch.from_numpy(ids[np.arange(B), lens - 1]).cuda()
    ln = torch.from_numpy(lens).cuda()
    size = B * m.config.vocab_size
    buf = torch.full((size + 4,), 7.0, dtype=torch.float32, device="cuda")
    logits = buf[shift:shift + size].view(B, -1)
    nxt = torch.empty(B, dtype=torch.int32, device="cuda")
    m.decode_paged(tok, pool, p, bt, 2, ln - 1, ln, 32, logits, nxt)
    torch.cuda.synchronize()
    for b in range(B):
        want, _ = ref.prompt(ids[b, :lens[b]])
        assert _rel(logits[b], want) < 4e-3, b
    assert torch.equal(nxt.long(), logits.argmax(1))
    assert bool((buf[:shift] == 7).all()) and bool((buf[shift + size:] == 7).all())
    m.close()
