"""SwiGLU in the gate/up projection of a prompt: the bits of the separate SwiGLU
operator over the same fp16 gates and values, between gates of -30 and 19.

A two-layer model lays the products bare: x has two nonzero columns, so that gate
and up are single exact products rounded to fp16; the first layer's attention
output is zero and its down projection copies; the second layer's V pages are its
RMSNorm of the result.  The same steps through the row-wise operators must give
equal bits (an exponential of the rounded product -1.4427 g, 60 units of 2^-24 off
at g = -70 where expf is 2.4 off, moved about one in 2000 of these values).
"""
import numpy as np
import pytest

import kvhp
from gpu_util import note

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

H = F = 1024


@pytest.mark.parametrize("n", [33, 130, 700])
def test_prompt_swiglu_bits(n):
    note(f"prompt swiglu n={n}")
    d, heads, vocab = 64, H // 64, 1024
    m = kvhp.LlamaModel(kvhp.LlamaConfig(vocab, H, 2, heads, heads, d, F, 1e-5, 10000.0, 0), 1, n)
    rng = np.random.default_rng(n)
    angle = rng.uniform(0.5, 1.1, vocab)               # both columns positive
    embed = np.zeros((vocab, H), np.float16)
    embed[:, 0], embed[:, 1] = np.cos(angle), np.sin(angle)
    # gates 16..28 times the weight; up sized so that the product is a normal fp16
    alpha = rng.uniform(-1.05, 0.65, F).astype(np.float16)
    beta = np.where(alpha < 0, np.exp(np.clip(-26.0 * alpha.astype(np.float64), 0, 7.0)), 0.01)
    beta = (beta * rng.uniform(0.5, 1.0, F)).astype(np.float16)
    gate_up = np.zeros((2 * F, H), np.float16)
    gate_up[:F, 0], gate_up[F:, 1] = alpha, beta
    down = np.eye(H, F, dtype=np.float16)
    down[:2] = 0
    qkv = np.zeros((3 * H, H), np.float16)
    qkv[2 * H:] = np.eye(H, dtype=np.float16)
    m.set_tensor(-1, kvhp.LLAMA_EMBED, embed)
    m.set_tensor(0, kvhp.LLAMA_W_O, np.zeros((H, H), np.float16))
    m.set_tensor(0, kvhp.LLAMA_W_GATE_UP, gate_up)
    m.set_tensor(0, kvhp.LLAMA_W_DOWN, down)
    m.set_tensor(1, kvhp.LLAMA_W_QKV, qkv)
    ones = torch.ones(H, dtype=torch.float16, device="cuda")
    for l in range(2):
        m.set_tensor(l, kvhp.LLAMA_ATTN_NORM, ones.cpu().numpy())
        m.set_tensor(l, kvhp.LLAMA_FFN_NORM, ones.cpu().numpy())
    ids = rng.permutation(vocab)[:n].astype(np.int32)
    p = (n + 15) // 16
    pool = torch.zeros((2, 2, heads, p, 16, d), dtype=torch.float16, device="cuda")
    m.prefill_paged(ids, pool, p, torch.arange(p, dtype=torch.int32, device="cuda"), p)
    m.close()

    x = torch.from_numpy(embed[ids]).cuda()
    xn = torch.empty_like(x)
    kvhp.rmsnorm(x, ones, xn, n, H, 1e-5)
    g = (xn[:, :1].float() * torch.from_numpy(alpha).cuda().float()).half()
    u = (xn[:, 1:2].float() * torch.from_numpy(beta).cuda().float()).half()
    act = torch.empty((n, F), dtype=torch.float16, device="cuda")
    kvhp.swiglu_rows(torch.cat([g, u], 1).contiguous(), act, n, F)
    act[:, :2] = x[:, :2]
    want = torch.empty_like(act)
    kvhp.rmsnorm(act, ones, want, n, H, 1e-5)
    torch.cuda.synchronize()
    assert float(g.min()) < -20 and float(g.max()) > 10 and bool(act.isfinite().all())
    got = pool[1, 1].reshape(heads, -1, d)[:, :n].transpose(0, 1).reshape(n, H)
    assert torch.equal(got, want), f"{int((got != want).sum())} of {got.numel()} differ"
