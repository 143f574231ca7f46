"""The batch-1 GEMVs at every way a wave covers K: whole rows of K % 8 == 0 in
registers (up to 4096 columns), slabs of 4096 columns beyond, and the
element-wise kernel for other K or unaligned weights.  Reference: the same
product in 64 bits over the RMSNorm output rounded to fp16, as the kernels
round it.  Tolerance 1e-3 + 2e-3 |r|: the fp16 result's rounding (2^-11 |r|), an
RMSNorm operand one fp16 step apart in a few columns (2^-10 * 0.02 each), and
fp32 sums of at most 12K products of size 0.1 (below 1e-4).
"""
import numpy as np
import pytest

import kvhp
import oracle
from gpu_util import note, to_gpu

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

EPS = 1e-5
KS = [8, 504, 512, 896, 1024, 1032, 2040, 2056, 4088, 4096, 4104, 4864, 5640, 8192, 8200, 11264,
      12296, 1001]


def _close(got, ref, what):
    got, ref = got.double().cpu(), torch.as_tensor(ref).double().cpu()
    bad = (got - ref).abs() > 1e-3 + 2e-3 * ref.abs()
    assert not bool(bad.any()), f"{what}: {int(bad.sum())} of {bad.numel()} off, " \
                                f"max {float((got - ref).abs().max()):.3g}"


def _norm16(x, w):
    x64 = x.double()
    rs = 1.0 / torch.sqrt(x64.square().mean() + EPS)
    return (x64 * rs * w.double()).half().double()


def _inputs(n, k, seed):
    rng = np.random.default_rng(seed)
    W = to_gpu(oracle.normal_f16(rng, (n, k), 0.02))
    x = to_gpu(oracle.normal_f16(rng, (k,)))
    nw = to_gpu(oracle.normal_f16(rng, (k,), 0.3)) + 1.0
    return W, x, nw


def _unaligned(t):
    buf = torch.empty(t.numel() + 8, dtype=t.dtype, device=t.device)
    v = buf[1:1 + t.numel()].view(t.shape)
    v.copy_(t)
    return v


@pytest.mark.parametrize("k", KS)
def test_gemv_covers(k):
    n = 37
    note(f"gemv covers {n}x{k}")
    W, x, nw = _inputs(n, k, k)
    r = x.new_tensor(np.linspace(-2, 2, n))
    y = torch.full((n + 1,), 9.0, dtype=torch.float16, device="cuda")
    y32 = torch.empty(n, dtype=torch.float32, device="cuda")
    y16 = torch.empty(n, dtype=torch.float16, device="cuda")
    plain = W.double() @ x.double()
    kvhp.gemv(W, x, y, n, k)
    torch.cuda.synchronize()
    assert float(y[n]) == 9.0
    _close(y[:n], plain, "gemv")
    kvhp.gemv_residual(_unaligned(W), x, r, y16, n, k)
    _close(y16, plain + r.double(), "gemv_residual, unaligned weights")
    kvhp.gemv_residual(W, x, r, r, n, k)                   # in place
    _close(r, plain + torch.linspace(-2, 2, n, dtype=torch.float64, device="cuda").half(),
           "gemv_residual")
    normed = W.double() @ _norm16(x, nw)
    kvhp.rmsnorm_gemv(W, x, nw, EPS, n, k, y32=y32)
    kvhp.rmsnorm_gemv(W, x, nw, EPS, n, k, y16=y16)
    torch.cuda.synchronize()
    _close(y32, normed, "rmsnorm_gemv fp32")
    _close(y16, normed, "rmsnorm_gemv fp16")


@pytest.mark.parametrize("k", [8, 896, 1024, 2040, 4096, 4104, 8200, 1001])
def test_swiglu_and_qkv_covers(k):
    note(f"swiglu and qkv covers K={k}")
    n = 13
    W, x, nw = _inputs(2 * n, k, k + 1)
    xn = _norm16(x, nw)
    gu = (W.double() @ xn).half().double()
    out = torch.empty(n, dtype=torch.float16, device="cuda")
    kvhp.rmsnorm_gemv_swiglu(W, x, nw, EPS, out, n, k)
    g, u = gu[:n], gu[n:]
    _close(out, g * torch.sigmoid(g) * u, "swiglu")

    hq, hkv, d, pos = 6, 2, 16, 21
    W, x, nw = _inputs((hq + 2 * hkv) * d, k, k + 2)
    pool_k = torch.zeros((hkv, 3, 16, d), dtype=torch.float16, device="cuda")
    pool_v = torch.zeros_like(pool_k)
    q = torch.empty((hq, d), dtype=torch.float16, device="cuda")
    bt = torch.tensor([0, 2, 1], dtype=torch.int32, device="cuda")
    ln = torch.tensor([pos + 1], dtype=torch.int32, device="cuda")
    kvhp.rmsnorm_qkv_rope_append(W, x, nw, EPS, ln, 10000.0, q, pool_k, pool_v, bt, hq, hkv, d, k)
    torch.cuda.synchronize()
    y = (W.double() @ _norm16(x, nw)).half().view(hq + 2 * hkv, d).cpu().numpy()
    rq, rk = oracle.apply_rope(np.ascontiguousarray(y[None, :hq]),
                               np.ascontiguousarray(y[None, hq:hq + hkv]), hq, hkv, d, pos, 10000.0)
    _close(q.reshape(-1), np.asarray(rq).reshape(-1), "q")
    _close(pool_k[:, 2, pos % 16].reshape(-1), np.asarray(rk).reshape(-1), "k")
    _close(pool_v[:, 2, pos % 16].reshape(-1), y[hq + hkv:].reshape(-1), "v")
    pool_k[:, 2, pos % 16] = 0
    assert not bool(pool_k.any())                          # nothing else written
