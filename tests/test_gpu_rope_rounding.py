"""The batched QKV projection rotates q and k with the bits of the separate
split + RoPE operator: each rotated value is rounded to fp16 once, from the fused
multiply-add.  Held in fp32 and rounded again it is another fp16 value about once
in 2^13.

The inputs make the projections exact in any order of the sums (x = +-1 without
an epsilon, so the norm's operand is +-w; one nonzero weight a row), so that the
rotation is all that could differ: equal bits are asserted.
"""
import numpy as np
import pytest

import kvhp
import oracle
from gpu_util import note, to_gpu

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("batch,hq,hkv,d,k", [(32, 32, 8, 128, 2048), (17, 32, 4, 64, 2048),
                                              (16, 16, 16, 64, 256)])
def test_batched_rotation_bits(batch, hq, hkv, d, k):
    note(f"rope rounding B={batch} {hq}/{hkv}x{d} K={k}")
    rng = np.random.default_rng(batch + k)
    n = (hq + 2 * hkv) * d
    val, col = oracle.normal_f16(rng, (n,)), rng.integers(0, k, n)
    W = np.zeros((n, k), np.float16)
    W[np.arange(n), col] = val
    x = rng.choice(np.array([-1, 1], np.float16), (batch, k))
    w = oracle.normal_f16(rng, (k,))
    proj = ((x * w)[:, col].astype(np.float32) * val.astype(np.float32)).astype(np.float16)
    pages = 256
    pos = rng.integers(0, 16 * pages, batch).astype(np.int32)
    # one page a sequence: every table entry names it
    tables = to_gpu(np.repeat(np.arange(batch, dtype=np.int32)[:, None], pages, 1))
    pool_k = torch.zeros((hkv, batch, 16, d), dtype=torch.float16, device="cuda")
    pool_v = torch.zeros_like(pool_k)
    q, posd = torch.empty((batch, hq, d), dtype=torch.float16, device="cuda"), to_gpu(pos)
    kvhp.rmsnorm_qkv_rope_append_rows(to_gpu(W), to_gpu(x), to_gpu(w), 0.0, posd, 10000.0, q,
                                      pool_k, pool_v, tables, hq, hkv, d, k, batch)
    rq, rk = torch.empty_like(q), torch.empty((batch, hkv, d), dtype=torch.float16, device="cuda")
    rv = torch.empty_like(rk)
    kvhp.split_qkv_rope_rows(to_gpu(proj), batch, hq, hkv, d, posd, 10000.0, rq, rk, rv)
    torch.cuda.synchronize()
    at = (torch.arange(batch, device="cuda"), posd.long() % 16)
    assert torch.equal(pool_v[:, at[0], at[1]].transpose(0, 1), rv)    # the projections agree
    assert torch.equal(q, rq)
    assert torch.equal(pool_k[:, at[0], at[1]].transpose(0, 1), rk)
