"""The row-wise prompt operators' 16-byte kernels at their edges: the same call
on tensors shifted by one element (2-byte aligned) takes the element-wise
kernels, so each route is checked against the oracle and against the other.
RoPE and the embedding use the same arithmetic on both routes: equal bits.
SwiGLU's last product may be rounded to fp16 at once or through fp32, and
RMSNorm adds its squares in another order (fp32 sums of at most 16K terms,
far below the fp16 result's rounding): those agree within one fp16 step
(2^-10 relative).
"""
import numpy as np
import pytest

import kvhp
import oracle
from gpu_util import note, to_gpu

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _shifted(t):
    """A copy of t whose data starts 2 bytes past a 16-byte boundary."""
    buf = torch.empty(t.numel() + 8, dtype=t.dtype, device=t.device)
    v = buf[1:1 + t.numel()].view(t.shape)
    v.copy_(t)
    assert v.data_ptr() % 16 == 2
    return v


def _close(got, ref, what):
    got, ref = got.float().cpu().numpy(), np.asarray(ref, np.float32)
    err = np.abs(got - ref)
    bad = err > 1e-3 + 2e-3 * np.abs(ref)
    assert not bad.any(), f"{what}: {bad.sum()} of {bad.size} off, max abs {err.max():.3g}"


@pytest.mark.parametrize("rows,dim", [(1, 8), (5, 504), (3, 1024), (6, 1032), (4, 2048), (1, 2056),
                                      (3, 4096), (2, 4104), (3, 8192), (2, 8200), (1, 16384),
                                      (2, 16392), (9, 896)])
def test_rmsnorm_routes(rows, dim):
    note(f"rmsnorm {rows}x{dim}")
    rng = np.random.default_rng(rows * 31 + dim)
    x = oracle.normal_f16(rng, (rows, dim))
    w = oracle.normal_f16(rng, (dim,))
    ref = oracle.rmsnorm(x, w, 1e-5)
    xd, wd = to_gpu(x), to_gpu(w)
    out = torch.full((rows + 1, dim), 7.0, dtype=torch.float16, device="cuda")
    kvhp.rmsnorm(xd, wd, out, rows, dim, 1e-5)
    out2 = _shifted(torch.zeros_like(xd))
    kvhp.rmsnorm(_shifted(xd), wd, out2, rows, dim, 1e-5)
    kvhp.rmsnorm(xd, wd, xd, rows, dim, 1e-5)            # in place
    torch.cuda.synchronize()
    assert bool((out[rows] == 7.0).all())                # nothing past the rows
    _close(out[:rows], ref, "rmsnorm")
    assert torch.equal(out[:rows], xd)
    a, b = out[:rows].double(), out2.double()
    assert bool(((a - b).abs() <= 2.0 ** -10 * b.abs() + 2.0 ** -24).all())


@pytest.mark.parametrize("s,hq,hkv,d,start", [(1, 1, 1, 16, 0), (9, 3, 1, 16, 5), (5, 14, 2, 64, 0),
                                              (7, 32, 8, 128, 4000), (3, 4, 2, 256, 17),
                                              (3, 2, 1, 512, 3), (1, 64, 8, 96, 2), (6, 5, 1, 48, 1),
                                              (17, 40, 8, 80, 100)])
def test_split_qkv_rope_routes(s, hq, hkv, d, start):
    note(f"split_qkv_rope {s} tokens {hq}/{hkv}x{d}")
    rng = np.random.default_rng(s + d)
    qkv = oracle.normal_f16(rng, (s, hq + 2 * hkv, d))
    rq, rk = oracle.apply_rope(np.ascontiguousarray(qkv[:, :hq]),
                               np.ascontiguousarray(qkv[:, hq:hq + hkv]), hq, hkv, d, start,
                               10000.0)
    src = to_gpu(qkv)
    pos = torch.arange(start, start + s, dtype=torch.int32, device="cuda")
    new = lambda h: torch.empty((s, h, d), dtype=torch.float16, device="cuda")  # noqa: E731
    outs = []
    for data, positions in ((src, None), (_shifted(src), None), (src, pos)):
        q, k, v = new(hq), new(hkv), new(hkv)
        if positions is None:
            kvhp.split_qkv_rope(data, s, hq, hkv, d, start, 10000.0, q, k, v)
        else:
            kvhp.split_qkv_rope_rows(data, s, hq, hkv, d, positions, 10000.0, q, k, v)
        outs.append((q, k, v))
    torch.cuda.synchronize()
    _close(outs[0][0].reshape(-1), np.asarray(rq).reshape(-1), "q")
    _close(outs[0][1].reshape(-1), np.asarray(rk).reshape(-1), "k")
    assert np.array_equal(outs[0][2].cpu().numpy(), qkv[:, hq + hkv:])
    for other in outs[1:]:
        for a, b in zip(outs[0], other):
            assert torch.equal(a, b)


@pytest.mark.parametrize("rows,n", [(1, 8), (3, 2056), (33, 40), (2, 5632)])
def test_swiglu_routes(rows, n):
    rng = np.random.default_rng(rows + n)
    gu = oracle.normal_f16(rng, (rows, 2 * n), 3.0)
    gu[0, :4] = [np.inf, -np.inf, 60000.0, -60000.0]     # gates at the ends of the range
    d = to_gpu(gu)
    a = torch.empty((rows, n), dtype=torch.float16, device="cuda")
    b = _shifted(a)
    kvhp.swiglu_rows(d, a, rows, n)
    kvhp.swiglu_rows(_shifted(d), b, rows, n)
    flat = d[:, :n].contiguous()
    kvhp.swiglu(flat, d[:, n:].contiguous(), flat, rows * n)     # in place
    torch.cuda.synchronize()
    for o in (b, flat.view_as(a)):
        assert torch.equal(a.isnan(), o.isnan()) and torch.equal(a.isinf(), o.isinf())
        x, y = a.double().nan_to_num(0, 0, 0), o.double().nan_to_num(0, 0, 0)
        assert bool(((x - y).abs() <= 2.0 ** -10 * y.abs() + 2.0 ** -24).all())
    _close(a[:, 4:], oracle.swiglu(gu[:, 4:n], gu[:, n + 4:]), "swiglu")


@pytest.mark.parametrize("n,hidden", [(1, 8), (5, 896), (33, 40), (300, 2048)])
def test_embedding_routes(n, hidden):
    rng = np.random.default_rng(n + hidden)
    table = oracle.normal_f16(rng, (50, hidden), 0.02)
    ids = rng.integers(-2, 53, n).astype(np.int32)
    a = torch.empty((n, hidden), dtype=torch.float16, device="cuda")
    b = _shifted(a)
    kvhp.embedding(to_gpu(ids), to_gpu(table), a, n, hidden, 50)
    kvhp.embedding(to_gpu(ids), _shifted(to_gpu(table)), b, n, hidden, 50)
    torch.cuda.synchronize()
    exp = np.where(((ids >= 0) & (ids < 50))[:, None], table[np.clip(ids, 0, 49)],
                   np.float16(0))
    assert np.array_equal(a.cpu().numpy().view(np.uint16), exp.view(np.uint16))
    assert torch.equal(a.view(torch.int16), b.view(torch.int16))
