"""Device memory that a prompt behind a cached prefix takes beyond its model's: the
flash route with one split of the keys needs no attention partials, and no copy of
the block tables for each row.
"""
import numpy as np
import pytest

import kvhp
from gpu_util import note

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _grown(n, first, width):
    """Bytes by which free device memory falls over a first cached prompt (a
    whole prompt ran before it), with block tables of `width` pages."""
    v, hq, hkv, d = 512, 32, 4, 64
    m = kvhp.LlamaModel(kvhp.LlamaConfig(v, hq * d, 1, hq, hkv, d, 256, 1e-5, 10000.0, 0), 2, n)
    ids = np.random.default_rng(n).integers(0, v, n).astype(np.int32)
    pages = (n + 15) // 16
    pool = torch.zeros((1, 2, hkv, pages, 16, d), dtype=torch.float16, device="cuda")
    bt = torch.full((width,), -1, dtype=torch.int32, device="cuda")
    bt[:pages] = torch.arange(pages, device="cuda")
    _, whole = m.prefill_paged(ids, pool, pages, bt, width)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    _, got = m.prefill_cached(ids, first, pool, pages, bt, width)
    torch.cuda.synchronize()
    grown = free - torch.cuda.mem_get_info()[0]
    m.close()
    assert np.linalg.norm(got - whole) < 4e-3 * np.linalg.norm(whole)
    return grown


def test_one_split_takes_no_partials():
    """2048 rows over 4096 keys, one split: as decode rows their partials are
    4 x 2048 x 32 x 66 floats, 69 MB."""
    note("cached prompt: 2048 rows behind 2048 keys, memory")
    assert _grown(4096, 2048, 256) < 24 << 20


def test_no_tables_per_row():
    """2048 rows with tables of 4096 pages: a read and a write table a row are
    2 x 2048 x 4096 words, 67 MB."""
    note("cached prompt: 2048 rows with tables of 4096 pages, memory")
    assert _grown(4096, 2048, 4096) < 24 << 20
