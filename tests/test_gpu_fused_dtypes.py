"""The fused append on f32 and q8_0 pools: the decode kernels write the new
row of the query's last partition (or part) before they read it. Pools,
scales and outputs equal ltkv_write then ltkv_decode_attention bit for bit,
at the edges of blocks, parts and partitions, in small launches (a wave per
part) and large ones, with skipped cells and cells outside the pool."""

from __future__ import annotations

import numpy as np
import pytest

from helpers import BLOCK, fill_sequences

pytestmark = pytest.mark.gpu

CTX = [0, 15, 16, 17, 63, 127, 128, 300, 1023, 1024, 2047, 4100]


@pytest.mark.parametrize("dtype,n_heads,n_kv,hd", [
    ("f32", 32, 4, 64), ("f32", 9, 3, 64), ("f32", 32, 8, 128), ("f32", 7, 1, 128),
    ("q8_0", 32, 8, 128), ("q8_0", 28, 4, 128), ("q8_0", 16, 4, 64), ("q8_0", 9, 3, 64),
])
@pytest.mark.parametrize("copies", [1, 12], ids=["small", "large"])
def test_fused_append(gpu, dtype, n_heads, n_kv, hd, copies):
    import torch

    from langtrain_studio_amd import KvCache

    ctx = CTX * copies
    print(f"fused {dtype} {n_heads}/{n_kv}/{hd} x{copies}", flush=True)
    rng = np.random.default_rng(n_heads + hd + copies)
    kvd, n = n_kv * hd, len(ctx)
    blocks = sum(-(-(c + 1) // BLOCK) for c in ctx) + 3
    order = rng.permutation(blocks)
    a, b = (KvCache(1, kvd, blocks * BLOCK, dtype=dtype, device=0) for _ in range(2))
    for c in (a, b):
        c.init_free_order(order)
    fill_sequences([("gpu", a), ("gpu", b)], dict(enumerate(ctx)), rng, kvd)
    seqs, pos = np.arange(n, dtype=np.uint32), np.array(ctx, dtype=np.uint64)
    sm = a.append_batch(seqs, pos).copy()
    np.testing.assert_array_equal(b.append_batch(seqs, pos), sm)
    sm[4], sm[8] = -1, blocks * BLOCK  # skipped; outside the pool
    k, v = (torch.from_numpy(rng.standard_normal((n, kvd), dtype=np.float32)).to(gpu) for _ in range(2))
    k[2, :32] = 0.0  # an all-zero group
    q = torch.from_numpy(rng.standard_normal((n, n_heads * hd), dtype=np.float32)).to(gpu)
    dsm, lens = torch.from_numpy(sm).to(gpu), torch.from_numpy(np.array(ctx, np.int32) + 1).to(gpu)
    tables = torch.from_numpy(a.block_tables(seqs)).to(gpu)
    a.write_batch(0, dsm, k, v)
    two = a.decode_attention(0, q, tables, lens, n_heads, hd)
    one = b.append_decode_attention(0, dsm, k, v, q, tables, lens, n_heads, hd)
    assert torch.equal(one.view(torch.int32), two.view(torch.int32))
    for pa, pb in zip(a.read_pool(0), b.read_pool(0)):
        np.testing.assert_array_equal(pa, pb)
    if dtype == "q8_0":
        for pa, pb in zip(a.read_scales(0), b.read_scales(0)):
            np.testing.assert_array_equal(pa, pb)
