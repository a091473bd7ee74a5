"""Small decode launches run one wave per part of a partition
(attention_subs) and merge the parts' states; larger ones stream whole
partitions and fold the parts as they go. A query's bits must be the same
either way, at the edges of the parts (128 or 256 tokens, twice that past
8192), of the partitions and of a 16-token tile, through every entry point,
and within the attention tolerance of the oracle."""

from __future__ import annotations

import numpy as np
import pytest

from helpers import BLOCK, attention_close, fill_sequences, tables_and_lens

pytestmark = pytest.mark.gpu

SHORT = [1, 15, 16, 17, 64, 127, 128, 129, 257, 1024, 1025, 2048, 2049, 2177, 4096, 4097]
LONG = [8191, 8192, 8193, 8321, 16385]


@pytest.mark.parametrize("dtype,n_heads,n_kv,hd", [
    ("f16", 32, 8, 128),   # two kv heads a wave
    ("f16", 28, 4, 128),   # one kv head a wave, seven query heads
    ("f16", 32, 4, 64),
    ("f16", 9, 3, 64),
    ("q8_0", 32, 8, 128),  # partitions cut in two
    ("q8_0", 28, 4, 128),
    ("q8_0", 16, 4, 64),
])
@pytest.mark.parametrize("lens", [SHORT, LONG], ids=["short", "long"])
def test_parts_match_whole_partitions(gpu, dtype, n_heads, n_kv, hd, lens):
    import torch

    from langtrain_studio_amd import KvCache
    from oracle import OracleKv

    print(f"parts {dtype} {n_heads}/{n_kv}/{hd} {lens[-1]}", flush=True)
    rng = np.random.default_rng(n_heads * hd + len(lens))
    kvd = n_kv * hd
    blocks = sum(-(-n // BLOCK) for n in lens) + 4
    order = rng.permutation(blocks)
    g, o = KvCache(1, kvd, blocks * BLOCK, dtype=dtype, device=0), OracleKv(1, kvd, blocks * BLOCK, dtype=dtype)
    g.init_free_order(order)
    o.init_free_order(order)
    fill_sequences([("gpu", g), ("oracle", o)], dict(enumerate(lens)), rng, kvd)
    n = len(lens)
    q = rng.standard_normal((n, n_heads * hd), dtype=np.float32)
    tables, la = tables_and_lens(g, list(range(n)), lens)
    # 288 queries (every query 18 times or more) stream whole partitions
    pick = np.arange(288) % n
    dq, dt, dl = (torch.from_numpy(np.ascontiguousarray(x)).to(gpu) for x in (q, tables, la))
    whole = g.decode_attention(0, dq[pick].contiguous(), dt[pick].contiguous(), dl[pick].contiguous(), n_heads,
                               hd).cpu().numpy()[:n]
    for i in range(n):
        width = -(-lens[i] // BLOCK)
        args = (0, dq[i:i + 1].contiguous(), dt[i:i + 1, :width].contiguous(), dl[i:i + 1].contiguous(), n_heads, hd)
        for noalloc in (False, True):
            one = g.decode_attention(*args, noalloc=noalloc).cpu().numpy()
            np.testing.assert_array_equal(one[0].view(np.uint32), whole[i].view(np.uint32), err_msg=f"len {lens[i]}")
    # two queries of different lengths over the widest table (waves past the
    # short one's parts), by tables, resident rows and a plan
    pair = [0, n - 1]
    two = g.decode_attention(0, dq[pair].contiguous(), dt[pair].contiguous(), dl[pair].contiguous(), n_heads,
                             hd).cpu().numpy()
    rows = torch.from_numpy(g.seq_rows(pair).astype(np.int32)).to(gpu)
    by_rows = g.decode_attention_rows(0, dq[pair].contiguous(), rows, dl[pair].contiguous(), n_heads, hd).cpu().numpy()
    g.plan_attention(np.array(pair, np.uint32), np.array([lens[i] for i in pair], np.uint32), n_heads, hd)
    planned = g.planned_attention(0, dq[pair].contiguous()).cpu().numpy()
    for got in (two, by_rows, planned):
        np.testing.assert_array_equal(got.view(np.uint32), whole[pair].view(np.uint32))
    want = o.attention_tables(0, tables, la, q, n_heads, hd, threads=8)
    attention_close(whole, want, dtype)


def test_parts_under_capture_and_growth(gpu):
    """The states' memory is held from the cache's creation: a small launch is
    captured on a cache that has run nothing, and the graph's replays stay
    right after larger launches have replaced the workspace."""
    import torch

    from langtrain_studio_amd import KvCache

    rng = np.random.default_rng(3)
    lens = [700, 3000]
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        g = KvCache(1, 1024, 400 * BLOCK, dtype="f16", device=0, stream=stream)
        fill_sequences([("gpu", g)], dict(enumerate(lens)), rng, 1024)
        tables, la = tables_and_lens(g, [0, 1], lens)
        dt, dl = torch.from_numpy(tables).to(gpu), torch.from_numpy(la).to(gpu)
        q = torch.randn((2, 32 * 128), device=gpu)
        out = torch.zeros_like(q)
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            g.decode_attention(0, q, dt, dl, 32, 128, out=out)
        pick = np.arange(200) % 2
        for _ in range(3):
            q.normal_()
            graph.replay()
            got = out.clone()
            want = g.decode_attention(0, q[pick].contiguous(), dt[pick].contiguous(), dl[pick].contiguous(), 32, 128)
            stream.synchronize()
            assert torch.equal(got.view(torch.int32), want[:2].view(torch.int32))


# Fixed partitions whose launches end in the middle of a four-wave work-group
# (1, 2 or 3 waves past the last item; head groups of 1, 2 and 3).
@pytest.mark.parametrize("dtype,n_heads,n_kv,hd,part,n,longest", [
    ("f16", 8, 1, 128, 640, 41, 3200),     # 1025 waves
    ("f16", 9, 3, 64, 768, 23, 3200),      # 1035
    ("f16", 14, 2, 64, 576, 57, 1600),     # 1026
    ("f16", 24, 6, 128, 320, 23, 1600),    # 1035, two kv heads a wave
    ("q8_0", 8, 1, 128, 320, 69, 1600),    # 1035
    ("q8_0", 24, 6, 128, 1088, 13, 3200),  # 1170, partitions cut in two
])
def test_waves_past_the_last_part(gpu, dtype, n_heads, n_kv, hd, part, n, longest):
    """The append fused into the launch, the plain launch and a plan, against
    the same queries in a launch of whole partitions (bit-equal; query 0's
    states lie behind the last slot of the partials) and the pools of a cache
    that was written row by row."""
    import torch

    from langtrain_studio_amd import KvCache
    from oracle import OracleKv

    print(f"past the last part {dtype} {n_heads}/{n_kv}/{hd} {part} x {n}", flush=True)
    rng = np.random.default_rng(part + n)
    kvd = n_kv * hd
    lens = [longest] + [int(x) for x in rng.integers(1, longest + 1, n - 1)]
    blocks = sum(-(-x // BLOCK) for x in lens) + 4
    order = rng.permutation(blocks)
    g, o = KvCache(1, kvd, blocks * BLOCK, dtype=dtype, device=0), OracleKv(1, kvd, blocks * BLOCK, dtype=dtype)
    g.set_attention_partition(part)
    g.init_free_order(order)
    o.init_free_order(order)
    fill_sequences([("gpu", g), ("oracle", o)], {s: x - 1 for s, x in enumerate(lens)}, rng, kvd)
    seqs, pos = np.arange(n, dtype=np.uint32), np.array(lens, np.uint64) - 1
    sm = g.append_batch(seqs, pos)
    np.testing.assert_array_equal(sm, o.append_batch(seqs, pos))
    k, v = (rng.standard_normal((n, kvd), dtype=np.float32) for _ in range(2))
    q = rng.standard_normal((n, n_heads * hd), dtype=np.float32)
    tables, la = tables_and_lens(g, list(range(n)), lens)
    dsm, dk, dv, dq, dt, dl = (torch.from_numpy(np.ascontiguousarray(x)).to(gpu) for x in (sm, k, v, q, tables, la))
    fused = g.append_decode_attention(0, dsm, dk, dv, dq, dt, dl, n_heads, hd).cpu().numpy()
    o.write_batch(0, sm, k, v)
    for got, want in zip(g.read_pool(0), o.pool(0)):
        np.testing.assert_array_equal(got, want)
    pick = np.arange(n * 24) % n
    whole = g.decode_attention(0, dq[pick].contiguous(), dt[pick].contiguous(), dl[pick].contiguous(), n_heads,
                               hd).cpu().numpy()[:n]
    plain = g.decode_attention(0, dq, dt, dl, n_heads, hd).cpu().numpy()
    g.plan_attention(seqs, np.array(lens, np.uint32), n_heads, hd)
    planned = g.planned_attention(0, dq).cpu().numpy()
    for got in (fused, plain, planned):
        np.testing.assert_array_equal(got.view(np.uint32), whole.view(np.uint32))
    attention_close(whole, o.attention_tables(0, tables, la, q, n_heads, hd, threads=8), dtype)


def test_held_memory_follows_the_cache(gpu):
    """A cache of one block holds little more than its pools. Part states that
    its held memory is too small for (8 queries of 2000 tokens on one sequence:
    2 129 920 bytes, 2 048 000 held) go to the scratch, to a buffer allocated once,
    or, under capture on a cache that has none, nowhere: the launch runs whole
    partitions. All with the same bits."""
    import torch

    from langtrain_studio_amd import KvCache

    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info(gpu)[0]
    small = KvCache(1, 1024, BLOCK, dtype="f32", device=0)
    assert free - torch.cuda.mem_get_info(gpu)[0] < 16 << 20  # allocations come in steps of up to a few MiB
    del small

    rng = np.random.default_rng(12)
    n, length = 8, 2000
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        g = KvCache(1, 1024, length, dtype="f16", device=0, stream=stream)
        fill_sequences([("gpu", g)], {0: length}, rng, 1024)
        tables, la = tables_and_lens(g, [0] * n, [length] * n)
        dt, dl = torch.from_numpy(tables).to(gpu), torch.from_numpy(la).to(gpu)
        q = torch.randn((n, 32 * 128), device=gpu)
        out = torch.zeros_like(q)
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            g.decode_attention(0, q, dt, dl, 32, 128, out=out)
        pick = np.arange(200) % n
        whole = lambda: g.decode_attention(0, q[pick].contiguous(), dt[pick].contiguous(), dl[pick].contiguous(), 32,
                                           128)[:n]
        for _ in range(3):
            q.normal_()
            graph.replay()
            got = [out.clone(), g.decode_attention(0, q, dt, dl, 32, 128, noalloc=True),
                   g.decode_attention(0, q, dt, dl, 32, 128), g.decode_attention(0, q, dt, dl, 32, 128, noalloc=True)]
            want = whole()
            stream.synchronize()
            for x in got:
                assert torch.equal(x.view(torch.int32), want.view(torch.int32))
