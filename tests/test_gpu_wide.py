"""Decode attention on f16 pools of shapes outside head_dim 64 / 128 and
groups of up to 8 (attn_wide_kernel): against the oracle at the edges of a
tile (16 tokens), of the four waves' tiles (64), of the parts (a sixteenth of
a query up to 4096 tokens, 128 at least, 256 tokens up to 8192, 32 a query
beyond) and of the padded widths, alone and in a batch with the same bits; a
launch whose part states exceed 32 MiB streams whole contexts, with the same
bits; elements beyond f16 stay infinities, under any weight; Q of any
magnitude keeps f32 accuracy."""

from __future__ import annotations

import numpy as np
import pytest

from helpers import BLOCK, attention_close, fill_sequences, tables_and_lens

pytestmark = pytest.mark.gpu


def _pair(kvd, blocks, rng):
    from langtrain_studio_amd import KvCache
    from oracle import OracleKv

    order = rng.permutation(blocks)
    g, o = KvCache(1, kvd, blocks * BLOCK, dtype="f16", device=0), OracleKv(1, kvd, blocks * BLOCK, dtype="f16")
    g.init_free_order(order)
    o.init_free_order(order)
    return g, o


@pytest.mark.parametrize("n_heads,n_kv,hd", [
    (3, 3, 8), (8, 2, 16), (6, 2, 40), (17, 1, 64), (8, 2, 72), (20, 4, 80), (32, 8, 96), (32, 2, 96), (5, 1, 104),
    (16, 1, 128), (40, 1, 128), (8, 4, 160), (4, 1, 200), (8, 1, 256),
])
def test_wide_shapes(gpu, n_heads, n_kv, hd):
    import torch

    print(f"wide {n_heads}/{n_kv}/{hd}", flush=True)
    rng = np.random.default_rng(n_heads * 1000 + hd)
    lens = [1, 15, 16, 17, 63, 64, 65, 127, 128, 129, 255, 256, 2047, 2049, 4097, 8193]
    blocks = sum(-(-n // BLOCK) for n in lens) + 3
    kvd = n_kv * hd
    g, o = _pair(kvd, blocks, rng)
    fill_sequences([("gpu", g), ("oracle", o)], dict(enumerate(lens)), rng, kvd)
    n = len(lens)
    q = rng.standard_normal((n, n_heads * hd), dtype=np.float32)
    q[5] *= 1e6  # beyond the f16 range
    tables, la = tables_and_lens(g, list(range(n)), lens)
    dq, dt, dl = (torch.from_numpy(np.ascontiguousarray(x)).to(gpu) for x in (q, tables, la))
    full = g.decode_attention(0, dq, dt, dl, n_heads, hd).cpu().numpy()
    attention_close(full, o.attention_tables(0, tables, la, q, n_heads, hd, threads=8), "f16")
    for i in range(n):
        one = g.decode_attention(0, dq[i:i + 1].contiguous(), dt[i:i + 1, :-(-lens[i] // BLOCK)].contiguous(),
                                 dl[i:i + 1].contiguous(), n_heads, hd, noalloc=i % 2 == 0).cpu().numpy()
        np.testing.assert_array_equal(one[0].view(np.uint32), full[i].view(np.uint32), err_msg=f"len {lens[i]}")
    rows = torch.from_numpy(g.seq_rows(list(range(n))).astype(np.int32)).to(gpu)
    by_rows = g.decode_attention_rows(0, dq, rows, dl, n_heads, hd).cpu().numpy()
    np.testing.assert_array_equal(by_rows.view(np.uint32), full.view(np.uint32))
    # so many queries that their part states exceed the 32 MiB buffer
    reps = (32 << 20) // (n * n_heads * 32 * (hd + 2) * 4) + 1
    pick = np.arange(n * reps) % n
    many = g.decode_attention(0, dq[pick].contiguous(), dt[pick].contiguous(), dl[pick].contiguous(), n_heads, hd)
    want = torch.from_numpy(full).to(gpu)[torch.from_numpy(pick).to(gpu)]
    assert torch.equal(many.view(torch.int32), want.view(torch.int32))


def test_wide_infinities(gpu):
    """V beyond f16 stores as an infinity and stays one in its column; a key
    whose score is -infinity has no weight; the other heads are untouched."""
    import torch

    rng = np.random.default_rng(9)
    n_heads, n_kv, hd, n = 8, 2, 96, 70
    g, _ = _pair(n_kv * hd, 8, rng)
    sm = g.append_batch(np.zeros(n, np.uint32), np.arange(n, dtype=np.uint64))
    k, v = (rng.standard_normal((n, n_kv * hd)).astype(np.float32) for _ in range(2))
    q = rng.standard_normal((1, n_heads * hd)).astype(np.float32)
    q[0, :4 * hd] = np.abs(q[0, :4 * hd])
    v[11, 5] = 1e6       # kv head 0, column 5
    k[40, 7] = -1e6      # kv head 0: every score of token 40 is -inf
    g.write_batch(0, torch.from_numpy(sm).to(gpu), torch.from_numpy(k).to(gpu), torch.from_numpy(v).to(gpu))
    tables = torch.from_numpy(g.block_tables(np.zeros(1, np.uint32))).to(gpu)
    got = g.decode_attention(0, torch.from_numpy(q).to(gpu), tables, torch.tensor([n], dtype=torch.int32, device=gpu),
                             n_heads, hd).cpu().numpy().reshape(n_heads, hd)
    with np.errstate(over="ignore", invalid="ignore"):
        kh, vh = k.astype(np.float16).astype(np.float64), v.astype(np.float16).astype(np.float64)
        for h in range(n_heads):
            a = h // 4
            s = kh[:, a * hd:(a + 1) * hd] @ q[0, h * hd:(h + 1) * hd].astype(np.float64) / np.sqrt(hd)
            p = np.exp(s - s.max())
            want = (p / p.sum())[:, None] * vh[:, a * hd:(a + 1) * hd]
            want[p == 0] = 0
            want = want.sum(axis=0)
            assert np.isinf(got[h, 5]) == (a == 0) and np.isinf(want[5]) == (a == 0)
            fin = np.isfinite(want)
            np.testing.assert_allclose(got[h][fin], want[fin], rtol=0, atol=1e-5)


def _attend64(kh, vh, q, n_heads, n_kv, hd):
    """softmax(q k / sqrt(hd)) v over the stored rows, in 64 bits; tokens of
    weight zero are left out (an infinite V element there has no part)."""
    out = np.empty((n_heads, hd))
    with np.errstate(over="ignore", invalid="ignore"):
        for h in range(n_heads):
            a = h // (n_heads // n_kv)
            s = kh[:, a * hd:(a + 1) * hd] @ q[h * hd:(h + 1) * hd].astype(np.float64) / np.sqrt(hd)
            p = np.exp(s - s.max())
            live = p > 0
            out[h] = (p[live] / p.sum()) @ vh[live, a * hd:(a + 1) * hd]
    return out


@pytest.mark.parametrize("n_heads,n_kv,hd", [(8, 2, 96), (16, 1, 128), (5, 1, 40)])
@pytest.mark.parametrize("q_scale,k_scale", [(1e-4, 1e3), (1e-7, 3e4), (1.0, 1.0), (3e3, 1e-3), (1e-30, 3e4)])
def test_wide_magnitudes(gpu, n_heads, n_kv, hd, q_scale, k_scale):
    """Q of any magnitude keeps f32 accuracy. With sigma = q_scale * k_scale the
    sums of |q k| / sqrt(hd) are about 0.64 sqrt(hd) sigma, so f32 scores are
    good to (hd + 2) 2^-24 times that and the weighted sums to 2 n 2^-24 in the
    worst case: 1.3e-4 for the largest of these (sigma 3), of which rounding
    errors of random sign leave a fiftieth. 3e-6 is asked for."""
    import torch

    rng = np.random.default_rng(hd)
    n, kvd = 700, n_kv * hd
    g, _ = _pair(kvd, 48, rng)
    sm = g.append_batch(np.zeros(n, np.uint32), np.arange(n, dtype=np.uint64))
    k = rng.standard_normal((n, kvd)).astype(np.float32) * np.float32(k_scale)
    k = np.clip(k, -65504, 65504)
    v = rng.standard_normal((n, kvd)).astype(np.float32)
    q = rng.standard_normal((1, n_heads * hd)).astype(np.float32) * np.float32(q_scale)
    g.write_batch(0, *(torch.from_numpy(x).to(gpu) for x in (sm, k, v)))
    tables = torch.from_numpy(g.block_tables(np.zeros(1, np.uint32))).to(gpu)
    got = g.decode_attention(0, torch.from_numpy(q).to(gpu), tables, torch.tensor([n], dtype=torch.int32, device=gpu),
                             n_heads, hd).cpu().numpy().reshape(n_heads, hd).astype(np.float64)
    want = _attend64(k.astype(np.float16).astype(np.float64), v.astype(np.float16).astype(np.float64), q[0], n_heads,
                     n_kv, hd)
    rel = np.linalg.norm(got - want) / np.linalg.norm(want)
    print(f"wide magnitudes {n_heads}/{n_kv}/{hd} {q_scale} {k_scale}: {rel:.2e}", flush=True)
    assert rel <= 3e-6


@pytest.mark.parametrize("bits", [20, 30, 60, 100])
def test_wide_infinities_under_small_factors(gpu, bits):
    """An infinite V element under a weight of 2^-bits of the largest is an
    infinity in the result; an infinite K element times a Q element 2^-bits of
    the head's largest decides the score's sign (here: no weight)."""
    import torch

    rng = np.random.default_rng(bits)
    n_heads, n_kv, hd, n = 8, 2, 96, 70
    g, _ = _pair(n_kv * hd, 8, rng)
    sm = g.append_batch(np.zeros(n, np.uint32), np.arange(n, dtype=np.uint64))
    k, v = (rng.standard_normal((n, n_kv * hd)).astype(np.float32) * 0.1 for _ in range(2))
    q = rng.standard_normal((1, n_heads * hd)).astype(np.float32) * 0.1
    for h in range(n_heads):
        q[0, h * hd] = 8.0
        q[0, h * hd + 7] = 2.0 ** (3 - bits)
    k[:, [0, hd]] = 0.0
    k[:, [7, hd + 7]] = 1.0
    k[11, [0, hd]] = np.float32(-bits * np.log(2.0) * np.sqrt(hd) / 8.0)  # weight 2^-bits, about
    v[11, 5] = 1e6        # kv head 0, column 5
    k[40, hd + 7] = -1e6  # kv head 1: every score of token 40 is -inf
    g.write_batch(0, *(torch.from_numpy(x).to(gpu) for x in (sm, k, v)))
    tables = torch.from_numpy(g.block_tables(np.zeros(1, np.uint32))).to(gpu)
    got = g.decode_attention(0, torch.from_numpy(q).to(gpu), tables, torch.tensor([n], dtype=torch.int32, device=gpu),
                             n_heads, hd).cpu().numpy().reshape(n_heads, hd).astype(np.float64)
    with np.errstate(over="ignore"):
        want = _attend64(k.astype(np.float16).astype(np.float64), v.astype(np.float16).astype(np.float64), q[0],
                         n_heads, n_kv, hd)
    assert np.isposinf(want[:4, 5]).all() and np.isinf(want).sum() == 4
    np.testing.assert_array_equal(np.isposinf(got), np.isposinf(want))
    fin = np.isfinite(want)
    np.testing.assert_allclose(got[fin], want[fin], rtol=0, atol=1e-5)


def test_wide_nonfinite_queries(gpu):
    """A NaN or infinite Q element makes its own head NaN (infinite scores of
    both signs) and leaves the bits of the others."""
    import torch

    rng = np.random.default_rng(17)
    n_heads, n_kv, hd, n = 8, 2, 96, 130
    g, _ = _pair(n_kv * hd, 10, rng)
    sm = g.append_batch(np.zeros(n, np.uint32), np.arange(n, dtype=np.uint64))
    k, v = (rng.standard_normal((n, n_kv * hd)).astype(np.float32) for _ in range(2))
    q = rng.standard_normal((2, n_heads * hd)).astype(np.float32)
    q[1] = q[0]
    q[1, 2 * hd + 3] = np.nan
    q[1, 5 * hd + 90] = -np.inf
    g.write_batch(0, *(torch.from_numpy(x).to(gpu) for x in (sm, k, v)))
    tables = torch.from_numpy(g.block_tables(np.zeros(2, np.uint32))).to(gpu)
    got = g.decode_attention(0, torch.from_numpy(q).to(gpu), tables,
                             torch.tensor([n, n], dtype=torch.int32, device=gpu), n_heads, hd).cpu().numpy()
    got = got.reshape(2, n_heads, hd)
    bad = np.isin(np.arange(n_heads), [2, 5])
    assert np.isfinite(got[0]).all() and np.isnan(got[1, bad]).all()
    np.testing.assert_array_equal(got[1, ~bad].view(np.uint32), got[0, ~bad].view(np.uint32))
