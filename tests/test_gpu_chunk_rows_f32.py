"""Prompt chunks on f32 pools (KVCache.attention_batch): row groups of 32 / G
tokens on the f32 MFMA, on the MI355X against float64 attention of the same
K / V: chunk lengths around a group, contexts of one and of several partitions,
chunks beside decodes, both mappings, head counts and sizes, bf16 queries,
strided and unaligned queries (the latter take the per-row decodes).  Tolerance
1e-5 absolute (f32), 2e-2 for bf16 outputs."""
import ctypes
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _ref(q, k, v, heads, hkv, mapping, start):
    t, _, d = q.shape
    g = heads // hkv
    out = torch.empty(q.shape, dtype=torch.float64)
    see = torch.arange(k.shape[0])[None] <= start + torch.arange(t)[:, None]
    for h in range(heads):
        kv = h // g if mapping == "grouped" else h % hkv
        w = (q[:, h].double() @ k[:, kv].double().T / math.sqrt(d)).masked_fill(~see, float("-inf"))
        out[:, h] = torch.softmax(w, 1) @ v[:, kv].double()
    return out


@pytest.mark.parametrize("H,Hkv,D,mapping,qdt", [(32, 8, 128, "grouped", torch.float32), (4, 4, 128, "grouped", torch.float32),
                                                 (4, 2, 64, "modulo", torch.float32), (16, 2, 64, "grouped", torch.float32),
                                                 (16, 2, 128, "modulo", torch.bfloat16)])
@pytest.mark.parametrize("layout", ["packed", "strided", "unaligned"])
def test_chunks_match_float64(H, Hkv, D, mapping, qdt, layout):
    from zealot_amd import BlockManager, KVCache
    nt = 32 * Hkv // H
    n = [1, nt - 1 or 2, nt, nt + 1, 3 * nt + 2, 1, 40, 2]
    before = [300, 0, 15, 16, 130, 0, 1000, 511]
    total = [a + b for a, b in zip(n, before)]
    bm = BlockManager(400, 16)
    cache = KVCache(400, 16, 2, Hkv, D, dtype=torch.float32, max_seqs=8, max_blocks_per_seq=80)
    g = torch.Generator().manual_seed(H + D)
    ids = [f"s{i}" for i in range(len(n))]
    kv = [(torch.randn(t, Hkv, D, generator=g), torch.randn(t, Hkv, D, generator=g)) for t in total]
    for sid, t in zip(ids, total):
        cache.register_seq(sid, 80)
        for _ in range(-(-t // 16)):
            cache.alloc_block(sid, bm)
    for part in (0, 1):  # the cached tokens, then the step's
        lens = before if part == 0 else n
        rows = [[x[:b] if part == 0 else x[b:] for x in p] for p, b in zip(kv, before)]
        k, v = (torch.cat([r[j] for r in rows]).cuda() for j in (0, 1))
        for layer in ((0, 1) if part == 0 else (0,)):
            cache.write_batch(layer, ids, lens, k, v)
    q = torch.randn(sum(n), H, D, generator=g).to(qdt)
    if layout == "packed":
        qd = q.cuda()
    else:  # rows inside a wider buffer, one element off for "unaligned"
        off = 1 if layout == "unaligned" else 4 * D
        buf = torch.zeros(sum(n), H * D + 8 * D, dtype=qdt, device="cuda")
        qd = buf[:, off:off + H * D].view(sum(n), H, D)
        qd.copy_(q)
    got = cache.attention_batch(0, ids, n, qd, mapping=mapping).cpu().double()
    row = 0
    for (k, v), t, b in zip(kv, n, before):
        want = _ref(q[row:row + t], k, v, H, Hkv, mapping, b)
        assert (got[row:row + t] - want).abs().max() <= (1e-5 if qdt == torch.float32 else 2e-2)
        row += t


def test_chunk_only_steps_refuse_what_decodes_refuse():
    """A step of chunks alone, as one with a decode beside them: a query type that
    is not f32 or bf16, an unknown head mapping."""
    from zealot_amd import BlockManager, KVCache, ZealotError, _lib
    from zealot_amd.kv_cache import SeqBatch
    H, Hkv, D, t = 8, 2, 128, 20
    bm = BlockManager(8, 16)
    cache = KVCache(8, 16, 1, Hkv, D, dtype=torch.float32, max_seqs=2, max_blocks_per_seq=4)
    cache.register_seq("s", 4)
    for _ in range(2):
        cache.alloc_block("s", bm)
    kv = torch.zeros((t, Hkv, D), device="cuda")
    cache.write_batch(0, ["s"], [t], kv, kv)
    out = torch.full((t, H, D), 7.0, device="cuda")
    q = torch.zeros((t, H, D), device="cuda")
    for dtype in (torch.uint8, torch.float8_e4m3fn):
        with pytest.raises(ZealotError, match="q dtype"):
            cache.attention_batch(0, ["s"], [t], torch.zeros((t, H, D), dtype=torch.uint8, device="cuda").view(dtype))
    b, n = SeqBatch(["s"]), (ctypes.c_int32 * 1)(t)
    for qdt, mapping, what in ((_lib.FP8_E4M3, _lib.GQA_GROUPED, "q dtype"), (7, _lib.GQA_GROUPED, "q dtype"), (_lib.F32, 7, "mapping")):
        rc = _lib.lib().zk_cache_attention_batch(cache._h, 0, b.arr, ctypes.addressof(n), 1, q.data_ptr(), qdt, 0, out.data_ptr(), H,
                                                 0.1, mapping)
        with pytest.raises(ZealotError, match=what):
            _lib.check(rc)
    torch.cuda.synchronize()
    assert bool((out == 7.0).all())  # nothing was launched


@pytest.mark.parametrize("H,Hkv,D", [(32, 8, 128), (4, 4, 64), (16, 2, 128)])
@pytest.mark.parametrize("before,t", [(0, 40), (13, 70), (600, 33)])
def test_rows_do_not_see_later_tokens_infinities(H, Hkv, D, before, t):
    """Infinities and NaN in K and V of a token reach the rows from that token
    on and no earlier one, also inside a row group and a page; every row against
    float64 attention of its own keys alone."""
    from zealot_amd import BlockManager, KVCache
    bm = BlockManager(60, 16)
    cache = KVCache(60, 16, 1, Hkv, D, dtype=torch.float32, max_seqs=1, max_blocks_per_seq=50)
    g = torch.Generator().manual_seed(H + before)
    n = before + t
    k, v, q = torch.randn(n, Hkv, D, generator=g), torch.randn(n, Hkv, D, generator=g), torch.randn(t, H, D, generator=g)
    v[before + 5, 0, 3] = float("inf")
    v[before + 6, 0, D - 1] = float("-inf")
    v[before + 18, 1, 0] = float("nan")
    v[before + t - 1, 1, 7] = float("inf")
    k[before + 21, 1, 2] = float("nan")
    cache.register_seq("s", 50)
    for _ in range(-(-n // 16)):
        cache.alloc_block("s", bm)
    for lo, hi in ((0, before), (before, n)):
        if hi > lo:
            cache.write_batch(0, ["s"], [hi - lo], k[lo:hi].cuda(), v[lo:hi].cuda())
    got = cache.attention_batch(0, ["s"], [t], q.cuda()).cpu().double()
    for i in range(t):
        want = _ref(q[i:i + 1], k[:before + i + 1], v[:before + i + 1], H, Hkv, "grouped", before + i)[0]
        fin = torch.isfinite(want)
        assert torch.equal(torch.isfinite(got[i]), fin), i
        assert (got[i][fin] - want[fin]).abs().max() <= 1e-5, i
        inf = torch.isinf(want)
        assert torch.equal(got[i][inf], want[inf]), i


def test_more_rows_than_one_grid_holds():
    """66000 rows of one chunk in several partitions: more than the 65535 that
    a launch of the merge takes; rows from all over the chunk against float64."""
    from zealot_amd import BlockManager, KVCache
    H, D, t = 1, 64, 66000
    pages = -(-t // 16)
    bm = BlockManager(pages, 16)
    cache = KVCache(pages, 16, 1, H, D, dtype=torch.float32, max_seqs=1, max_blocks_per_seq=pages)
    cache.register_seq("s", pages)
    for _ in range(pages):
        cache.alloc_block("s", bm)
    g = torch.Generator(device="cuda").manual_seed(5)
    k, v, q = (torch.randn((t, H, D), generator=g, device="cuda") for _ in range(3))
    cache.write_batch(0, ["s"], [t], k, v)
    got = cache.attention_batch(0, ["s"], [t], q)
    for i in (0, 31, 32, 16383, 16384, 40000, 65503, 65504, 65534, 65535, 65536, t - 1):
        w = torch.softmax(k[:i + 1, 0].double() @ q[i, 0].double() / math.sqrt(D), 0)
        assert (got[i, 0].double() - w @ v[:i + 1, 0].double()).abs().max() <= 1e-5, i


def test_rows_of_one_partition_take_no_partials():
    """8192 rows whose contexts are one partition each: no space for partials
    (a slot a row and head would be 140 MB)."""
    from zealot_amd import BlockManager, KVCache
    H, Hkv, D, t = 32, 8, 128, 8192
    bm = BlockManager(t // 16, 16)
    cache = KVCache(t // 16, 16, 1, Hkv, D, dtype=torch.float32, max_seqs=1, max_blocks_per_seq=t // 16)
    cache.register_seq("s", t // 16)
    for _ in range(t // 16):
        cache.alloc_block("s", bm)
    kv = torch.randn((t, Hkv, D), device="cuda")
    q = torch.randn((t, H, D), device="cuda")
    out = torch.empty_like(q)
    cache.write_batch(0, ["s"], [t], kv, kv)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    cache.attention_batch(0, ["s"], [t], q, out=out)
    torch.cuda.synchronize()
    assert free - torch.cuda.mem_get_info()[0] < 32 << 20
    for i in (0, 4095, t - 1):
        w = torch.softmax(kv[:i + 1, 0].double() @ q[i, 0].double() / math.sqrt(D), 0)
        assert (out[i, 0].double() - w @ kv[:i + 1, 0].double()).abs().max() <= 1e-5, i
