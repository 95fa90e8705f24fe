"""Planless chunked prefill (small batches; items split over their keys) on the
MI355X against the oracle's or_paged_prefill: chunks behind contexts that several
splits share, chunk ends at tile edges, more sequences than a wave looks up at
once, tables cut in every split, and one batch large enough for the planned
launch with the same cuts.  Tolerance 2e-2 absolute, as tests/test_gpu_prefill.py."""
import math

import numpy as np
import pytest
import torch

import oracle
from tests.gpu_util import as_f32, max_abs_err, to_dev, to_host
from tests.test_gpu_prefill import _case, _run

pytestmark = pytest.mark.gpu


def _check(H, Hkv, D, starts, chunks, kv="bf16", causal=True, mapping="grouped", cuts=None, seed=300):
    q, kp, vp, kvdt, bt, cu, ks, vs = _case(seed, H, Hkv, D, starts, chunks, kv)
    bt = bt.copy()
    for n, page in (cuts or {}).items():
        bt[n, page] = -1
    out = _run(q, kp, vp, bt, cu, starts, causal, mapping, ks, vs)
    ref = oracle.paged_prefill(as_f32(q, oracle.BF16), kp, vp, kvdt, bt, cu, starts, Hkv, D, 16, np.float32(1 / math.sqrt(D)), causal,
                               oracle.GROUPED if mapping == "grouped" else oracle.MODULO, ks, vs)
    assert max_abs_err(as_f32(out, oracle.BF16), ref) <= 2e-2


@pytest.mark.parametrize("H,Hkv,D,kv,causal", [(8, 2, 128, "bf16", True), (8, 2, 128, "bf16", False), (2, 2, 128, "bf16", True),
                                               (16, 2, 64, "bf16", True), (4, 2, 64, "fp8", True), (8, 2, 128, "fp8", False)])
def test_split_contexts(H, Hkv, D, kv, causal):
    for starts, chunks in (([1500], [33]), ([1039, 0], [1, 130]), ([700, 15, 0], [128, 129, 64])):
        _check(H, Hkv, D, starts, chunks, kv, causal, "modulo" if H == 16 else "grouped", seed=300 + len(starts))


def test_many_short_chunks():
    rng = np.random.default_rng(5)
    _check(8, 2, 128, [int(x) for x in rng.integers(0, 40, 70)], [int(x) for x in rng.integers(0, 20, 69)] + [3])


@pytest.mark.parametrize("kv", ["bf16", "fp8"])
def test_cut_in_every_split(kv):
    n, pages = 6, 60
    starts, chunks = [16 * pages - 40] * n, [35] * n
    _check(8, 2, 128, starts, chunks, kv, cuts=dict(zip(range(n), (0, 1, 10, 31, 45, pages - 1))))


def test_planned_launch_with_cuts():
    rng = np.random.default_rng(6)
    chunks = [int(x) for x in rng.integers(30, 90, 60)]
    starts = [int(x) for x in rng.integers(0, 100, 60)]
    _check(32, 32, 64, starts, chunks, cuts={3: 0, 10: 1, 33: 2})


@pytest.mark.parametrize("start,chunk,best", [(0, 40, 11), (1500, 33, 3), (1500, 33, 1100), (1500, 33, 1510), (2000, 33, None)])
def test_scores_far_below_zero(start, chunk, best):
    """Scores of some -1e31 (powers of two, so that scaling them is exact) have the
    weights their differences give, with one split and with several: key `best`
    alone, or all the same."""
    H, Hkv, D = 8, 2, 128
    q, kp, vp, _, bt, cu, _, _ = _case(340, H, Hkv, D, [start], [chunk], "bf16")
    bits = oracle.bf16_bits_from_f32
    q[:, :, 0] = bits(np.full((1,), 2.0**40, np.float32))[0]
    kp[:, :, :, 0] = bits(np.full((1,), -2.0**67, np.float32))[0]
    if best is not None:
        kp[bt[0, best // 16], :, best % 16, 0] = bits(np.full((1,), -2.0**66, np.float32))[0]
    out = as_f32(_run(q, kp, vp, bt, cu, [start], True, "grouped", None, None), oracle.BF16)
    t = np.arange(start + chunk)
    v = as_f32(vp, oracle.BF16)[bt[0, t // 16], :, t % 16]  # [tokens, Hkv, D]
    for i in range(chunk):
        seen = start + i + 1
        want = v[best] if best is not None and best < seen else v[:seen].mean(0, dtype=np.float64)
        assert max_abs_err(out[i].reshape(Hkv, H // Hkv, D), want[:, None]) <= 2e-2, i


def test_cache_keeps_its_prefill_workspace():
    """Steps of any chunks run in the workspace of the cache's first one: a
    small batch may need more space than a large one."""
    from zealot_amd import BlockManager, KVCache
    H, Hkv, D = 32, 8, 128
    bm = BlockManager(1200, 16)
    cache = KVCache(1200, 16, 1, Hkv, D, dtype=torch.bfloat16, max_seqs=60, max_blocks_per_seq=20)
    ids = [f"s{i}" for i in range(60)]
    for sid in ids:
        cache.register_seq(sid, 20)
        for _ in range(20):
            cache.alloc_block(sid, bm)
    x = torch.randn((60 * 100, Hkv, D), device="cuda").bfloat16()
    q = torch.randn((60 * 100, H, D), device="cuda").bfloat16()
    out = torch.empty_like(q)
    free = []
    for n, chunk in ((1, 20), (30, 2), (60, 100), (3, 40), (12, 9), (60, 2)):
        rows = n * chunk
        cache.write_batch(0, ids[:n], [chunk] * n, x[:rows], x[:rows])
        cache.attention_batch(0, ids[:n], [chunk] * n, q[:rows], out=out[:rows])
        torch.cuda.synchronize()
        free.append(torch.cuda.mem_get_info()[0])
    assert free[0] - min(free) < 8 << 20, [free[0] - f for f in free]


def test_workspace_without_partials():
    """A workspace that holds the plan and no partials: the same rows, unsplit."""
    from zealot_amd import ops
    H, Hkv, D, starts, chunks = 8, 2, 128, [1500, 40], [33, 5]
    q, kp, vp, kvdt, bt, cu, _, _ = _case(350, H, Hkv, D, starts, chunks)
    plan = 256 + 2048 + -(-16 * (-(-sum(chunks) // 32) + len(chunks)) * Hkv // 256) * 256
    assert ops.prefill_workspace_bytes(len(chunks), sum(chunks), H, Hkv) > plan
    args = [to_dev(x) for x in (q, kp, vp, bt, cu, np.asarray(starts, np.int32))]
    out = ops.paged_prefill(*args, workspace=torch.empty(plan, dtype=torch.uint8, device="cuda"))
    ref = oracle.paged_prefill(as_f32(q, oracle.BF16), kp, vp, kvdt, bt, cu, starts, Hkv, D, 16, np.float32(1 / math.sqrt(D)))
    assert max_abs_err(as_f32(to_host(out), oracle.BF16), ref) <= 2e-2
    with pytest.raises(RuntimeError, match="workspace"):
        ops.paged_prefill(*args, workspace=torch.empty(plan - 256, dtype=torch.uint8, device="cuda"))
