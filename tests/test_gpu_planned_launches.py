"""Which launch a paged decode takes and the planned ones at small sizes, on the
MI355X.  Batches over the line run the planned launch, whose plan the layers of a
step share; most others run without a plan, so the decode suites run once more in
a process where every decode is planned (ZEALOT_DECODE_PART_PAGES).  Prefills of
both launches at sizes the other tests leave out.  Tolerances
(absolute): 1e-5 f32, 2e-2 bf16, as tests/test_gpu_decode.py."""
import ctypes
import math
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

import oracle
from tests.gpu_util import as_f32, decode_case, max_abs_err, normal, to_dev, to_host
from tests.test_gpu_decode import TOL, _oracle
from tests.test_gpu_prefill import _case, _run

pytestmark = pytest.mark.gpu

PLANNED = "ZEALOT_DECODE_PART_PAGES" in os.environ


def _plans(fn, name=b"decode_plan") -> int:
    """Plan launches while fn runs."""
    from zealot_amd import _lib
    L, n, ms = _lib.lib(), ctypes.c_int64(), ctypes.c_double()
    L.zk_timing_reset()
    L.zk_timing_enable(1)
    fn()
    torch.cuda.synchronize()
    L.zk_timing_enable(0)
    _lib.check(L.zk_timing_query(name, ctypes.byref(n), ctypes.byref(ms)))
    L.zk_timing_reset()
    return n.value


@pytest.mark.skipif(PLANNED, reason="every decode is planned")
@pytest.mark.parametrize("layers,dtype,first,want", [(4, torch.bfloat16, 4200, 1), (4, torch.bfloat16, 3000, 0),
                                                     (1, torch.bfloat16, 4200, 0), (1, torch.bfloat16, 8000, 1),
                                                     (4, torch.float32, 1300, 1), (4, torch.float32, 1000, 0)])
def test_layers_share_a_plan(layers, dtype, first, want):
    """One long sequence beside 99 short ones: the tables' capacity (100 x the
    longest, 16-token pages of 8 kv-heads of 128) decides, and the layers count.
    Three steps, the second over the first's lengths; every layer against float64."""
    from zealot_amd import BlockManager, KVCache
    H, Hkv, D, n = 32, 8, 128, 100
    lens = [first] + [5 + i % 40 for i in range(n - 1)]
    pages = [(t + 4) // 16 + 1 for t in lens]
    bm = BlockManager(sum(pages), 16)
    cache = KVCache(sum(pages), 16, layers, Hkv, D, dtype=dtype, max_seqs=n, max_blocks_per_seq=max(pages))
    ids = [f"s{i}" for i in range(n)]
    for sid, p in zip(ids, pages):
        cache.register_seq(sid, p)
        for _ in range(p):
            cache.alloc_block(sid, bm)
    g = torch.Generator(device="cuda").manual_seed(first)

    def rand(*shape):
        return torch.randn(shape, generator=g, device="cuda").to(dtype)

    kv = []  # per layer: K and V of all sequences, packed
    for layer in range(layers):
        kv.append([[rand(t, Hkv, D) for t in lens] for _ in range(2)])
        cache.write_batch(layer, ids, lens, torch.cat(kv[-1][0]), torch.cat(kv[-1][1]))
    outs = []
    for step in range(3):
        if step == 2:  # one more token a sequence: another plan
            for layer in range(layers):
                new = [rand(n, Hkv, D) for _ in range(2)]
                cache.append_kv_batch(layer, ids, *new)
                kv[layer] = [[torch.cat([x, y[i:i + 1]]) for i, x in enumerate(old)] for old, y in zip(kv[layer], new)]
        qs = [rand(n, H, D) for _ in range(layers)]
        plans = _plans(lambda: outs.extend(cache.paged_decode(layer, ids, q) for layer, q in enumerate(qs)))
        assert plans == (0 if step == 1 else want), (step, plans)
        for layer, q in enumerate(qs):
            out = outs[step * layers + layer].double()
            for i in (0, 1, 40, 99):
                k, v = (x[i].double().repeat_interleave(H // Hkv, 1) for x in kv[layer])
                w = torch.softmax(torch.einsum("hd,thd->ht", q[i].double(), k) / D ** 0.5, 1)
                want_out = torch.einsum("ht,thd->hd", w, v)
                assert (out[i] - want_out).abs().max() <= (1e-5 if dtype == torch.float32 else 2e-2), (step, layer, i)


@pytest.mark.parametrize("dt", [oracle.F32, oracle.BF16])
@pytest.mark.parametrize("H,Hkv,D", [(32, 8, 128), (8, 8, 64)])
def test_wide_tables_are_planned(dt, H, Hkv, D):
    """A table wide enough for the planned launch over a small pool, with cuts."""
    from zealot_amd import ops
    lens = [0, 16 * 100 + 3, 700, 700, 40, 900, 1, 255]
    q, kp, vp, bt, nb = decode_case(1200 + D, H, Hkv, D, lens, dt)
    page = 2 * Hkv * 16 * D * (4 if dt == oracle.F32 else 2)
    wide = -np.ones((len(lens), int(3.1e9 / page / len(lens))), np.int32)
    wide[:, :bt.shape[1]] = bt
    wide[2, 7], wide[3, 33] = -1, nb
    ref = [*lens[:2], 7 * 16, 33 * 16, *lens[4:]]
    out = []
    args = [to_dev(x) for x in (q, kp, vp, wide, np.asarray(lens, np.int32))]
    assert _plans(lambda: out.append(ops.paged_decode(*args))) == 1
    got = as_f32(to_host(out[0]), dt)
    assert np.all(got[0] == 0)
    assert max_abs_err(got, _oracle(q, kp, vp, bt, ref, dt, dt, "grouped")) <= TOL[dt]


@pytest.mark.skipif(PLANNED, reason="every decode is planned")
@pytest.mark.parametrize("dt", [oracle.F32, oracle.BF16])
def test_longest_partitions_without_a_plan(dt):
    """Tables of 64 pages in one partition each (a table entry a lane): full,
    nearly full, cut at the last entries; sequences share the pool's blocks."""
    from zealot_amd import ops
    H, Hkv, D, mb, nb = 16, 8, 128, 64, 300
    n = 640 if dt == oracle.BF16 else 320  # 2.7 GB of capacity
    rng = np.random.default_rng(41)
    lens = rng.integers(1, 1025, n)
    lens[:6] = 1024, 1023, 1009, 1008, 1024, 1024
    kp, vp = (normal(rng, (nb, Hkv, 16, D), dt) for _ in range(2))
    q = normal(rng, (n, H, D), dt)
    bt = rng.integers(0, nb, (n, mb)).astype(np.int32)
    bt[4, 63], bt[5, 62] = -1, 1 << 20
    ref = lens.copy()
    ref[4], ref[5] = 1008, 992
    out = []
    args = [to_dev(x) for x in (q, kp, vp, bt, lens.astype(np.int32))]
    assert _plans(lambda: out.append(ops.paged_decode(*args))) == 0
    got, some = as_f32(to_host(out[0]), dt), np.r_[:12, n - 8:n]
    want = _oracle(q[some], kp, vp, np.maximum(bt[some], 0) % nb, [int(x) for x in ref[some]], dt, dt, "grouped")
    assert max_abs_err(got[some], want) <= TOL[dt]


@pytest.mark.parametrize("H,Hkv,D,kv,causal,mapping", [(8, 8, 64, "fp8", True, "grouped"), (16, 8, 128, "bf16", False, "modulo"),
                                                       (32, 8, 64, "bf16", True, "modulo"), (64, 8, 128, "fp8", False, "grouped")])
def test_planned_prefill_of_short_chunks(H, Hkv, D, kv, causal, mapping):
    """Many short chunks in wide tables, two of them cut, take the planned launch."""
    rng = np.random.default_rng(42)
    n = 210
    chunks = [int(x) for x in rng.integers(0, 12, n)]
    starts = [int(x) for x in rng.integers(0, 60, n)]
    chunks[3], starts[3], chunks[7], starts[7], chunks[9], starts[9] = 9, 0, 5, 40, 5, 40
    q, kp, vp, kvdt, bt, cu, ks, vs = _case(1400, H, Hkv, D, starts, chunks, kv)
    wide = -np.ones((n, 260), np.int32)
    wide[:, :bt.shape[1]] = bt
    wide[7, 1], wide[9, 2] = -1, 1 << 20
    out = []
    assert _plans(lambda: out.append(_run(q, kp, vp, wide, cu, starts, causal, mapping, ks, vs)), b"prefill_plan") == 1
    wide[9, 2] = -1  # (the oracle's walk ends at negative entries only)
    ref = oracle.paged_prefill(as_f32(q, oracle.BF16), kp, vp, kvdt, wide, cu, starts, Hkv, D, 16, np.float32(1 / math.sqrt(D)), causal,
                               oracle.GROUPED if mapping == "grouped" else oracle.MODULO, ks, vs)
    assert max_abs_err(as_f32(out[0], oracle.BF16), ref) <= 2e-2


@pytest.mark.parametrize("kv", ["bf16", "fp8"])
def test_unsplit_prefill_of_long_tables_without_a_plan(kv):
    """Contexts of more pages than a wave's lanes hold entries of (256): whole,
    and cut before and behind that many."""
    H = Hkv = 8
    n, D = 64, 64
    chunks, starts = [3] * n, [20] * n
    for i in (0, 20, 63):
        starts[i] = 4290 + i
    q, kp, vp, kvdt, bt, cu, ks, vs = _case(1500, H, Hkv, D, starts, chunks, kv)
    bt = bt.copy()
    bt[20, 261], bt[63, 100] = -1, -1
    out = []
    assert _plans(lambda: out.append(_run(q, kp, vp, bt, cu, starts, True, "grouped", ks, vs)), b"prefill_plan") == 0
    ref = oracle.paged_prefill(as_f32(q, oracle.BF16), kp, vp, kvdt, bt, cu, starts, Hkv, D, 16, np.float32(1 / math.sqrt(D)), True,
                               oracle.GROUPED, ks, vs)
    assert max_abs_err(as_f32(out[0], oracle.BF16), ref) <= 2e-2


@pytest.mark.skipif(PLANNED, reason="this run is that process")
def test_decode_suites_with_planned_launches():
    here = os.path.dirname(os.path.abspath(__file__))
    files = ["test_gpu_planned_launches", "test_gpu_decode_planless", "test_gpu_prefix_planless", "test_gpu_kv_cache", "test_gpu_decode"]
    r = subprocess.run([sys.executable, "-u", "-m", "pytest", "-x", "-q", "-m", "gpu", "-p", "no:cacheprovider", "-k", "not full_size and not prefill",
                        *(os.path.join(here, f + ".py") for f in files)], cwd=os.path.dirname(here), capture_output=True, text=True,
                       timeout=170, env={**os.environ, "ZEALOT_DECODE_PART_PAGES": "16"})
    assert r.returncode == 0, r.stdout[-4000:] + r.stderr[-2000:]


@pytest.mark.skipif(not PLANNED, reason="small batches are planned only with ZEALOT_DECODE_PART_PAGES")
def test_small_batches_are_planned_here():
    from zealot_amd import ops
    lens = [40, 300]
    for dt in (oracle.F32, oracle.BF16):
        args = [to_dev(x) for x in (*decode_case(5, 8, 2, 64, lens, dt)[:4], np.asarray(lens, np.int32))]
        assert _plans(lambda: ops.paged_decode(*args)) == 1
