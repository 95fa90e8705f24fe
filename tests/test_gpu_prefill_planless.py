"""Planless chunked prefill (small batches; items split over their keys) on the
MI355X against the oracle's or_paged_prefill: chunks behind contexts that several
splits share, chunk ends at tile edges, more sequences than a wave looks up at
once, tables cut in every split, and one batch large enough for the planned
launch with the same cuts.  Tolerance 2e-2 absolute, as tests/test_gpu_prefill.py."""
import math

import numpy as np
import pytest

import oracle
from tests.gpu_util import as_f32, max_abs_err
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
