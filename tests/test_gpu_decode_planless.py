"""Planless paged decode (small and mid-sized batches: one workgroup per
kv-head, partition and sequence, partitions of at least 8 pages) and the f32
MFMA kernel on the MI355X, against the CPU oracle: lengths around the
partition edges, tables cut by a sentinel or an out-of-range id in every part
of the walk (a cut inside one partition drops all after it), more partitions
than one wave merges, f32 operands off their 16-byte alignment (the generic
kernel).  Tolerances (absolute): 1e-5 f32, 2e-2 bf16, as tests/test_gpu_decode.py."""
import numpy as np
import pytest
import torch

import oracle
from tests.gpu_util import as_f32, decode_case, max_abs_err, to_dev, to_host
from tests.test_gpu_decode import TOL, _oracle

pytestmark = pytest.mark.gpu

PART = 8 * 16  # tokens of the smallest partition


def _decode(q, kp, vp, bt, lens, mapping="grouped"):
    from zealot_amd import ops
    out = ops.paged_decode(to_dev(q), to_dev(kp), to_dev(vp), to_dev(bt), to_dev(np.asarray(lens, np.int32)), mapping=mapping)
    torch.cuda.synchronize()
    return as_f32(to_host(out), oracle.BF16 if out.dtype == torch.bfloat16 else oracle.F32)


@pytest.mark.parametrize("dt", [oracle.F32, oracle.BF16])
@pytest.mark.parametrize("H,Hkv,D", [(32, 8, 128), (8, 8, 128), (16, 8, 64), (64, 8, 128)])
def test_partition_edges(dt, H, Hkv, D):
    lens = [0, 1, 16, PART - 1, PART, PART + 1, 2 * PART, 7 * PART + 17, 20 * PART + 5]  # 21 partitions: the many-part merge
    q, kp, vp, bt, _ = decode_case(900 + H + D, H, Hkv, D, lens, dt)
    for mapping in ("grouped", "modulo"):
        got = _decode(q, kp, vp, bt, lens, mapping)
        assert np.all(got[0] == 0)
        assert max_abs_err(got, _oracle(q, kp, vp, bt, lens, dt, dt, mapping)) <= TOL[dt]


@pytest.mark.parametrize("dt", [oracle.F32, oracle.BF16])
@pytest.mark.parametrize("H,Hkv,D,pages", [(32, 8, 128, 30), (16, 16, 64, 30), (32, 8, 128, 200)])
def test_cut_tables(dt, H, Hkv, D, pages):
    cuts = [0, 1, 7, 8, 9, 16, pages // 2, pages - 1]
    lens = [16 * pages - 3] * len(cuts)
    q, kp, vp, bt, nb = decode_case(950 + D + pages, H, Hkv, D, lens, dt)
    bt = bt.copy()
    for i, c in enumerate(cuts):
        bt[i, c] = -1 if i % 2 else nb + i
    ref = [16 * c for c in cuts]
    got = _decode(q, kp, vp, bt, lens)
    assert np.all(got[0] == 0)
    assert max_abs_err(got, _oracle(q, kp, vp, bt, ref, dt, dt, "grouped")) <= TOL[dt]


def test_f32_operands_off_their_alignment():
    from zealot_amd import ops
    lens = [5, 300, 700]
    q, kp, vp, bt, _ = decode_case(970, 32, 8, 128, lens, oracle.F32)

    def off(a):  # the same values one element past an aligned address
        t = torch.empty(a.size + 1, dtype=torch.float32, device="cuda")
        t[1:] = torch.from_numpy(a).flatten().cuda()
        return t[1:].view(a.shape)

    ref = _oracle(q, kp, vp, bt, lens, oracle.F32, oracle.F32, "grouped")
    args = (to_dev(bt), to_dev(np.asarray(lens, np.int32)))
    for qq, kk, vv in ((off(q), to_dev(kp), to_dev(vp)), (to_dev(q), off(kp), off(vp))):
        out = ops.paged_decode(qq, kk, vv, *args)
        assert max_abs_err(to_host(out), ref) <= TOL[oracle.F32]


@pytest.mark.parametrize("dt", [oracle.F32, oracle.BF16])
@pytest.mark.parametrize("H,Hkv,D", [(32, 8, 128), (8, 8, 128), (16, 8, 64)])
def test_pages_of_minus_infinity(dt, H, Hkv, D):
    """Keys whose scores are all -inf (whole pages, whole partitions, at the
    start, inside and at the end of a partition) have weight 0; a context of
    nothing else is NaN, as a softmax of it is; an empty one is zeros."""
    dead = {0: [(0, 16)], 1: [(0, 2 * PART)], 2: [(PART, PART + 40)], 3: [(PART, 2 * PART), (4 * PART - 16, 4 * PART)],
            4: [(0, 5 * PART + 3)], 5: [(0, 90)], 7: [(0, 26 * PART - 1)]}
    lens = [40, 5 * PART + 3, 5 * PART + 3, 5 * PART + 3, 5 * PART + 3, 90, 0, 26 * PART]
    q, kp, vp, bt, _ = decode_case(980 + H + D, H, Hkv, D, lens, dt)
    qf = as_f32(q, dt).copy()
    qf[:, :, 0] = np.abs(qf[:, :, 0]) + 0.5
    q = qf if dt == oracle.F32 else oracle.bf16_bits_from_f32(qf).reshape(qf.shape)
    for n, spans in dead.items():
        for lo, hi in spans:
            for t in range(lo, hi):
                kp[bt[n, t // 16], :, t % 16, 0] = -np.inf if dt == oracle.F32 else 0xff80
    got = _decode(q, kp, vp, bt, lens)
    kf, vf, qf = (as_f32(x, dt).astype(np.float64) for x in (kp, vp, q))
    for n, length in enumerate(lens):
        alive = np.ones(length, bool)
        for lo, hi in dead.get(n, []):
            alive[lo:hi] = False
        if not alive.any():
            assert np.isnan(got[n]).all() if length else np.all(got[n] == 0)
            continue
        t = np.flatnonzero(alive)
        for h in range(H):
            k, v = (x[bt[n, t // 16], h // (H // Hkv), t % 16] for x in (kf, vf))
            w = k @ qf[n, h] / np.sqrt(D)
            w = np.exp(w - w.max())
            assert max_abs_err(got[n, h], w @ v / w.sum()) <= TOL[dt], (n, h)
