"""zk_fp8_scales on the MI355X, value for value against numpy: rows of whole and
of ragged 16-byte chunks, empty and one-token sequences, more chunks than one
round of a workgroup's loads, all-zero heads (scale 1), NaN (ignored) and
infinities, and a source off its 16-byte alignment."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [128, 64, 96, 100, 7])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("off", [0, 1])
def test_scales_match_numpy(D, dtype, off):
    from zealot_amd import ops
    hkv, lens = 3, [0, 1, 3, 700, 64, 513]
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    T = int(cu[-1])
    store = torch.randn(T * hkv * D + off, generator=torch.Generator().manual_seed(D + off)).to(dtype)
    x = store[off:].view(T, hkv, D)
    x[1:4, 1] = 0.0
    x[4 + 650, 2, D - 1] = 1000.0  # the last element of a late row
    x[10, 0, 0] = float("nan")
    x[-1, 0, 0] = float("-inf")
    dev = store.cuda()[off:].view(T, hkv, D)
    got = ops.fp8_scales(dev, torch.from_numpy(cu).cuda()).cpu().numpy()
    a = np.abs(x.float().numpy())
    for n, length in enumerate(lens):
        m = np.nanmax(a[cu[n]:cu[n + 1]], axis=(0, 2)) if length else np.zeros(hkv, np.float32)
        want = np.where(m > 0, m.astype(np.float32) / np.float32(448.0), np.float32(1.0))
        np.testing.assert_array_equal(got[n], want)


def test_trailing_dimensions_of_one():
    """x may carry dimensions of one behind [T, Hkv, D]; no sequences, no scales."""
    from zealot_amd import ops
    x = torch.randn((900, 2, 64), generator=torch.Generator().manual_seed(1)).cuda()
    cu = torch.tensor([0, 300, 900], device="cuda")
    assert torch.equal(ops.fp8_scales(x.unsqueeze(-1), cu), ops.fp8_scales(x, cu))
    assert ops.fp8_scales(x, cu[:1]).shape == (0, 2)


@pytest.mark.parametrize("n,tokens,want", [(8, 512, 0), (8, 2000, 1), (1, 700, 0), (1, 4000, 1)])
def test_short_prompts_take_one_launch(n, tokens, want):
    """Only prompts long enough to gain from parts pay for the launch that merges them."""
    from zealot_amd import _lib, ops
    x = torch.randn((n * tokens, 8, 128), device="cuda").bfloat16()
    cu = (torch.arange(n + 1) * tokens).cuda()
    lib, launches, ms = _lib.lib(), ctypes.c_int64(), ctypes.c_double()
    lib.zk_timing_reset()
    lib.zk_timing_enable(1)
    got = ops.fp8_scales(x, cu)
    torch.cuda.synchronize()
    lib.zk_timing_enable(0)
    _lib.check(lib.zk_timing_query(b"fp8_scales_merge", ctypes.byref(launches), ctypes.byref(ms)))
    lib.zk_timing_reset()
    assert launches.value == want
    amax = x.view(n, tokens, 8, 128).abs().amax((1, 3)).float().cpu().numpy()
    np.testing.assert_array_equal(got.cpu().numpy(), amax / np.float32(448.0))
