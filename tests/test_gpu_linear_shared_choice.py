"""Decode-sized products (m <= 64) with the same number of 16-row tiles run one
configuration: the first shape's timing decides for the others, row-major and
tiled, and the products still match float64 (bf16 rounding of the sums: 2^-8 of
the largest output, as k = 2048 f32 accumulation adds far less)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tiled", [False, True])
def test_same_tiles_same_choice(tiled):
    from zealot_amd import dense
    n, k = 2048, 2048  # n k = 4M: the deep search
    g = torch.Generator(device="cuda").manual_seed(3)
    w = (torch.randn((n, k), generator=g, device="cuda") / k ** 0.5).bfloat16()
    wt = dense.tile_weight(w) if tiled else w
    for ms in ((33, 40, 48), (1, 16), (64, 50)):
        seen = set()
        for m in ms:
            x = torch.randn((m, k), generator=g, device="cuda").bfloat16()
            y = dense.linear(x, wt)
            want = x.double() @ w.double().T
            assert (y.double() - want).abs().max() <= want.abs().max() / 256
            seen.add(tuple(sorted(dense.linear_choice(m, n, k, tiled=tiled).items())))
        assert len(seen) == 1, seen
