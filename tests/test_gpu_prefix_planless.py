"""Shared-prefix decode without a plan (small and mid-sized batches) on the
MI355X against float64 attention: prefixes around the shared partitions' 10
pages, two members and more than one subgroup's worth, forks that diverged by
several partitions of their own, sequences that share nothing beside them, with
and without the fused append.  Tolerance 2e-2 absolute (bf16)."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,Hkv,D", [(32, 8, 128), (8, 8, 64), (16, 2, 128)])
@pytest.mark.parametrize("append", [False, True])
def test_forks_match_float64(H, Hkv, D, append):
    from zealot_amd import BlockManager, KVCache
    g = torch.Generator(device="cuda").manual_seed(H + D)
    nb, mb = 900, 80
    bm = BlockManager(nb, 16)
    cache = KVCache(nb, 16, 2, Hkv, D, dtype=torch.bfloat16, max_seqs=64, max_blocks_per_seq=mb)

    def rows(n):
        return torch.randn((n, Hkv, D), generator=g, device="cuda").bfloat16()

    held = {}  # K, V of every sequence at layer 0

    def grow(sid, n):
        have = held[sid][0].shape[0]
        for _ in range(-(-(have + n) // 16) - -(-have // 16)):
            cache.alloc_block(sid, bm)
        k, v = rows(n), rows(n)
        for layer in (0, 1):
            cache.write_batch(layer, [sid], [n], k, v)
        held[sid] = (torch.cat([held[sid][0], k]), torch.cat([held[sid][1], v]))

    ids = []
    for p, (tokens, forks, tails) in enumerate([(16 * 16, 2, (1, 17)), (16 * 20 + 3, 3, (5, 1, 300)), (16 * 31, 9, (1,) * 9), (40, 2, (2, 2))]):
        cache.register_seq(f"p{p}", mb)
        held[f"p{p}"] = (rows(0), rows(0))
        grow(f"p{p}", tokens)
        for f in range(forks):
            sid = f"p{p}.{f}"
            cache.fork_seq(f"p{p}", sid)
            held[sid] = held[f"p{p}"]
            grow(sid, tails[f])
            ids.append(sid)
    cache.register_seq("alone", mb)
    held["alone"] = (rows(0), rows(0))
    grow("alone", 700)
    ids.insert(3, "alone")
    q = torch.randn((len(ids), H, D), generator=g, device="cuda").bfloat16()
    if append:
        for sid in ids:
            if held[sid][0].shape[0] % 16 == 0:
                cache.alloc_block(sid, bm)
        k, v = rows(len(ids)), rows(len(ids))
        out = cache.decode_append(0, ids, k, v, q)
        for i, sid in enumerate(ids):
            held[sid] = (torch.cat([held[sid][0], k[i:i + 1]]), torch.cat([held[sid][1], v[i:i + 1]]))
    else:
        out = cache.paged_decode(0, ids, q)
    assert cache.decode_sharing()[0] >= 3
    for i, sid in enumerate(ids):
        kk, vv = (x.double() for x in held[sid])
        for h in range(H):
            w = torch.softmax(kk[:, h * Hkv // H] @ q[i, h].double() / math.sqrt(D), 0)
            assert (out[i, h].double() - w @ vv[:, h * Hkv // H]).abs().max() <= 2e-2, (sid, h)
