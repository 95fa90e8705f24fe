"""Performance cases of the paged-KV framework: the calls a serving program makes.

A case is a dict of plain values; `kind` names the path:

  decode   ops.paged_decode over a batch of sequences (one query row each)
  prefill  ops.paged_prefill of prompt chunks behind cached tokens
  append   ops.append of prompt chunks; fp8 pools first take their scales
           (ops.fp8_scales), as a prompt's first append does
  prefix   KVCache.decode_append over the layers of one decode step, for
           sequences forked from shared prefixes
  step     KVCache.write_batch + attention_batch: one layer of a runner step
           that mixes decodes and prompt chunks
  model    Scheduler + HipModelRunner: a batch of prompts prefilled in one
           step, then a few decode steps, logits of every step

Every size and the draw of the lengths (`lens_seed`) belong to the case, the
values to the seed.  32 / 8 heads of 128 with 16-token blocks is the shape of
the repository's benchmark; its decode, append, prefix and chunk workloads are
listed at their own sizes.
"""
import math
import random

import numpy as np
import torch

from zealot_amd import BlockManager, KVCache, PagedKVRunner, Scheduler, SchedulerConfig, SeqBatch, dense, ops
from zealot_amd.model import HipModelRunner, LayerWeights, LlamaConfig, LlamaWeights

BS = 16  # tokens per block
GQA = {"heads": 32, "kv_heads": 8, "dim": 128}
_TORCH = {"bf16": torch.bfloat16, "f32": torch.float32}
_BYTES = {"bf16": 2, "f32": 4, "fp8": 1}


def listed():
    return [
        # a lightly loaded server: four short chats, one step's attention of one layer
        dict(name="decode_few", kind="decode", seqs=4, lo=17, hi=1000, kv="bf16", q="bf16", mapping="grouped", lens_seed=1, **GQA),
        # a full serving batch: the headline workload
        dict(name="decode_batch", kind="decode", seqs=256, lo=512, hi=8192, kv="bf16", q="bf16", mapping="grouped", lens_seed=2, **GQA),
        # two users with long documents: few sequences, long contexts
        dict(name="decode_long", kind="decode", seqs=2, lo=20000, hi=32000, kv="bf16", q="bf16", mapping="grouped", lens_seed=3, **GQA),
        # fp8 KV, where contexts are long and memory decides the batch
        dict(name="decode_fp8", kind="decode", seqs=96, lo=1024, hi=16384, kv="fp8", q="bf16", mapping="grouped", lens_seed=4, **GQA),
        # f32 KV, the cache's default type
        dict(name="decode_f32", kind="decode", seqs=48, lo=128, hi=4096, kv="f32", q="f32", mapping="grouped", lens_seed=5, **GQA),
        # chunked prefill of a full batch: 64 chunks of 512 behind up to 4095 cached tokens
        dict(name="prefill_chunks", kind="prefill", seqs=64, lo=512, hi=512, start_lo=1, start_hi=4095, kv="bf16", q="bf16",
             mapping="grouped", lens_seed=6, **GQA),
        # one user's prompt, its last and ragged chunk behind a long context
        dict(name="prefill_prompt", kind="prefill", seqs=1, lo=389, hi=389, start_lo=7680, start_hi=7680, kv="bf16", q="bf16",
             mapping="grouped", lens_seed=7, **GQA),
        # the KV write of the same full batch of chunks
        dict(name="append_chunks", kind="append", seqs=64, lo=512, hi=512, start_lo=1, start_hi=4095, kv="bf16", src="bf16",
             lens_seed=8, **GQA),
        # prompts of mixed lengths into fp8 pools: scales of K and V, then the quantising write
        dict(name="append_fp8", kind="append", seqs=12, lo=60, hi=2000, start_lo=0, start_hi=0, kv="fp8", src="bf16", lens_seed=9, **GQA),
        # 16 shared prompts with 8 samples each, four layers of a decode step
        dict(name="prefix_decode", kind="prefix", prefixes=16, forks=8, tokens_lo=2049, tokens_hi=2063, layers=4, lens_seed=10, **GQA),
        # a runner step on f32 pools: a prompt chunk beside running decodes
        dict(name="step_f32", kind="step", decodes=12, lo=100, hi=2000, chunks=1, chunk=150, start_hi=600, kv="f32", lens_seed=11, **GQA),
        # the whole call: eight prompts through scheduler and model, then three decode steps
        dict(name="model", kind="model", prompts=8, lo=20, hi=150, new=4, layers=2, hidden=4096, inter=14336, vocab=32000,
             lens_seed=12, **GQA),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _shape(rng):
    return rng.choice([GQA, GQA, {"heads": 32, "kv_heads": 32, "dim": 128}, {"heads": 16, "kv_heads": 8, "dim": 64},
                       {"heads": 64, "kv_heads": 8, "dim": 128}])


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "append", "append", "prefix", "step", "model"])
    base = {"kind": kind, "lens_seed": rng.randrange(1 << 20)}
    if kind == "decode":
        seqs = _log_int(rng, 1, 256)
        hi = _log_int(rng, 40, min(32000, 1200000 // seqs))
        kv = rng.choice(["bf16", "bf16", "fp8", "f32"])
        s = GQA if kv == "f32" else _shape(rng)
        hi = min(hi, 32000 * 32 * 8 // (seqs * s["kv_heads"])) if kv == "bf16" else min(hi, 400000 // seqs)
        hi = max(hi, 20)
        return dict(base, seqs=seqs, lo=max(1, hi // rng.choice([2, 8, 16])), hi=hi, kv=kv, q="f32" if kv == "f32" else "bf16",
                    mapping=rng.choice(["grouped", "modulo"]), **s)
    if kind == "prefill":
        seqs = _log_int(rng, 1, 32)
        hi = _log_int(rng, 20, 1024 if seqs <= 16 else 512)
        start = _log_int(rng, 1, 12000 if seqs <= 4 else 3000)
        return dict(base, seqs=seqs, lo=max(2, hi // rng.choice([1, 4])), hi=hi, start_lo=rng.choice([0, start // 2]), start_hi=start,
                    kv=rng.choice(["bf16", "bf16", "bf16", "fp8"]), q="bf16", mapping="grouped", **_shape(rng))
    if kind == "append":
        seqs = _log_int(rng, 1, 64)
        hi = _log_int(rng, 1, 1000)
        kv = rng.choice(["bf16", "fp8", "f32"])
        return dict(base, seqs=seqs, lo=max(1, hi // 8), hi=hi, start_lo=0, start_hi=0 if kv == "fp8" else rng.choice([0, 2000]), kv=kv,
                    src="f32" if kv == "f32" else "bf16", **_shape(rng))
    if kind == "prefix":
        lo = _log_int(rng, 300, 4000)
        return dict(base, prefixes=_log_int(rng, 1, 16), forks=rng.choice([2, 4, 8, 11]), tokens_lo=lo, tokens_hi=lo + 200, layers=4, **GQA)
    if kind == "step":
        kv = rng.choice(["bf16", "f32"])
        wide = kv == "bf16"
        return dict(base, decodes=_log_int(rng, 1, 200 if wide else 16), lo=50, hi=_log_int(rng, 100, 6000 if wide else 2000),
                    chunks=rng.choice([1, 1, 3]) if wide else 1, chunk=_log_int(rng, 17, 512 if wide else 150),
                    start_hi=_log_int(rng, 1, 3000 if wide else 600), kv=kv, **GQA)
    return dict(base, prompts=rng.randrange(1, 11), lo=10, hi=_log_int(rng, 20, 130), new=rng.choice([2, 4]), layers=2, hidden=4096,
                inter=14336, vocab=32000, **GQA)


# ------------------------------------------------------------------ sizes and values

def _randint(rng, lo, hi):
    return rng.randint(min(lo, hi), hi)


def _lens(case):
    """(chunk or context lengths, cached tokens before each chunk) of the case."""
    rng = random.Random(case["lens_seed"])
    k = case["kind"]
    if k == "decode":
        return [_randint(rng, case["lo"], case["hi"]) for _ in range(case["seqs"])], None
    if k in ("prefill", "append"):
        n = [_randint(rng, case["lo"], case["hi"]) for _ in range(case["seqs"])]
        return n, [_randint(rng, case["start_lo"], case["start_hi"]) for _ in n]
    if k == "prefix":
        return [_randint(rng, case["tokens_lo"], case["tokens_hi"]) for _ in range(case["prefixes"])], None
    if k == "step":
        n = [1] * case["decodes"] + [case["chunk"]] * case["chunks"]
        before = [_randint(rng, case["lo"], case["hi"]) - 1 for _ in range(case["decodes"])]
        return n, before + [_randint(rng, 0, case["start_hi"]) for _ in range(case["chunks"])]
    return [_randint(rng, case["lo"], case["hi"]) for _ in range(case["prompts"])], None


def _gen(seed, tag):
    return torch.Generator(device="cuda").manual_seed(seed * 64 + tag)


def _normal(shape, dtype, gen):
    """N(0, 1) values, filled in pieces (large pools at once would need a
    large temporary)."""
    out = torch.empty(shape, dtype=dtype, device="cuda")
    flat = out.view(-1)
    for i in range(0, flat.numel(), 1 << 27):
        flat[i:i + (1 << 27)].normal_(generator=gen)
    return out


def _codes(shape, gen):
    """e4m3 codes of N(0, 1) rows quantised to their largest value."""
    out = torch.empty(shape, dtype=torch.float8_e4m3fn, device="cuda")
    flat = out.view(-1)
    for i in range(0, flat.numel(), 1 << 26):
        x = torch.empty(min(1 << 26, flat.numel() - i), device="cuda").normal_(generator=gen).mul_(95.0).clamp_(-448.0, 448.0)
        flat[i:i + x.numel()] = x.to(torch.float8_e4m3fn)
    return out


def _tables(lens, seed):
    """Random, non-contiguous block tables [N, max pages] and the pool's blocks."""
    pages = [max(1, -(-n // BS)) for n in lens]
    blocks = int(sum(pages) * 1.1) + 4
    perm = np.random.default_rng(seed).permutation(blocks).astype(np.int32)
    bt = -np.ones((len(lens), max(pages)), np.int32)
    o = 0
    for i, p in enumerate(pages):
        bt[i, :p] = perm[o:o + p]
        o += p
    return bt, blocks


def _dev(a, dtype=None):
    return torch.as_tensor(a, dtype=dtype).to("cuda")


def _slots(bt, lens, starts):
    """int64 pool slots of the tokens start .. start + len of every sequence."""
    return np.concatenate([bt[i][(s + np.arange(n)) // BS].astype(np.int64) * BS + (s + np.arange(n)) % BS
                           for i, (n, s) in enumerate(zip(lens, starts))])


def _paged(case, seed, contexts):
    """Tables, pools and (fp8) scales that hold `contexts` tokens a sequence."""
    bt, blocks = _tables(contexts, case["lens_seed"] + 1000003 * seed)
    shape = (blocks, case["kv_heads"], BS, case["dim"])
    s = {"bt": bt, "ks": None, "vs": None}
    if case["kv"] == "fp8":
        s["kp"], s["vp"] = _codes(shape, _gen(seed, 1)), _codes(shape, _gen(seed, 2))
        g = _gen(seed, 3)
        for name in ("ks", "vs"):
            s[name] = 0.0105 + 0.001 * torch.rand((len(contexts), case["kv_heads"]), generator=g, device="cuda")
    else:
        t = _TORCH[case["kv"]]
        s["kp"], s["vp"] = _normal(shape, t, _gen(seed, 1)), _normal(shape, t, _gen(seed, 2))
    return s


# ------------------------------------------------------------------ decode, prefill

def _attention_inputs(case, seed):
    n, starts = _lens(case)
    ctx = n if starts is None else [a + b for a, b in zip(n, starts)]
    s = _paged(case, seed, ctx)
    rows = len(n) if starts is None else sum(n)
    s["q"] = _normal((rows, case["heads"], case["dim"]), _TORCH[case["q"]], _gen(seed, 4))
    return s, n, starts, ctx


def _prepare_decode(case, seed):
    s, _, _, ctx = _attention_inputs(case, seed)
    bt = s["bt"]
    s.update(bt=_dev(bt), lens=_dev(ctx, torch.int32), out=torch.empty_like(s["q"]), mapping=case["mapping"])
    s["ws"] = torch.empty(ops.decode_workspace_bytes(len(ctx), case["heads"], case["dim"], bt.shape[1], BS), dtype=torch.uint8,
                          device="cuda")
    return s


def _run_decode(s):
    return ops.paged_decode(s["q"], s["kp"], s["vp"], s["bt"], s["lens"], mapping=s["mapping"], k_scales=s["ks"], v_scales=s["vs"],
                            out=s["out"], workspace=s["ws"])


def _prepare_prefill(case, seed):
    s, n, starts, _ = _attention_inputs(case, seed)
    s.update(bt=_dev(s["bt"]), cu=_dev(np.concatenate([[0], np.cumsum(n)]), torch.int64), start=_dev(starts, torch.int32),
             out=torch.empty_like(s["q"]), mapping=case["mapping"])
    s["ws"] = torch.empty(ops.prefill_workspace_bytes(len(n), sum(n), case["heads"], case["kv_heads"]), dtype=torch.uint8, device="cuda")
    return s


def _run_prefill(s):
    return ops.paged_prefill(s["q"], s["kp"], s["vp"], s["bt"], s["cu"], s["start"], mapping=s["mapping"], k_scales=s["ks"],
                             v_scales=s["vs"], out=s["out"], workspace=s["ws"])


def _attend64(q, k, v, heads, kv_heads, mapping, causal_from):
    """softmax(q k^T / sqrt(D)) v in 64 bits: q [T, H, D], k and v [L, Hkv, D];
    row t sees the first causal_from + t + 1 keys."""
    t, _, d = q.shape
    g = heads // kv_heads
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    see = (torch.arange(k.shape[0], device=q.device)[None] <= causal_from + torch.arange(t, device=q.device)[:, None]).repeat(g, 1)
    for h in range(kv_heads):
        heads_of = [h * g + j if mapping == "grouped" else h + j * kv_heads for j in range(g)]
        qq = q[:, heads_of].double().transpose(0, 1).reshape(g * t, d)
        w = (qq @ k[:, h].double().T / math.sqrt(d)).masked_fill_(~see, float("-inf"))
        out[:, heads_of] = (torch.softmax(w, 1) @ v[:, h].double()).view(g, t, d).transpose(0, 1)
    return out


def _exact_attention(case, seed):
    s, n, starts, ctx = _attention_inputs(case, seed)
    out = torch.empty(s["q"].shape, dtype=torch.float64, device="cuda")
    row = 0
    for i, length in enumerate(ctx):
        rows = n[i] if starts is not None else 1
        blocks = _dev(s["bt"][i, :-(-length // BS)], torch.int64)
        kv = []
        for pool, scale in ((s["kp"], s["ks"]), (s["vp"], s["vs"])):
            x = pool.view(torch.uint8)[blocks].view(pool.dtype) if case["kv"] == "fp8" else pool[blocks]
            x = x.double().transpose(1, 2).reshape(-1, case["kv_heads"], case["dim"])[:length]
            kv.append(x if scale is None else x * scale[i].double()[None, :, None])
        out[row:row + rows] = _attend64(s["q"][row:row + rows], kv[0], kv[1], case["heads"], case["kv_heads"], case["mapping"],
                                        length - rows)
        row += rows
    return out


# ------------------------------------------------------------------ append

def _append_inputs(case, seed):
    n, starts = _lens(case)
    bt, blocks = _tables([a + b for a, b in zip(n, starts)], case["lens_seed"] + 1000003 * seed)
    rows = (sum(n), case["kv_heads"], case["dim"])
    t = _TORCH[case["src"]]
    return n, starts, bt, blocks, _normal(rows, t, _gen(seed, 1)), _normal(rows, t, _gen(seed, 2))


def _prepare_append(case, seed):
    n, starts, bt, blocks, k, v = _append_inputs(case, seed)
    pool = torch.float8_e4m3fn if case["kv"] == "fp8" else _TORCH[case["kv"]]
    shape = (blocks, case["kv_heads"], BS, case["dim"])
    s = {"k": k, "v": v, "slots": _dev(_slots(bt, n, starts)), "kp": torch.zeros(shape, dtype=pool, device="cuda"),
         "vp": torch.zeros(shape, dtype=pool, device="cuda"), "fp8": case["kv"] == "fp8"}
    if s["fp8"]:
        s["cu"] = _dev(np.concatenate([[0], np.cumsum(n)]), torch.int64)
        s["row"] = _dev(np.repeat(np.arange(len(n)), n), torch.int32)
    return s


def _run_append(s):
    if not s["fp8"]:
        ops.append(s["kp"], s["vp"], s["k"], s["v"], s["slots"])
        return s["kp"], s["vp"]
    ks, vs = ops.fp8_scales(s["k"], s["cu"]), ops.fp8_scales(s["v"], s["cu"])
    ops.append(s["kp"], s["vp"], s["k"], s["v"], s["slots"], k_scales=ks, v_scales=vs, token_row=s["row"])
    return s["kp"].view(torch.uint8), s["vp"].view(torch.uint8), ks, vs


def _exact_append(case, seed):
    n, starts, bt, blocks, k, v = _append_inputs(case, seed)
    slots = _dev(_slots(bt, n, starts))
    outs = []
    for x in (k, v):
        pool = torch.zeros((blocks, BS, case["kv_heads"], case["dim"]), dtype=torch.float64, device="cuda")
        pool.view(-1, case["kv_heads"], case["dim"])[slots] = x.double()
        outs.append(pool.transpose(1, 2).contiguous())
    if case["kv"] != "fp8":
        return tuple(outs)
    scales = [torch.stack([p.double().abs().amax((0, 2)) / 448.0 for p in x.split(n)]) for x in (k, v)]
    return None, None, scales[0], scales[1]  # the pools are bytes: the same on every side


# ------------------------------------------------------------------ prefix

def _prefix_inputs(case, seed):
    lens, _ = _lens(case)
    n = case["prefixes"] * case["forks"]
    g = _gen(seed, 1)
    kv = (case["kv_heads"], case["dim"])
    ctx = [[(_normal((t, *kv), torch.bfloat16, g), _normal((t, *kv), torch.bfloat16, g)) for t in lens] for _ in range(case["layers"] + 1)]
    new = [(_normal((n, *kv), torch.bfloat16, g), _normal((n, *kv), torch.bfloat16, g),
            _normal((n, case["heads"], case["dim"]), torch.bfloat16, g)) for _ in range(case["layers"])]
    return lens, ctx, new


def _prepare_prefix(case, seed):
    # the forks hold their own copy of the partial tail block (their first
    # write), and the last layer of the cache is not written, so that every
    # pass is the same step: each layer's new token is written and attended
    lens, ctx, new = _prefix_inputs(case, seed)
    layers, forks = case["layers"], case["forks"]
    pages = -(-max(lens) // BS) + 2
    blocks = sum(-(-t // BS) for t in lens) + 3 * len(lens) * forks + 8
    bm = BlockManager(blocks, BS)
    cache = KVCache(blocks, BS, layers + 1, case["kv_heads"], case["dim"], dtype=torch.bfloat16, max_seqs=len(lens) * (forks + 1),
                    max_blocks_per_seq=pages)
    ids = []
    for p, t in enumerate(lens):
        cache.register_seq(f"p{p}", pages)
        for _ in range(-(-t // BS)):
            cache.alloc_block(f"p{p}", bm)
        for layer in range(layers + 1):
            cache.store_kv(layer, f"p{p}", *ctx[layer][p], 0, t)
        for f in range(forks):
            cache.fork_seq(f"p{p}", f"p{p}.{f}")
            ids.append(f"p{p}.{f}")
            if t % BS == 0:
                cache.alloc_block(ids[-1], bm)
    batch = SeqBatch(ids)
    for layer in range(layers):
        cache.append_kv_batch(layer, batch, new[layer][0], new[layer][1])
    return {"bm": bm, "cache": cache, "batch": batch, "new": new, "out": [torch.empty_like(q) for _, _, q in new]}


def _run_prefix(s):
    for layer, (k, v, q) in enumerate(s["new"]):
        s["cache"].decode_append(layer, s["batch"], k, v, q, out=s["out"][layer])
    return s["out"]


def _exact_prefix(case, seed):
    lens, ctx, new = _prefix_inputs(case, seed)
    outs = []
    for layer, (k, v, q) in enumerate(new):
        out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
        for i in range(q.shape[0]):
            pk, pv = ctx[layer][i // case["forks"]]
            out[i] = _attend64(q[i:i + 1], torch.cat([pk, k[i:i + 1]]), torch.cat([pv, v[i:i + 1]]), case["heads"], case["kv_heads"],
                               "grouped", pk.shape[0])[0]
        outs.append(out)
    return outs


# ------------------------------------------------------------------ step

def _step_inputs(case, seed):
    n, before = _lens(case)
    t = _TORCH[case["kv"]]
    kv = (case["kv_heads"], case["dim"])
    g = _gen(seed, 1)
    ctx = [_normal((max(1, sum(before)), *kv), t, g)[:sum(before)] for _ in range(2)]
    k, v = (_normal((sum(n), *kv), t, g) for _ in range(2))
    return n, before, ctx, k, v, _normal((sum(n), case["heads"], case["dim"]), t, g)


def _prepare_step(case, seed):
    # layer 0 of a two-layer cache: its tokens are rewritten by every pass, so
    # that every pass is the same step
    n, before, ctx, k, v, q = _step_inputs(case, seed)
    pages = [-(-(a + b) // BS) for a, b in zip(n, before)]
    bm = BlockManager(sum(pages) + 8, BS)
    cache = KVCache(sum(pages) + 8, BS, 2, case["kv_heads"], case["dim"], dtype=_TORCH[case["kv"]], max_seqs=len(n),
                    max_blocks_per_seq=max(pages))
    ids = [f"s{i}" for i in range(len(n))]
    for sid, p in zip(ids, pages):
        cache.register_seq(sid, p)
        for _ in range(p):
            cache.alloc_block(sid, bm)
    batch = SeqBatch(ids)
    if sum(before):
        for layer in range(2):
            cache.write_batch(layer, batch, before, ctx[0], ctx[1])
    return {"bm": bm, "cache": cache, "batch": batch, "n": n, "k": k, "v": v, "q": q, "out": torch.empty_like(q)}


def _run_step(s):
    s["cache"].write_batch(0, s["batch"], s["n"], s["k"], s["v"])
    return s["cache"].attention_batch(0, s["batch"], s["n"], s["q"], out=s["out"])


def _exact_step(case, seed):
    n, before, ctx, k, v, q = _step_inputs(case, seed)
    out, row, at = torch.empty(q.shape, dtype=torch.float64, device="cuda"), 0, 0
    for t, b in zip(n, before):
        kk, vv = (torch.cat([c[at:at + b], x[row:row + t]]) for c, x in zip(ctx, (k, v)))
        out[row:row + t] = _attend64(q[row:row + t], kk, vv, case["heads"], case["kv_heads"], "grouped", b)
        row, at = row + t, at + b
    return out


# ------------------------------------------------------------------ model

def _model_inputs(case, seed):
    """Row-major weights and token ids (prompt, then the tokens fed to the decode steps)."""
    lens, _ = _lens(case)
    g = _gen(seed, 1)
    hid, qd, kd = case["hidden"], case["heads"] * case["dim"], case["kv_heads"] * case["dim"]

    def lin(n, k):
        return (_normal((n, k), torch.float32, g) / math.sqrt(k)).to(torch.bfloat16)

    def norm():
        return (1 + 0.1 * _normal((hid,), torch.float32, g)).to(torch.bfloat16)

    w = {"emb": _normal((case["vocab"], hid), torch.bfloat16, g), "final": norm(), "head": lin(case["vocab"], hid),
         "layers": [dict(an=norm(), qkv=lin(qd + 2 * kd, hid), o=lin(hid, qd), fn=norm(), gate=lin(case["inter"], hid),
                         up=lin(case["inter"], hid), down=lin(hid, case["inter"])) for _ in range(case["layers"])]}
    rng = random.Random(seed)
    return w, lens, [[rng.randrange(case["vocab"]) for _ in range(t + case["new"])] for t in lens]


def _prepare_model(case, seed):
    w, lens, toks = _model_inputs(case, seed)
    cfg = LlamaConfig(case["vocab"], case["hidden"], case["inter"], case["layers"], case["heads"], case["kv_heads"], case["dim"])

    def tile(t):
        return dense.tile_weight(t, keep_full=True)

    layers = [LayerWeights(lw["an"], lw["qkv"], lw["o"], lw["fn"], tile(dense.interleave_gate_up(lw["gate"], lw["up"])), tile(lw["down"]))
              for lw in w["layers"]]
    blocks = sum(-(-(t + case["new"]) // BS) + 1 for t in lens)
    bm = BlockManager(blocks, BS)
    cache = KVCache(blocks, BS, case["layers"], case["kv_heads"], case["dim"], dtype=torch.bfloat16, max_seqs=len(lens),
                    max_blocks_per_seq=-(-(max(lens) + case["new"]) // BS) + 1)
    sched = Scheduler(SchedulerConfig(max_num_seqs=len(lens), block_size=BS, num_gpu_blocks=blocks, max_prefill_tokens=sum(lens),
                                      prefill_chunk_size=max(lens)), block_manager=bm)
    runner = HipModelRunner(cfg, LlamaWeights(w["emb"], layers, w["final"], tile(w["head"])), PagedKVRunner(cache, bm))
    return {"sched": sched, "runner": runner, "lens": lens, "toks": toks, "new": case["new"]}


def _run_model(s):
    # the engine's loop; the tokens that follow the prompts are given, so that
    # the logits of every step can be compared
    sched, runner, new = s["sched"], s["runner"], s["new"]
    for i, (t, toks) in enumerate(zip(s["lens"], s["toks"])):
        sched.submit(str(i), toks[:t], new)
    logits, fed = [], [0] * len(s["lens"])
    while not sched.is_idle():
        out = sched.schedule()
        logits.append(runner.step(out))
        for e in out.batch:
            i = int(e.request_id)
            e.push_token(s["toks"][i][s["lens"][i] + fed[i]])
            fed[i] += 1
            if e.is_prefill():
                e.mark_prefilled()
                sched.advance_prefill(e.request_id)
            if fed[i] == new:
                runner.drop_state(e.request_id)
                sched.finish(e.request_id)
    return logits


def _exact_model(case, seed):
    w, lens, toks = _model_inputs(case, seed)
    h, hkv, d, eps = case["heads"], case["kv_heads"], case["dim"], 1e-6

    def norm(x, wt):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * wt.double()

    seqs = [t + case["new"] - 1 for t in lens]  # tokens fed to the model
    x = w["emb"][_dev([t for s, n in zip(toks, seqs) for t in s[:n]])].double()
    for lw in w["layers"]:
        q, k, v = (norm(x, lw["an"]) @ lw["qkv"].double().T).split([h * d, hkv * d, hkv * d], 1)
        a = [_attend64(qq.reshape(-1, h, d), kk.reshape(-1, hkv, d), vv.reshape(-1, hkv, d), h, hkv, "grouped", 0).view(-1, h * d)
             for qq, kk, vv in zip(q.split(seqs), k.split(seqs), v.split(seqs))]
        x = x + torch.cat(a) @ lw["o"].double().T
        y = norm(x, lw["fn"])
        x = x + (torch.nn.functional.silu(y @ lw["gate"].double().T) * (y @ lw["up"].double().T)) @ lw["down"].double().T
    y = [p[-case["new"]:] for p in norm(x, w["final"]).split(seqs)]
    return [torch.stack([p[i] for p in y]) @ w["head"].double().T for i in range(case["new"])]


# ------------------------------------------------------------------ the interface

_PREPARE = {"decode": _prepare_decode, "prefill": _prepare_prefill, "append": _prepare_append, "prefix": _prepare_prefix,
            "step": _prepare_step, "model": _prepare_model}
_RUN = {"decode": _run_decode, "prefill": _run_prefill, "append": _run_append, "prefix": _run_prefix, "step": _run_step,
        "model": _run_model}
_EXACT = {"decode": _exact_attention, "prefill": _exact_attention, "append": _exact_append, "prefix": _exact_prefix,
          "step": _exact_step, "model": _exact_model}


def prepare(case, seed):
    return case["kind"], _PREPARE[case["kind"]](case, seed)


def run(state):
    return _RUN[state[0]](state[1])


def exact(case, seed):
    return _EXACT[case["kind"]](case, seed)


def work(case):
    k, h, hkv, d = case["kind"], case["heads"], case["kv_heads"], case["dim"]
    n, starts = _lens(case)
    elt = _BYTES[case.get("kv", "bf16")]
    token = 2 * hkv * d  # values of K and V a token
    io = _BYTES["f32"] if case.get("kv") == "f32" else 2
    if k == "append":
        src = _BYTES[case["src"]]
        return {"bytes": sum(n) * (token * (src + elt) + 8), "flops": 0}
    if k in ("decode", "prefill", "step"):
        before = starts if starts is not None else [t - 1 for t in n]
        rows = n if starts is not None else [1] * len(n)
        keys = sum(r * b + r * (r + 1) // 2 for r, b in zip(rows, before))
        ctx = sum(r + b for r, b in zip(rows, before))
        new = sum(rows) * token * 2 * elt if k == "step" else 0
        return {"bytes": ctx * token * elt + 2 * sum(rows) * h * d * io + new, "flops": 4 * d * h * keys}
    if k == "prefix":
        seqs = len(n) * case["forks"]
        per_layer = (sum(n) + 3 * seqs) * token * 2 + 2 * seqs * h * d * 2
        return {"bytes": case["layers"] * per_layer, "flops": case["layers"] * 4 * d * h * case["forks"] * sum(t + 1 for t in n)}
    hid, inter, new = case["hidden"], case["inter"], case["new"]
    proj = case["layers"] * ((h * d + token) * hid + hid * h * d + 3 * hid * inter)
    fed = sum(n) + (new - 1) * len(n)
    keys = sum(m * (m + 1) // 2 for m in (t + new - 1 for t in n))
    return {"bytes": new * (proj + case["vocab"] * hid) * 2 + new * len(n) * case["vocab"] * 4,
            "flops": 2 * proj * fed + 2 * case["vocab"] * hid * new * len(n) + 4 * d * h * keys * case["layers"]}


def tolerance(case):
    k, kv = case["kind"], case.get("kv", "bf16")
    if k == "append":
        return {"rel": 1e-6, "differ": 0.0} if kv == "fp8" else "exact"
    if k == "model":
        return {"rel": 0.023, "max": 0.3}
    if kv == "f32":
        return {"rel": 4e-6, "max": 1e-4}
    return {"rel": 1e-2, "max": 0.1}
