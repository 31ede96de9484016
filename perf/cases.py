"""The work a user of triebwerk_amd has it do, as cases that a timing program can prepare, run and compare.

A case is a dict of plain values.  Its "kind" says which public entry points it goes through:

  layer      Engine.layer_step, eager: append + attention of a batch, layer after layer
  decode     Engine.set_positions, then Engine.decode_step as a captured graph, `steps` tokens for every sequence
  rollout    the same with the rest of the generation loop: QK norm and RoPE with the step (Engine.set_producers),
             begin_generation, record_tokens, check_stops, output
  single     Engine.single_step / single_advance: generate() for one sequence, every layer called by itself
  paged      tw_paged_turbo_append_attention_batch (or the two fp16 calls) over a shuffled block table
  launchers  the reference engine's own launchers, called as its forward_layer_batch calls them
  prompt     Engine.prompt_layer over one prompt
  group      prompts of a group rollout: Engine.prompt_layer for every prompt, broadcast_prefix to its group

A pass may be repeated on the same state: positions start from the same values every time and a row that is appended
again gets the same contents.  All passes of a process run on one stream, as a serving program's do.
"""
from __future__ import annotations

import functools

import numpy as np
import torch

from triebwerk_amd import Engine, kvcache

D = 128                                   # head dimension of every kernel
HEAD_BYTES = {0: 256, 4: 66, 2: 34}       # one K or V head of one token: fp16 row, or packed codes + fp16 norm
KV_BOUNDS = {4: (-0.21224, -0.16299, -0.12701, -0.09715, -0.07068, -0.04619, -0.02284, 0.0,
                 0.02284, 0.04619, 0.07068, 0.09715, 0.12701, 0.16299, 0.21224),
             2: (-0.08677, 0.0, 0.08677)}  # decision boundaries of the two code widths (unit-norm vectors)


def listed():
    return [
        # one layer of a small fp16 batch: bench.py's config1, the smallest call there is
        dict(name="layer_fp16_b4", kind="layer", bits=0, layers=1, heads=16, kv_heads=8, batch=4, ctx_min=613, ctx_max=613),
        # generate() for one long conversation on a compressed cache, 28 layers called one by one
        dict(name="single_kv4_long", kind="single", bits=4, layers=28, heads=16, kv_heads=8, ctx=16001, steps=4),
        # bench.py's config2: a small batch at a few hundred tokens
        dict(name="decode_kv4_b4", kind="decode", bits=4, layers=28, heads=16, kv_heads=8, batch=4, ctx_min=613, ctx_max=613, steps=32),
        # bench.py's config5 in the middle of its 512 steps, with everything a rollout loop does around the step
        dict(name="rollout_kv4_b128", kind="rollout", bits=4, layers=28, heads=16, kv_heads=8, batch=128, ctx_min=489, ctx_max=489, steps=48),
        # bench.py's target workload, its headline
        dict(name="decode_kv4_b64_ctx8192", kind="decode", bits=4, layers=28, heads=16, kv_heads=8, batch=64, ctx_min=8192, ctx_max=8192, steps=4),
        # bench.py's config4: the 8B-like shape, four query heads to a KV head, 2 bit
        dict(name="decode_kv2_gqa4_b16", kind="decode", bits=2, layers=36, heads=32, kv_heads=8, batch=16, ctx_min=4097, ctx_max=4097, steps=8),
        # the target workload on an fp16 cache (8 of the 28 layers, so that three states fit)
        dict(name="decode_fp16_b64_ctx8192", kind="decode", bits=0, layers=8, heads=16, kv_heads=8, batch=64, ctx_min=8192, ctx_max=8192, steps=4),
        # bench.py's config3: serving, every sequence at another length, pages of 16 tokens in any order
        dict(name="paged_kv4_b64_ragged", kind="paged", bits=4, layers=8, heads=16, kv_heads=8, batch=64, ctx_min=512, ctx_max=8192),
        # the reference's engine re-linked against this library, 2-bit cache, ragged batch of an odd size
        dict(name="launchers_kv2_b47_ragged", kind="launchers", bits=2, layers=8, heads=16, kv_heads=8, batch=47, ctx_min=300, ctx_max=5003),
        # the start of a group rollout (config5): short prompts, each prefilled once and handed to its group
        dict(name="group_kv4_16x8", kind="group", bits=4, layers=28, heads=16, kv_heads=8, prompts=16, group=8, t_min=97, t_max=256),
        # long prompts: bench.py's 8192 tokens on an fp16 cache, and an odd length on a compressed one with QK norm and RoPE
        dict(name="prompt_fp16_8192", kind="prompt", bits=0, layers=4, heads=16, kv_heads=8, tokens=8192, producers=False),
        dict(name="prompt_kv4_4111", kind="prompt", bits=4, layers=4, heads=16, kv_heads=8, tokens=4111, producers=True),
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, spread evenly over its logarithm."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    """One more case; one that would cost more than the largest listed one gets fewer steps, then fewer sequences."""
    c = _draw(rng)
    most = max(_cost(x) for x in listed())
    while _cost(c) > most:
        for key in ("steps", "batch", "prompts"):
            if c.get(key, 1) > 1:
                c[key] = max(1, c[key] * 3 // 4)
                break
    return c


def _cost(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 50)


def _draw(rng):
    kind = rng.choice(["layer", "single", "decode", "decode", "rollout", "paged", "launchers", "group", "prompt", "prompt"])
    bits = rng.choice([0, 4, 4, 2])
    layers, heads, kv_heads = rng.choice([(28, 16, 8), (28, 16, 8), (36, 32, 8), (28, 8, 8)])
    c = dict(kind=kind, bits=bits, heads=heads, kv_heads=kv_heads)
    if kind == "prompt":
        c.update(layers=4, tokens=_log(rng, 64, 8192 * 16 // max(heads, 16) if bits == 0 else 6000 * 16 // max(heads, 16)), producers=rng.random() < 0.5)
        return c
    if kind == "group":
        t = _log(rng, 32, 512)
        c.update(layers=layers, prompts=rng.randint(2, 12), group=rng.randint(2, 8), t_min=max(1, int(t * rng.uniform(0.4, 1.0))), t_max=t)
        return c
    if kind == "single":
        c.update(layers=28, ctx=_log(rng, 64, 25600 if bits else 7168), steps=4)
        return c
    # batches: at most a quarter million tokens a layer on the fp16 cache, half a million on a compressed one
    batch = _log(rng, 1, 160)
    ctx = _log(rng, 64, 8192)
    ctx = max(64, min(ctx, (500_000 if bits else 260_000) // batch))
    if kind == "layer":
        c.update(layers=rng.randint(1, 4), batch=batch)
    elif kind in ("paged", "launchers"):
        c.update(layers=rng.randint(2, 6), batch=batch)
    else:
        c.update(layers=layers if bits or batch * ctx < 60_000 else 8, batch=batch)
        c["steps"] = rng.randint(9, 24) if kind == "rollout" else rng.randint(2, 6)
    spread = rng.choice([1.0, 0.9, 0.1]) if kind in ("layer", "paged", "launchers") else rng.choice([1.0, 0.93])
    c.update(ctx_min=max(1, int(ctx * spread)), ctx_max=ctx)
    return c


# ---------------------------------------------------------------- inputs

@functools.lru_cache(maxsize=None)
def _stream():
    return torch.cuda.Stream()


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _randn(g, *shape, scale=1.0):
    out = torch.empty(shape, dtype=torch.float16, device="cuda")
    flat = out.view(-1)
    for i in range(0, flat.numel(), 1 << 27):
        n = min(1 << 27, flat.numel() - i)
        flat[i:i + n] = scale * torch.randn(n, generator=g, device="cuda")
    return out


class _Filler:
    """Cache contents from one block of fresh values: every 4 MB piece of a cache is the block from another place."""
    PIECE = 1 << 22

    def __init__(self, g, seed, bits):
        self.rng = np.random.Generator(np.random.Philox(int(seed)))
        n = 3 * self.PIECE
        if bits == 0:
            self.block = torch.randn(n // 2, generator=g, device="cuda").to(torch.float16).view(torch.uint8)
        else:
            per = 8 // bits
            x = torch.randn((n, per), generator=g, device="cuda") / D ** 0.5     # coordinates of rotated unit vectors
            codes = torch.bucketize(x, torch.tensor(KV_BOUNDS[bits], device="cuda"), right=True)
            shifts = bits * torch.arange(per, device="cuda")
            self.block = (codes << shifts).sum(1).to(torch.uint8)
        self.norms = (11.3 + 0.7 * torch.randn(n // 2, generator=g, device="cuda")).to(torch.float16).view(torch.uint8)

    def fill(self, cache):
        for i, t in enumerate(cache):
            if t is None:
                continue
            src = self.block if i < 2 else self.norms
            flat = t.view(-1).view(torch.uint8)
            for at in range(0, flat.numel(), self.PIECE):
                n = min(self.PIECE, flat.numel() - at)
                o = 256 * int(self.rng.integers(0, (src.numel() - n) // 256))
                flat[at:at + n].copy_(src[o:o + n])


def _contexts(case, seed):
    """Tokens each sequence attends to in the first step, the appended one included."""
    lo, hi, n = case["ctx_min"], case["ctx_max"], case["batch"]
    if lo == hi:
        return np.full(n, hi, np.int64)
    got = lo + np.floor((hi - lo) * (np.arange(n) + 0.5) / n).astype(np.int64)     # even over the range, in any order
    return np.random.Generator(np.random.Philox(int(seed))).permutation(got)


def _rope_tables(rows):
    ang = torch.arange(rows, device="cuda", dtype=torch.float64)[:, None] * 1e6 ** (-2.0 * torch.arange(D // 2, device="cuda", dtype=torch.float64) / D)
    return torch.cos(ang).to(torch.float16), torch.sin(ang).to(torch.float16)


def _set_producers(eng, g, layers, rows):
    weights = [(1 + 0.1 * torch.randn((layers, D), generator=g, device="cuda")).to(torch.float16) for _ in range(2)]
    cos, sin = _rope_tables(rows)
    eng.set_producers(1, q_norm=weights[0], k_norm=weights[1], eps=1e-6, rope_cos=cos, rope_sin=sin, rope_dim=D)


def _engine(case, batch, max_seq_len):
    eng = Engine(max_seq_len=max_seq_len, kv_bits=case["bits"])
    eng.set_shape(case["layers"], case["heads"], case["kv_heads"], D)
    if case["kind"] == "single":
        eng.alloc_single()
    else:
        eng.alloc_batch(batch, max_seq_len)
    return eng


def _row_views(eng, layers, lo, hi):
    """Rows lo .. hi - 1 of every sequence and layer, as one view of each cache array (the layers of an engine's arena
    lie at equal distances)."""
    views = []
    first, second = eng.cache(0), eng.cache(min(1, layers - 1))
    for a, b in zip(first, second):
        if a is None:
            continue
        step = (b.data_ptr() - a.data_ptr()) // a.element_size()
        views.append(torch.as_strided(a, (layers, a.shape[0], hi - lo, a.shape[2]), (step, *a.stride()), a.storage_offset() + lo * a.stride(1)))
    return views


def prepare(case, seed):
    kind, bits, L, H, Hk = case["kind"], case["bits"], case["layers"], case["heads"], case["kv_heads"]
    g = _generator(seed)
    s = dict(case=case, stream=_stream())
    fill = _Filler(g, seed, bits)
    if kind in ("layer", "decode", "rollout", "paged", "launchers"):
        ctx = _contexts(case, seed)
        B, steps = case["batch"], case.get("steps", 1)
        rows = (int(ctx.max()) + steps + 255) // 256 * 256
        s["q"] = _randn(g, L, B, H * D, scale=2.0)
        s["k"], s["v"] = _randn(g, L, B, Hk * D), _randn(g, L, B, Hk * D)
        s["out"] = torch.zeros_like(s["q"])
        s["start"] = [int(c) - 1 for c in ctx]
    if kind in ("layer", "decode", "rollout"):
        eng = s["eng"] = _engine(case, B, rows)
        for l in range(L):
            fill.fill(eng.cache(l))
        eng.set_positions(s["start"])
        if kind == "rollout":
            _set_producers(eng, g, L, rows)
            if bits == 0:                 # the fp16 path transforms q and k in place: the projections' output, kept aside
                s["q0"], s["k0"] = s["q"].clone(), s["k"].clone()
            s["tokens"] = torch.randint(0, 150_000, (steps, B), generator=g, device="cuda", dtype=torch.int32)
        s["rows"] = _row_views(eng, L, min(s["start"]), max(s["start"]) + steps)
    elif kind in ("paged", "launchers"):
        s["positions"] = torch.tensor(s["start"], dtype=torch.int32, device="cuda")
        kvp = Hk * D * 2 if bits == 0 else Hk * D * bits // 8
        lead = (L, B * rows // 16, 16) if kind == "paged" else (L, B, rows)
        s["cache"] = [torch.empty((*lead, kvp), dtype=torch.uint8, device="cuda") for _ in range(2)]
        if bits == 0:
            s["cache"] = [t.view(torch.float16) for t in s["cache"]] + [None, None]
        else:
            s["cache"] += [torch.empty((*lead, Hk), dtype=torch.float16, device="cuda") for _ in range(2)]
        fill.fill(s["cache"])
        s["rotation"] = kvcache.make_rotation(D, 42).cuda()
        if kind == "paged":
            order = np.random.Generator(np.random.Philox(int(seed) + 1)).permutation(B * rows // 16).astype(np.int32)
            s["table"] = torch.from_numpy(order.reshape(B, rows // 16)).cuda()
            s["scratch"] = torch.empty(kvcache.attention_workspace_floats(B, H, rows), dtype=torch.float32, device="cuda")
        else:
            s["scratch"] = torch.empty(B * H * rows, dtype=torch.float32, device="cuda")
        s["max_seq_len"] = rows
    elif kind == "single":
        rows = (case["ctx"] + case["steps"] + 255) // 256 * 256
        eng = s["eng"] = _engine(case, 1, rows)
        for l in range(L):
            fill.fill(eng.single_cache(l))
        s["q"] = _randn(g, L, H * D, scale=2.0)
        s["k"], s["v"] = _randn(g, L, Hk * D), _randn(g, L, Hk * D)
        s["out"] = torch.zeros_like(s["q"])
        at = slice(case["ctx"] - 1, case["ctx"] - 1 + case["steps"])
        s["rows"] = [t[at] for l in range(L) for t in eng.single_cache(l)[:2]]
        for t in s["rows"]:
            t.owner = eng                 # memory of the engine, not of torch: whoever holds the outputs holds the engine
    elif kind == "prompt":
        T = case["tokens"]
        eng = s["eng"] = _engine(case, 1, (T + 255) // 256 * 256)
        s["q"] = _randn(g, L, T, H * D, scale=2.0)
        s["k"], s["v"] = _randn(g, L, T, Hk * D), _randn(g, L, T, Hk * D)
        s["out"] = torch.zeros_like(s["q"])
        s["iota"] = torch.arange(T, device="cuda", dtype=torch.int32)
        if case["producers"]:
            _set_producers(eng, g, L, T)
            s["q0"], s["k0"] = s["q"].clone(), s["k"].clone()
        s["rows"] = _row_views(eng, L, 0, T)
    else:                                                   # group
        P, lo, hi = case["prompts"], case["t_min"], case["t_max"]
        s["lens"] = [lo + (hi - lo) * (i * 7 % P) // max(P - 1, 1) for i in range(P)]
        eng = s["eng"] = _engine(case, P * case["group"], (hi + 255) // 256 * 256)
        s["q"] = _randn(g, P, L, hi, H * D, scale=2.0)
        s["k"], s["v"] = _randn(g, P, L, hi, Hk * D), _randn(g, P, L, hi, Hk * D)
        s["out"] = torch.zeros_like(s["q"])
        s["iota"] = torch.arange(hi, device="cuda", dtype=torch.int32)
        _set_producers(eng, g, L, hi)
        s["q0"], s["k0"] = s["q"].clone(), s["k"].clone()   # the producers work in place: the projections' output, kept aside
        s["rows"] = _row_views(eng, L, 0, hi)
    if kind == "group":
        s["calls"] = [[(l, *(s[n][p, l, :T] for n in ("q", "k", "v", "out"))) for l in range(L)] for p, T in enumerate(s["lens"])]
    else:
        s["calls"] = [(l, *(s[n][l] for n in ("q", "k", "v", "out"))) for l in range(L)]
        if "cache" in s:
            s["layer_cache"] = [[None if t is None else t[l] for t in s["cache"]] for l in range(L)]
    return s


# ---------------------------------------------------------------- one pass

def _restore_projections(s):
    if "q0" in s:
        with torch.cuda.stream(s["stream"]):
            s["q"].copy_(s["q0"])
            s["k"].copy_(s["k0"])


def _run_layers(s):
    eng, st = s["eng"], s["stream"]
    for l, q, k, v, out in s["calls"]:
        eng.layer_step(l, q, k, v, out, stream=st)
    return {"out": s["out"], "rows": s["rows"]}


def _run_decode(s):
    eng = s["eng"]
    eng.set_positions(s["start"])
    for _ in range(s["case"]["steps"]):
        eng.decode_step(s["q"], s["k"], s["v"], s["out"], use_graph=True, stream=s["stream"])
    return {"out": s["out"], "rows": s["rows"], "positions": eng.positions()}


def _run_rollout(s):
    eng, st, steps = s["eng"], s["stream"], s["case"]["steps"]
    eng.set_positions(s["start"])
    eng.begin_generation(steps, -1)
    for i in range(steps):
        _restore_projections(s)
        eng.decode_step(s["q"], s["k"], s["v"], s["out"], use_graph=True, stream=st)
        eng.record_tokens(s["tokens"][i], i, stream=st)
        eng.check_stops(i, stream=st)
    tokens = np.array([eng.output(b)[0] for b in range(s["case"]["batch"])], dtype=np.int32)
    return {"out": s["out"], "rows": s["rows"], "positions": eng.positions(), "tokens": tokens}


def _run_single(s):
    eng, st, c = s["eng"], s["stream"], s["case"]
    eng.single_set_pos(c["ctx"] - 1)
    for _ in range(c["steps"]):
        for l, q, k, v, out in s["calls"]:
            eng.single_step(l, q, k, v, out, stream=st)
        eng.single_advance(stream=st)
    return {"out": s["out"], "rows": s["rows"]}


def _run_paged(s):
    c = s["case"]
    H, Hk, B, bits = c["heads"], c["kv_heads"], c["batch"], c["bits"]
    pages, st = s["max_seq_len"] // 16, s["stream"]
    for (l, q, k, v, out), (ck, cv, kn, vn) in zip(s["calls"], s["layer_cache"]):
        if bits:
            kvcache.tw_paged_turbo_append_attention_batch(out, q, k, v, ck, cv, kn, vn, s["rotation"], s["scratch"], s["positions"],
                                                          s["table"], pages, s["max_seq_len"], B, H, Hk, D, H * D, Hk * D, bits, stream=st)
        else:
            kvcache.tw_paged_kv_cache_write_batch(ck, cv, k, v, s["positions"], s["table"], pages, B, Hk * D, stream=st)
            kvcache.tw_paged_gqa_attention_batch(out, q, ck, cv, s["scratch"], s["positions"], s["table"], pages, s["max_seq_len"], B, H, Hk, D,
                                                 H * D, Hk * D, stream=st)
    return {"out": s["out"], "cache": [t for t in s["cache"] if t is not None]}


def _run_launchers(s):
    c = s["case"]
    H, Hk, B, bits, msl = c["heads"], c["kv_heads"], c["batch"], c["bits"], s["max_seq_len"]
    pos, st = s["positions"], s["stream"]
    for (l, q, k, v, out), (ck, cv, kn, vn) in zip(s["calls"], s["layer_cache"]):
        if bits:
            kvcache.launch_turbo_kv_quantize_batch(ck, kn, k, s["rotation"], pos, msl, B, Hk, D, Hk * D, bits, stream=st)
            kvcache.launch_turbo_kv_quantize_batch(cv, vn, v, s["rotation"], pos, msl, B, Hk, D, Hk * D, bits, stream=st)
            kvcache.launch_turbo_gqa_attention_batch(out, q, ck, cv, kn, vn, s["rotation"], s["scratch"], pos, msl, B, H, Hk, D,
                                                     H * D, Hk * D, bits, stream=st)
        else:
            kvcache.launch_kv_cache_write_batch(ck, cv, k, v, pos, msl, B, Hk * D, stream=st)
            kvcache.launch_gqa_attention_batch(out, q, ck, cv, s["scratch"], pos, msl, B, H, Hk, D, H * D, Hk * D, stream=st)
    return {"out": s["out"], "cache": [t for t in s["cache"] if t is not None]}


def _run_prompt(s):
    eng, st = s["eng"], s["stream"]
    _restore_projections(s)
    for l, q, k, v, out in s["calls"]:
        eng.prompt_layer(l, 0, q, k, v, out, s["iota"], stream=st)
    return {"out": s["out"], "rows": s["rows"]}


def _run_group(s):
    eng, st, c = s["eng"], s["stream"], s["case"]
    _restore_projections(s)
    for p, T in enumerate(s["lens"]):
        first = p * c["group"]
        for l, q, k, v, out in s["calls"][p]:
            eng.prompt_layer(l, first, q, k, v, out, s["iota"], stream=st)
        eng.broadcast_prefix(first, first + 1, first + c["group"], T, stream=st)
    return {"out": s["out"], "rows": s["rows"]}


_RUN = {"layer": _run_layers, "decode": _run_decode, "rollout": _run_rollout, "single": _run_single, "paged": _run_paged,
        "launchers": _run_launchers, "prompt": _run_prompt, "group": _run_group}


def run(state):
    return _RUN[state["case"]["kind"]](state)


# ---------------------------------------------------------------- what a pass cannot do without

def work(case):
    """Cache bytes once per step (not once per query head), the appended rows, q, k, v and out; 4 * 128 operations for
    every (query head, attended token)."""
    kind, L, H, Hk, head = case["kind"], case["layers"], case["heads"], case["kv_heads"], HEAD_BYTES[case["bits"]]

    def rows(n):                          # n new tokens of a layer: q, k, v read, out and the cache rows written
        return n * (2 * H * D * 2 + 2 * Hk * D * 2 + 2 * Hk * head)

    if kind in ("prompt", "group"):
        if kind == "prompt":
            lens, copies = [case["tokens"]], 0
        else:
            P, lo, hi = case["prompts"], case["t_min"], case["t_max"]
            lens, copies = [lo + (hi - lo) * (i * 7 % P) // max(P - 1, 1) for i in range(P)], case["group"] - 1
        return {"bytes": L * sum(rows(t) + copies * t * 2 * Hk * head for t in lens),
                "flops": L * sum(4.0 * D * H * t * (t + 1) / 2 for t in lens)}
    steps = case.get("steps", 1)
    if kind == "single":
        batch, ctx = 1, case["ctx"]
    else:
        batch, ctx = case["batch"], float(_contexts(case, 0).mean())
    tokens = batch * sum(ctx + i for i in range(steps))
    return {"bytes": L * (tokens * 2 * Hk * head + steps * rows(batch)), "flops": L * 4.0 * D * H * tokens}


def tolerance(case):
    """Against the same path in 64 bits (contexts of 3000 to 4097 tokens, prompts of 1500): 2.1e-4 on the fp16 cache, which
    is the rounding of the fp16 output; 3.3e-4 at 4 bit, 2.1e-4 at 2 bit; largest single difference 1.4e-3 of the root mean
    square.  Codes, positions and tokens are whole numbers and stay the same."""
    return {"rel": 1.3e-3 if case["bits"] == 4 else 8.5e-4, "max": 6e-3}
