"""The compressed decode step with every layer in one launch (decode_layers_kernel) against the same step taken layer by
layer, whose kernels the other tests hold against the oracle: the caches bit for bit, the outputs within the parity
tolerance (another order of additions and one fp16 rounding).  Contexts at the edges of a tile of 32 tokens and of the
parts a sequence is cut into, ragged batches, every GQA group and number of heads per workgroup, the producers."""
import numpy as np
import pytest

import gen
from test_gpu_parity import D, TOL, assert_bytes_equal, dev, host, rel_err, rope_tables

pytestmark = pytest.mark.gpu


def _pair(bits, H, Hk, L, G, msl, producers):
    import torch
    from triebwerk_amd import Engine
    gt = torch.Generator(device="cuda"); gt.manual_seed(bits * 1000 + H + Hk + G)
    engines = []
    for _ in range(2):
        e = Engine(max_seq_len=msl, kv_bits=bits)
        e.set_shape(L, H, Hk, D)
        e.alloc_batch(G, msl)
        engines.append(e)
    for l in range(L):
        for i, (a, b) in enumerate(zip(engines[0].cache(l), engines[1].cache(l))):
            if a is None: continue
            if bits == 0: a.copy_(torch.randn(a.shape, generator=gt, device="cuda").to(torch.float16))
            elif i < 2: a.copy_(torch.randint(0, 256, a.shape, generator=gt, device="cuda", dtype=torch.uint8))
            else: a.copy_((11.3 + 0.7 * torch.randn(a.shape, generator=gt, device="cuda")).to(torch.float16))
            b.copy_(a)
    if producers:
        w = [(1 + 0.2 * torch.randn((L, D), generator=gt, device="cuda")).to(torch.float16) for _ in range(2)]
        ct, st = (torch.from_numpy(t).cuda() for t in rope_tables(msl, D))
        for e in engines:
            e.set_producers(1, w[0], w[1], 1e-6, False, ct, st, D)
    q = 2 * torch.randn((L, G, H * D), generator=gt, device="cuda", dtype=torch.float16)
    k, v = (torch.randn((L, G, Hk * D), generator=gt, device="cuda", dtype=torch.float16) for _ in range(2))
    torch.cuda.synchronize()
    return engines, q, k, v


@pytest.mark.parametrize("producers", [False, True])
@pytest.mark.parametrize("bits,H,Hk,L,lens,hkw,form", [
    (4, 16, 8, 3, [1, 2, 31, 32, 33, 63, 64, 65, 97], 0, "KV heads"),
    (2, 16, 8, 28, [1], 2, "two KV heads"),
    (4, 16, 8, 28, [2049, 31], 2, "two KV heads in eight"),
    (2, 8, 8, 28, [2047], 2, "two KV heads in eight"),
    (4, 32, 8, 36, [1027], 2, "two KV heads in eight"),
    (2, 8, 4, 28, [129] * 11, 2, "two KV heads in four"),
    (4, 8, 2, 5, [1, 127, 128, 129, 161] * 20, 2, "two KV heads in four"),
    (4, 12, 6, 28, [70, 64, 7] * 2, 0, "two KV heads"),
    (4, 16, 8, 28, [33, 64, 65, 31, 1] * 4, 8, "eight KV heads"),
    (2, 16, 8, 7, [100] * 43, 8, "eight KV heads"),
    (4, 8, 8, 9, [1, 500, 511, 512, 513] * 9, 8, "eight KV heads"),
    (2, 16, 16, 4, [161, 32] * 3, 8, "eight KV heads"),
    (4, 32, 8, 36, [65] * 7, 4, "four KV heads"),
    (2, 32, 8, 11, [300, 31, 32, 33, 1] * 9, 4, "four KV heads"),
    (2, 12, 12, 5, [95, 96, 97] * 13, 4, "four KV heads"),
])
def test_all_layers_in_one_launch(bits, H, Hk, L, lens, hkw, form, producers):
    import torch
    from triebwerk_amd import kvcache
    G, msl = len(lens), (max(lens) + 8 + 31) // 32 * 32
    engines, q, k, v = _pair(bits, H, Hk, L, G, msl, producers)
    outs = [torch.zeros_like(q) for _ in range(2)]
    for e in engines:
        e.set_positions([n - 1 for n in lens])
    for step in range(3):                          # eager, captured, replayed
        kvcache.set_fused_shape(hkw, 0)
        try:
            engines[0].decode_step(q, k, v, outs[0], use_graph=step > 0)
        finally:
            kvcache.set_fused_shape(0, 0)
        if step == 0:
            name = kvcache.last_scan_kernel()
            print(f"all layers: bits={bits} H={H} Hk={Hk} L={L} G={G}: {name}", flush=True)
        for l in range(L):
            engines[1].layer_step(l, q[l], k[l], v[l], outs[1][l])
        torch.cuda.synchronize()
        engines[1].set_positions([n + step for n in lens])
        assert engines[0].positions().tolist() == [n + step for n in lens]
        got, want = (host(o).reshape(L * G, H * D) for o in outs)
        assert rel_err(got, want) <= TOL, f"step {step}"
    assert "decode_layers_kernel" in name and form in name, name
    _same_caches(engines, L)


def _same_caches(engines, L):
    import torch
    for l in range(L):
        for i, (a, b) in enumerate(zip(engines[0].cache(l), engines[1].cache(l))):
            assert a is None or torch.equal(a, b), f"layer {l} array {i}"


@pytest.mark.parametrize("producers", [False, True])
@pytest.mark.parametrize("H,Hk,L,lens", [
    (16, 8, 28, [1]), (16, 8, 28, [7, 8, 9, 1]), (32, 8, 12, [500] * 3), (16, 8, 2, [2049]), (8, 8, 4, [63, 64, 65] * 30),
    (16, 16, 5, [1, 300, 17] * 4), (64, 8, 3, [130, 5]), (24, 8, 4, [257] * 9), (16, 8, 28, [129] * 40),
])
def test_all_layers_at_once_fp16(H, Hk, L, lens, producers):
    """The same on the fp16 cache: every layer's rows in one scan, with and without the contexts cut into pieces."""
    import torch
    from triebwerk_amd import kvcache
    G, msl = len(lens), (max(lens) + 8 + 31) // 32 * 32
    engines, q, k, v = _pair(0, H, Hk, L, G, msl, producers)
    outs = [torch.zeros_like(q) for _ in range(2)]
    for e in engines:
        e.set_positions([n - 1 for n in lens])
    for step in range(3):                          # eager, captured, replayed
        args = [(q.clone(), k.clone()) if step == 0 else args[i] for i in range(2)]     # (the producers work in place)
        for (qi, ki) in args:
            qi.copy_(q); ki.copy_(k)
        torch.cuda.synchronize()
        engines[0].decode_step(args[0][0], args[0][1], v, outs[0], use_graph=step > 0)
        if step == 0:
            name = kvcache.last_scan_kernel()
        for l in range(L):
            engines[1].layer_step(l, args[1][0][l], args[1][1][l], v[l], outs[1][l])
        torch.cuda.synchronize()
        engines[1].set_positions([n + step for n in lens])
        assert engines[0].positions().tolist() == [n + step for n in lens]
        got, want = (host(o).reshape(L * G, H * D) for o in outs)
        assert rel_err(got, want) <= TOL, f"step {step}"
        assert torch.equal(args[0][0], args[1][0]) and torch.equal(args[0][1], args[1][1]), f"step {step}: q or k"
    assert name == "attention_rows_kernel, every layer"
    _same_caches(engines, L)


def test_outputs_over_inputs_go_layer_by_layer():
    """An output that lies over the next layer's queries: the layers depend on each other and run one after the other."""
    import torch
    from triebwerk_amd import kvcache
    bits, H, Hk, L, G, msl = 4, 16, 8, 28, 4, 96
    engines, q, k, v = _pair(bits, H, Hk, L, G, msl, False)
    chain = torch.zeros((L + 1, G, H * D), dtype=torch.float16, device="cuda")
    chain[0] = q[0]
    want = chain.clone()
    for e in engines:
        e.set_positions([40] * G)
    torch.cuda.synchronize()
    engines[0].decode_step(chain[:L], k, v, chain[1:])
    assert "decode_layers_kernel" not in kvcache.last_scan_kernel()
    for l in range(L):
        engines[1].layer_step(l, want[l], k[l], v[l], want[l + 1])
    torch.cuda.synchronize()
    assert torch.equal(chain, want) and chain[L].abs().sum() > 0


@pytest.mark.parametrize("bits", [4, 2])
def test_layers_without_room_for_partials_stay_in_fp32(oracle, bits):
    """264 sequences of at most 256 rows: a layer by itself takes three launches there, which without room for partials are the
    kernel that keeps p * norm in fp32, and V norms past 65504 / 2^5 give the oracle's output."""
    import torch
    from triebwerk_amd import Engine, kvcache
    H, Hk, L, G, msl = 16, 8, 2, 264, 256
    r = gen.rng(5600 + bits)
    eng = Engine(max_seq_len=msl, kv_bits=bits)
    eng.set_shape(L, H, Hk, D)
    eng.alloc_batch(G, msl)
    pos = np.full(G, msl - 1, np.int32)
    eng.set_positions(pos)
    rot = host(eng.rotation())
    q = gen.normal_f16(r, (L, G, H * D)); k = gen.normal_f16(r, (L, G, Hk * D)); v = gen.normal_f16(r, (L, G, Hk * D))
    caches = []
    for l in range(L):
        c = [r.integers(0, 256, (G, msl, Hk * D * bits // 8), dtype=np.uint8) for _ in range(2)]
        c[0][:] = c[0][:, :1]
        c.append(np.ascontiguousarray(np.broadcast_to((5 + 8 * (np.arange(msl) // 32)).astype(np.float16)[None, :, None], (G, msl, Hk))))
        c.append((4000 + 300 * r.standard_normal((G, msl, Hk))).astype(np.float16))
        for t, x in zip(eng.cache(l), c):
            t.copy_(dev(x))
        caches.append(c)
    out = torch.zeros((L, G, H * D), dtype=torch.float16, device="cuda")
    eng.decode_step(dev(q), dev(k), dev(v), out)
    torch.cuda.synchronize()
    for l, c in enumerate(caches):
        oracle.turbo_kv_quantize_batch(c[0], c[2], k[l], rot, pos, msl, G, Hk, D, Hk * D, bits)
        oracle.turbo_kv_quantize_batch(c[1], c[3], v[l], rot, pos, msl, G, Hk, D, Hk * D, bits)
        want = np.zeros((G, H * D), np.float16)
        oracle.turbo_gqa_attention_batch(want, q[l], *c, rot, pos, msl, G, H, Hk, D, H * D, Hk * D, bits)
        assert rel_err(host(out[l]), want) <= TOL, f"layer {l}"
    assert kvcache.last_scan_kernel() == "attention_valu_kernel"


@pytest.mark.parametrize("bits", [4, 2, 0])
@pytest.mark.parametrize("hook,value", [("set_decode_fused", 2), ("set_decode_fused", 4), ("set_attention_variant", 3), ("set_num_splits", 3)])
def test_the_hooks_hold_in_an_engines_step(bits, hook, value):
    """What a hook forces is a layer's kernels: with one set, the step is the layers one by one, bit for bit."""
    import torch
    from triebwerk_amd import kvcache
    H, Hk, L, lens, msl = 16, 8, 4, [300, 77, 1200], 2048
    G = len(lens)
    engines, q, k, v = _pair(bits, H, Hk, L, G, msl, False)
    outs = [torch.zeros_like(q) for _ in range(2)]
    for e in engines:
        e.set_positions([n - 1 for n in lens])
    getattr(kvcache, hook)(value)
    try:
        engines[0].decode_step(q, k, v, outs[0], use_graph=True)
        name = kvcache.last_scan_kernel()
        for l in range(L):
            engines[1].layer_step(l, q[l], k[l], v[l], outs[1][l])
        torch.cuda.synchronize()
        assert name == kvcache.last_scan_kernel()
    finally:
        getattr(kvcache, hook)(0)
    assert torch.equal(*outs)
    _same_caches(engines, L)


@pytest.mark.parametrize("norm,biased,rope_dim", [(True, False, 0), (True, True, 0), (False, False, 128), (False, False, 16),
                                                  (True, True, 64), (True, False, 48)])
@pytest.mark.parametrize("bits", [4, 2, 0])
def test_producers_of_every_layer_in_one_launch(oracle, bits, norm, biased, rope_dim):
    """RMSNorm or RoPE alone, biased weights, a rotary part of the head, per-layer weights: against the oracle, from empty caches on."""
    import torch
    from triebwerk_amd import Engine, kvcache
    L, H, Hk, G, msl, steps = 3, 16, 8, 5, 48, 3
    q_dim, kv_dim = H * D, Hk * D
    r = gen.rng(5800 + bits + rope_dim + 2 * norm + biased)
    eng = Engine(max_seq_len=msl, kv_bits=bits)
    eng.set_shape(L, H, Hk, D)
    eng.alloc_batch(G, msl)
    pos = np.array([0, 3, 30, 31, 41], np.int32)
    eng.set_positions(pos)
    rot = host(eng.rotation()) if bits else None
    w = [((0.0 if biased else 1.0) + 0.2 * r.standard_normal((L, D))).astype(np.float16) for _ in range(2)]
    tables = rope_tables(msl, rope_dim) if rope_dim else ()
    d_w, d_tables = [dev(x) for x in w] if norm else [None] * 2, [dev(t) for t in tables] if rope_dim else [None] * 2
    eng.set_producers(1, *d_w, 1e-6, biased, *d_tables, rope_dim)
    width = kv_dim * bits // 8 if bits else kv_dim
    caches = [[np.zeros((G, msl, width), np.uint8 if bits else np.float16) for _ in range(2)] +
              ([np.zeros((G, msl, Hk), np.float16) for _ in range(2)] if bits else []) for _ in range(L)]
    out = torch.zeros((L, G, q_dim), dtype=torch.float16, device="cuda")
    for step in range(steps):
        q = gen.normal_f16(r, (L, G, q_dim)); k = gen.normal_f16(r, (L, G, kv_dim)); v = gen.normal_f16(r, (L, G, kv_dim))
        eng.decode_step(dev(q), dev(k), dev(v), out)
        torch.cuda.synchronize()
        assert "decode_layers_kernel" in kvcache.last_scan_kernel() or kvcache.last_scan_kernel() == "attention_rows_kernel, every layer"
        got = host(out)
        for l, c in enumerate(caches):
            want, ql, kl = np.zeros((G, q_dim), np.float16), q[l].copy(), k[l].copy()
            if norm: oracle.qk_norm_batch(ql, kl, w[0][l], w[1][l], H, Hk, D, G, 1e-6, q_dim, kv_dim, biased)
            if rope_dim: oracle.rope_batch(ql, kl, *tables, pos, msl, G, H, Hk, D, q_dim, kv_dim, rope_dim)
            if bits == 0:
                oracle.kv_cache_write_batch(*c, kl, v[l], pos, msl, G, kv_dim)
                oracle.gqa_attention_batch(want, ql, *c, pos, msl, G, H, Hk, D, q_dim, kv_dim)
            else:
                oracle.turbo_kv_quantize_batch(c[0], c[2], kl, rot, pos, msl, G, Hk, D, kv_dim, bits)
                oracle.turbo_kv_quantize_batch(c[1], c[3], v[l], rot, pos, msl, G, Hk, D, kv_dim, bits)
                oracle.turbo_gqa_attention_batch(want, ql, *c, rot, pos, msl, G, H, Hk, D, q_dim, kv_dim, bits)
            assert rel_err(got[l], want) <= TOL, f"step {step} layer {l}"
        pos += 1
    for l, c in enumerate(caches):
        for got, want, what in zip(eng.cache(l), c, ("K", "V", "K norms", "V norms")):
            assert_bytes_equal(host(got), want, f"layer {l} {what}")


@pytest.mark.parametrize("bits", [4, 2, 0])
@pytest.mark.parametrize("why", ["producers in launches of their own", "unaligned k"])
def test_what_one_launch_does_not_take_goes_layer_by_layer(bits, why):
    import torch
    from triebwerk_amd import kvcache
    H, Hk, L, lens, msl = 16, 8, 4, [70, 64, 7], 96
    G = len(lens)
    engines, q, k, v = _pair(bits, H, Hk, L, G, msl, False)
    outs = [torch.zeros_like(q) for _ in range(2)]
    if why == "unaligned k":
        flat = torch.zeros(k.numel() + 8, dtype=torch.float16, device="cuda")
        flat[2:2 + k.numel()].copy_(k.view(-1))
        k = flat[2:2 + k.numel()].view(k.shape)
    else:
        w = [torch.full((L, D), 1.25, dtype=torch.float16, device="cuda") for _ in range(2)]
        for e in engines:
            e.set_producers(2, *w)
    ins = [(q.clone(), k if why == "unaligned k" else k.clone()) for _ in range(2)]       # (the producers work in place)
    for e in engines:
        e.set_positions([n - 1 for n in lens])
    torch.cuda.synchronize()
    engines[0].decode_step(*ins[0], v, outs[0])
    name = kvcache.last_scan_kernel()
    assert "decode_layers_kernel" not in name and "every layer" not in name, name
    for l in range(L):
        engines[1].layer_step(l, ins[1][0][l], ins[1][1][l], v[l], outs[1][l])
    torch.cuda.synchronize()
    assert torch.equal(*outs) and outs[0].abs().sum() > 0
    _same_caches(engines, L)


@pytest.mark.parametrize("bits", [4, 2, 0])
def test_a_step_of_every_layer_captures_nothing_itself(capfd, bits):
    """With use_graph the few launches of all layers are issued as they are: nothing is captured for them, so inside a caller's capture
    nothing fails, and the caller's graph replays them."""
    import torch
    from triebwerk_amd import kvcache
    H, Hk, L, lens, msl = 16, 8, 6, [300, 77, 120], 512
    G = len(lens)
    engines, q, k, v = _pair(bits, H, Hk, L, G, msl, False)
    outs = [torch.zeros_like(q) for _ in range(2)]
    for e in engines:
        e.set_positions([n - 1 for n in lens])
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    capfd.readouterr()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream, capture_error_mode="relaxed"):
        engines[0].decode_step(q, k, v, outs[0], use_graph=True, stream=stream)
    assert "FAILED" not in capfd.readouterr().err
    assert engines[0].graph_state() == 1
    assert ("decode_layers_kernel" if bits else "attention_rows_kernel, every layer") in kvcache.last_scan_kernel()
    for step in range(3):
        graph.replay()
        for l in range(L):
            engines[1].layer_step(l, q[l], k[l], v[l], outs[1][l])
        torch.cuda.synchronize()
        engines[1].set_positions([n + step for n in lens])
        assert engines[0].positions().tolist() == [n + step for n in lens]
        got, want = (host(o).reshape(L * G, H * D) for o in outs)
        assert rel_err(got, want) <= TOL, f"step {step}"
        outs[0].zero_()
    _same_caches(engines, L)
