"""The automatic choice between the forms of a compressed decode step (one launch, one launch with a sequence's context
shared by workgroups, three launches) against the forms themselves, timed on the GPU at hand: the choice rests on
rates and fixed costs measured on one device (plan_constants in kv_decode_fused.hip), and this is the check that they
still describe the device the library runs on.  Each form runs graph-replayed steps of a few layers, one after the other; the automatic
choice must be within 5 % of the faster forced form (medians of several timings).  The same for a step whose layers may go into one
launch: as fast as layer by layer, and as fast as any other number of heads to a workgroup."""
import random
import statistics

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

D = 128


def _time_steps(eng, q, k, v, out, start, steps, stream):
    import torch
    eng.set_positions([start] * q.shape[1])
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    with torch.cuda.stream(stream):
        eng.decode_step(q, k, v, out, use_graph=True, stream=stream)        # capture (or replay) outside the timing
        e0.record(stream)
        for _ in range(steps):
            eng.decode_step(q, k, v, out, use_graph=True, stream=stream)
        e1.record(stream)
    stream.synchronize()
    return e0.elapsed_time(e1) / steps


@pytest.mark.parametrize("G,ctx,bits,H", [(64, 8192, 4, 16), (16, 8192, 4, 16), (96, 8192, 2, 16), (128, 512, 4, 16), (16, 4096, 2, 32)])
def test_automatic_choice_is_the_faster_form(G, ctx, bits, H):
    import torch
    from triebwerk_amd import Engine, kvcache
    L, Hk, steps, reps = 4, 8, 12, 5
    msl = ctx + (reps * 3 + 2) * (steps + 1) + 64
    msl = (msl + 255) // 256 * 256
    eng = Engine(max_seq_len=msl, kv_bits=bits)
    eng.set_shape(L, H, Hk, D)
    eng.alloc_batch(G, msl)
    gt = torch.Generator(device="cuda"); gt.manual_seed(3)
    for l in range(L):
        c = eng.cache(l)
        for i in range(2):
            c[i].view(torch.int32).copy_(torch.randint(-2 ** 31, 2 ** 31 - 1, tuple(c[i].view(torch.int32).shape), generator=gt,
                                                      device="cuda", dtype=torch.int32))
        for i in (2, 3):
            c[i].copy_((11.3 + 0.7 * torch.randn(c[i].shape, generator=gt, device="cuda")).to(torch.float16))
    q = torch.randn((L, G, H * D), generator=gt, device="cuda", dtype=torch.float16)
    k = torch.randn((L, G, Hk * D), generator=gt, device="cuda", dtype=torch.float16)
    v = torch.randn((L, G, Hk * D), generator=gt, device="cuda", dtype=torch.float16)
    out = torch.zeros_like(q)
    stream = torch.cuda.Stream()
    times = {4: [], 1: [], 2: []}
    try:
        for rep in range(reps):
            for mode in times:              # automatic layer by layer, one launch (shared where the library would share), three launches
                kvcache.set_decode_fused(mode)
                # a change of mode does not invalidate the captured step: other buffers make the engine capture again
                times[mode].append(_time_steps(eng, q, k, v, out, ctx - 1, steps, stream))
                assert "decode_layers_kernel" not in kvcache.last_scan_kernel()
                q = q.clone()
    finally:
        kvcache.set_decode_fused(0)
    auto, one, three = (statistics.median(times[m]) for m in times)
    print(f"plan check G={G} ctx={ctx} bits={bits}: automatic {auto:.4f} ms, one launch {one:.4f}, three launches {three:.4f}", flush=True)
    assert auto <= 1.05 * min(one, three), (auto, one, three)


def _ragged(G, lo, hi):
    return random.Random(G).sample(range(lo, hi + 1), G)


@pytest.mark.parametrize("bits,H,Hk,L,lens", [
    (4, 16, 8, 28, [613] * 4), (4, 16, 8, 12, [8192] * 64), (2, 32, 8, 12, [4097] * 16), (4, 16, 8, 2, [16000]), (2, 16, 8, 3, [8192] * 3),
    (4, 8, 2, 28, [300, 4000] * 8), (4, 8, 8, 28, [7000] + [100] * 10), (0, 16, 8, 28, [133]), (0, 16, 8, 2, [7000]), (0, 16, 8, 4, [8192] * 12),
    (0, 16, 8, 2, _ragged(83, 877, 8777)), (0, 8, 8, 4, _ragged(116, 538, 5383)), (0, 32, 8, 4, [7880] + [788] * 43)])
def test_every_layer_in_one_launch_is_no_slower(bits, H, Hk, L, lens):
    import torch
    from triebwerk_amd import Engine, kvcache
    G, steps, reps = len(lens), 8, 7
    msl = (max(lens) + steps + 2 + 255) // 256 * 256
    eng = Engine(max_seq_len=msl, kv_bits=bits)
    eng.set_shape(L, H, Hk, D)
    eng.alloc_batch(G, msl)
    gt = torch.Generator(device="cuda"); gt.manual_seed(4)
    for l in range(L):
        for i, c in enumerate(eng.cache(l)):
            if c is None: continue
            if bits and i < 2: c.copy_(torch.randint(0, 256, c.shape, generator=gt, device="cuda", dtype=torch.uint8))
            else: c.copy_(((11.3 if bits else 0) + 0.7 * torch.randn(c.shape, generator=gt, device="cuda")).to(torch.float16))
    q = torch.randn((L, G, H * D), generator=gt, device="cuda", dtype=torch.float16)
    k, v = (torch.randn((L, G, Hk * D), generator=gt, device="cuda", dtype=torch.float16) for _ in range(2))
    out = torch.zeros_like(q)
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()                    # the inputs were made on the default stream
    forms = [(0, 0), (4, 0)] + ([(0, h) for h in (2, 4, 8) if Hk % h == 0 and H // Hk * h <= 16] if bits else [])
    times, names = {f: [] for f in forms}, {}
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    try:
        for rep in range(reps):
            for form in random.Random(rep).sample(forms, len(forms)):       # (layers apart or not, KV heads to a workgroup)
                kvcache.set_decode_fused(form[0]); kvcache.set_fused_shape(form[1], 0)
                eng.set_positions([n - 1 for n in lens])
                with torch.cuda.stream(stream):
                    eng.decode_step(q, k, v, out, use_graph=True, stream=stream)          # captures where the form is another
                    e0.record(stream)
                    for _ in range(steps):
                        eng.decode_step(q, k, v, out, use_graph=True, stream=stream)
                    e1.record(stream)
                stream.synchronize()
                names[form] = kvcache.last_scan_kernel()
                times[form].append(e0.elapsed_time(e1) / steps / L * 1e3)
    finally:
        kvcache.set_decode_fused(0); kvcache.set_fused_shape(0, 0)
    us = {f: min(t) for f, t in times.items()}
    print(f"all layers G={G} longest={max(lens)} bits={bits} H={H} Hk={Hk} L={L}: " +
          "; ".join(f"{f}: {t:.2f} us {names[f]}" for f, t in us.items()), flush=True)
    assert "decode_layers_kernel" not in names[4, 0] and "every layer" not in names[4, 0]
    assert us[0, 0] <= 1.10 * min(us.values()), us
