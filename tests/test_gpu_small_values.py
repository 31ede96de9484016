"""Values far below one through the forms of a compressed step: what they rotate back keeps its 32 bits however small it is.  One token a
sequence, so that attention passes the value on as it lies in the cache and the rotation back is all there is to see."""
import numpy as np
import pytest

import gen
from test_gpu_parity import D, dev, host

pytestmark = pytest.mark.gpu

SIZES = [1.0, 1e-2, 1e-3, 1e-4, 1e-5]
SCALE = {4: np.float32(19.391284942626953), 2: np.float32(25.46918296813965)}      # the scans hold fp16(scale * centroid)


def _check(oracle, got, codes, norms, rot, H, bits, what):
    """got (G, H * D): what attention over one token with these codes and norms (G, Hk) gives"""
    G, Hk = norms.shape
    codes = codes.reshape(G, Hk, D * bits // 8)
    codes = np.stack([(codes >> (bits * i)) & (2 ** bits - 1) for i in range(8 // bits)], -1).reshape(G, Hk, D)
    centroids = (SCALE[bits] * oracle.centroids(bits)).astype(np.float16).astype(np.float64) / float(SCALE[bits])
    o = centroids[codes] * norms.astype(np.float64)[..., None]
    right = np.repeat(o @ rot.astype(np.float64), H // Hk, axis=1).astype(np.float16).reshape(G, H * D)
    # An output in fp32 is off by the value's rounding and those of the sums (less than 3e-7 of the vector's size): the half nearest to it
    # is another one where the exact value lies that near to the middle of two, which for steps of 2^-11 and more is at most one in 500
    # in the mean over the coordinates, and one in 100 with a margin.  With remainders in subnormal halves it was one in five.
    differ = float(np.mean(got != right))
    print(f"small values: bits={bits} {what}: {differ:.4f} of the halves are not the nearest", flush=True)
    assert differ <= 0.01


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("bits,form", [(4, "launcher"), (4, "paged"), (2, "launcher"), (2, "paged"), (4, "one head per wave"),
                                       (4, "one launch"), (2, "one launch")])
def test_the_merge_keeps_small_values(oracle, rotation_fixture, bits, form, size):
    import torch
    from triebwerk_amd import kvcache as kv
    G, H, Hk, pages = 40, 16, 8, 40
    msl = 16 * pages
    r = gen.rng(9700 + bits)
    rot = rotation_fixture
    c = [np.zeros((G, msl, Hk * D * bits // 8), np.uint8) for _ in range(2)] + [np.zeros((G, msl, Hk), np.float16) for _ in range(2)]
    for i in range(2): c[i][:, 0] = r.integers(0, 256, c[i][:, 0].shape, dtype=np.uint8)
    c[2][:, 0] = 11.3
    c[3][:, 0] = (size * (11.3 + 0.7 * r.standard_normal((G, Hk)))).astype(np.float16)
    q, pos = gen.normal_f16(r, (G, H * D)), np.zeros(G, np.int32)
    out = torch.zeros((G, H * D), dtype=torch.float16, device="cuda")
    scratch = torch.zeros(max(G * H * msl, kv.attention_workspace_floats(G, H, msl)), dtype=torch.float32, device="cuda")
    one = form == "one launch"
    if one:
        kv.set_fused_shape(2, 0)
    else:
        kv.set_decode_fused(2)                           # three launches
        kv.set_num_splits(2)
    if form == "one head per wave": kv.set_attention_variant(3)
    try:
        if form == "paged":
            table = dev(np.arange(G * pages, dtype=np.int32).reshape(G, pages))
            kv.tw_paged_turbo_gqa_attention_batch(out, dev(q), *map(dev, c), dev(rot), scratch, dev(pos), table, pages, msl, G, H, Hk, D, H * D, Hk * D, bits)
        else:
            kv.launch_turbo_gqa_attention_batch(out, dev(q), *map(dev, c), dev(rot), scratch, dev(pos), msl, G, H, Hk, D, H * D, Hk * D, bits)
        torch.cuda.synchronize()
    finally:
        kv.set_decode_fused(0); kv.set_num_splits(0); kv.set_attention_variant(0); kv.set_fused_shape(0, 0)
    assert kv.last_scan_kernel() == ("attention_mfma_kernel" if form == "one head per wave" else "attention_pair_kernel" if not one
                                     else "decode_fused_kernel, two KV heads per wave, attention alone")
    _check(oracle, host(out), c[1][:, 0], c[3][:, 0], rot, H, bits, f"{form} size={size}")


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("bits,H,Hk,hkw,shares", [(4, 16, 8, 2, 1), (4, 16, 8, 1, 1), (2, 32, 8, 8, 1), (4, 16, 8, 2, 2), (2, 8, 8, 1, 4), (4, 16, 8, 2, 0), (2, 32, 8, 4, 0)])
def test_a_step_keeps_small_values(oracle, bits, H, Hk, hkw, shares, size):
    """The first token of empty caches in one launch, also with the (one-token) context shared, and in one launch of every layer
    (shares 0)."""
    import torch
    from triebwerk_amd import Engine, kvcache as kv
    L, G, msl = 4, 20, 640
    r = gen.rng(9800 + bits + H + hkw)
    eng = Engine(max_seq_len=msl, kv_bits=bits)
    eng.set_shape(L, H, Hk, D)
    eng.alloc_batch(G, msl)
    rot = host(eng.rotation())
    eng.set_positions([0] * G)
    q, k = gen.normal_f16(r, (L, G, H * D)), gen.normal_f16(r, (L, G, Hk * D))
    v = (size * r.standard_normal((L, G, Hk * D))).astype(np.float16)
    out = torch.zeros((L, G, H * D), dtype=torch.float16, device="cuda")
    kv.set_fused_shape(hkw, shares)
    if shares: kv.set_decode_fused(1)
    try:
        eng.decode_step(dev(q), dev(k), dev(v), out)
        torch.cuda.synchronize()
    finally:
        kv.set_decode_fused(0); kv.set_fused_shape(0, 0)
    name = kv.last_scan_kernel()
    assert ("decode_fused_kernel" if shares else "decode_layers_kernel") in name and ("shared" in name) == (shares > 1), name
    for l in range(L):
        c = [host(t)[:, 0] for t in eng.cache(l)]
        _check(oracle, host(out[l]), c[1], c[3], rot, H, bits, f"step hkw={hkw} shares={shares} size={size} layer {l}")
