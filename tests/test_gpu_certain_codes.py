"""Codes decided from fp16 matrix sums where those are certain and by the fp32 chain where they are not: the oracle's bytes for vectors
whose rotated coordinates lie on the boundaries between buckets, that are zero, tiny or at the end of the fp16 range, and under
rotations that are no rotations (scaled rows, two equal rows).  The prompt's append in tiles of one stream and of two, the
step of one layer alone and with its context shared."""
import numpy as np
import pytest

import gen
from test_gpu_parity import D, assert_bytes_equal, dev, host, kv  # noqa: F401

pytestmark = pytest.mark.gpu


def _matrix(rotation, kind):
    r = rotation.astype(np.float32).copy()
    if kind == "scaled": r *= np.linspace(0.05, 3.0, D, dtype=np.float32)[:, None]
    if kind == "equal rows": r[1::2] = r[::2]
    return r.astype(rotation.dtype)


BOUNDS = {4: [0.02284, 0.04619, 0.07068, 0.09715, 0.12701], 2: [0.08677, 0.0]}      # between buckets, of unit vectors


def _hard_rows(r, rotation, n, heads, bits):
    """A third random; a third that the rotation takes to unit vectors with half of their coordinates on boundaries, but for the halves'
    rounding; the rest zero, tiny, large or of one coordinate."""
    x = r.standard_normal((n, heads, D)).astype(np.float32)
    rot = rotation.astype(np.float32)
    y = r.standard_normal((n, heads, D)).astype(np.float32)
    y[..., ::2] = np.float32(BOUNDS[bits])[r.integers(0, len(BOUNDS[bits]), (n, heads, D // 2))] * r.choice([-1, 1], (n, heads, D // 2))
    rest = np.maximum(1.0 - (y[..., ::2] ** 2).sum(-1, keepdims=True), 0.01)
    y[..., 1::2] *= np.sqrt(rest / (y[..., 1::2] ** 2).sum(-1, keepdims=True))
    x[1::3] = (8.0 * y @ rot)[1::3]
    for i, scale in ((2, 0.0), (5, 6e-8), (8, 3e-6), (11, 30000.0), (14, 1e-3)):
        x[i::15] *= np.float32(scale)
    x[17::30] = 0.0
    x[17::30, :, 5] = 1.0
    return np.clip(x, -65504, 65504).astype(np.float16).reshape(n, heads * D)


@pytest.mark.parametrize("kind", ["rotation", "scaled", "equal rows"])
@pytest.mark.parametrize("bits,T,streams", [(4, 257, 2), (4, 1366, 2), (2, 700, 2), (4, 300, 1), (2, 1100, 1)])
def test_prompt_append(oracle, rotation_fixture, bits, T, streams, kind):
    import torch
    from triebwerk_amd import kvcache as kvc
    Hk = 8
    r = gen.rng(9100 + bits + T)
    rot = _matrix(rotation_fixture, kind)
    kv_dim, msl = Hk * D, T + 1
    src = [_hard_rows(r, rot, T, Hk, bits) for _ in range(streams)]
    pos = r.permutation(msl)[:T].astype(np.int32)
    want = [(np.zeros((msl, kv_dim * bits // 8), np.uint8), np.zeros((msl, Hk), np.float16)) for _ in range(streams)]
    got = [tuple(dev(x) for x in w) for w in want]
    for s, (c, n) in zip(src, want):
        oracle.turbo_kv_quantize(c, n, s, rot, pos, msl, T, Hk, D, kv_dim, bits)
    if streams == 2:
        kvc.tw_turbo_kv_append_tokens(*got[0], *got[1], dev(src[0]), dev(src[1]), dev(rot), dev(pos), msl, T, Hk, D, kv_dim, bits)
    else:
        kvc.launch_turbo_kv_quantize(*got[0], dev(src[0]), dev(rot), dev(pos), msl, T, Hk, D, kv_dim, bits)
    torch.cuda.synchronize()
    for g, w in zip(got, want):
        for a, b, what in zip(g, w, ("codes", "norms")):
            assert_bytes_equal(host(a), b, what)


@pytest.mark.parametrize("kind", ["rotation", "scaled", "equal rows"])
@pytest.mark.parametrize("bits,H,Hk,G,hkw,shares", [(4, 16, 8, 61, 2, 1), (4, 16, 8, 61, 1, 1), (2, 32, 8, 30, 4, 2), (4, 6, 3, 80, 1, 2), (2, 8, 8, 64, 8, 1)])
def test_layer_step(kv, oracle, rotation_fixture, bits, H, Hk, G, hkw, shares, kind):  # noqa: F811
    """The first tokens of empty caches: what the step stores is the oracle's."""
    import torch
    r = gen.rng(9200 + bits + H + G)
    rot = _matrix(rotation_fixture, kind)
    msl, kv_dim, q_dim = 512, Hk * D, H * D
    want = [np.zeros((G, msl, kv_dim * bits // 8), np.uint8), np.zeros((G, msl, kv_dim * bits // 8), np.uint8),
            np.zeros((G, msl, Hk), np.float16), np.zeros((G, msl, Hk), np.float16)]
    d_c = [dev(x) for x in want]
    scratch = torch.zeros((G * H * msl,), dtype=torch.float32, device="cuda")
    tickets = torch.zeros(G * Hk, dtype=torch.int32, device="cuda")
    kv.set_decode_fused(1)
    kv.set_fused_shape(hkw, shares)
    try:
        for step in range(3):
            pos = np.full(G, step, np.int32)
            q = gen.normal_f16(r, (G, q_dim))
            k, v = _hard_rows(r, rot, G, Hk, bits), _hard_rows(r, rot, G, Hk, bits)
            out = torch.zeros((G, q_dim), dtype=torch.float16, device="cuda")
            kv.tw_layer_attention_step(out, dev(q), dev(k), dev(v), dev(pos), msl, G, H, Hk, D, q_dim, kv_dim, d_c[0], d_c[1], scratch,
                                       kv_bits=bits, k_norms=d_c[2], v_norms=d_c[3], rotation=dev(rot), tickets=tickets)
            torch.cuda.synchronize()
            assert "decode_fused_kernel" in kv.last_scan_kernel()
            oracle.turbo_kv_quantize_batch(want[0], want[2], k, rot, pos, msl, G, Hk, D, kv_dim, bits)
            oracle.turbo_kv_quantize_batch(want[1], want[3], v, rot, pos, msl, G, Hk, D, kv_dim, bits)
    finally:
        kv.set_fused_shape(0, 0)
        kv.set_decode_fused(0)
    for got, w, what in zip(d_c, want, ("K codes", "V codes", "K norms", "V norms")):
        assert_bytes_equal(host(got), w, what)


@pytest.mark.parametrize("bits,H,Hk,G,hkw", [(4, 16, 8, 31, 2), (4, 16, 8, 31, 8), (2, 32, 8, 15, 4)])
def test_every_layer_at_once(oracle, bits, H, Hk, G, hkw):
    """The same rows through the launch of all layers, whose rotation is the engine's own; positions advance."""
    import torch
    from triebwerk_amd import Engine, kvcache
    L, msl = 4, 64
    r = gen.rng(9300 + bits + G)
    eng = Engine(max_seq_len=msl, kv_bits=bits)
    eng.set_shape(L, H, Hk, D)
    eng.alloc_batch(G, msl)
    rot = host(eng.rotation())
    eng.set_positions([0] * G)
    k, v = (np.stack([_hard_rows(r, rot, G, Hk, bits) for _ in range(L)]) for _ in range(2))
    q = gen.normal_f16(r, (L, G, H * D))
    out = torch.zeros((L, G, H * D), dtype=torch.float16, device="cuda")
    kvcache.set_fused_shape(hkw, 0)
    try:
        for _ in range(2):
            eng.decode_step(dev(q), dev(k), dev(v), out)
            torch.cuda.synchronize()
    finally:
        kvcache.set_fused_shape(0, 0)
    assert "decode_layers_kernel" in kvcache.last_scan_kernel()
    assert eng.positions().tolist() == [2] * G
    for l in range(L):
        want = [np.zeros((G, msl, Hk * D * bits // 8), np.uint8) for _ in range(2)] + [np.zeros((G, msl, Hk), np.float16) for _ in range(2)]
        for p in range(2):
            pos = np.full(G, p, np.int32)
            oracle.turbo_kv_quantize_batch(want[0], want[2], k[l], rot, pos, msl, G, Hk, D, Hk * D, bits)
            oracle.turbo_kv_quantize_batch(want[1], want[3], v[l], rot, pos, msl, G, Hk, D, Hk * D, bits)
        for got, w, what in zip(eng.cache(l), want, ("K codes", "V codes", "K norms", "V norms")):
            assert_bytes_equal(host(got)[:, :2], w[:, :2], f"layer {l} {what}")


def _far_rows(r, n, heads):
    """A matrix whose rows are of norm 4e5 and vectors that it takes far out, but for every 16th row and the first head, whose values lie among the
    boundaries: there the first 56 coordinates meet the next 56 with the other sign, and the last 16 make the value.  What rounding does
    on the way is larger than the distance of two boundaries."""
    m = (r.uniform(20000, 65504, (D, D)) * r.choice([-1, 1], (D, D))).astype(np.float32)
    m[::16, 56:112] = -m[::16, :56]
    m[::16, 112:] = r.standard_normal((D // 16, 16))
    x = r.standard_normal((n, heads, D)).astype(np.float32)
    x[:, 0, 56:112] = x[:, 0, :56]
    x[:, 0, 112:] *= 0.5
    return m.astype(np.float16), x.astype(np.float16).reshape(n, heads * D)


@pytest.mark.parametrize("scale", [1.0, 0.03, 0.001])
@pytest.mark.parametrize("bits,T", [(4, 1366), (2, 700)])
def test_rows_of_any_norm(oracle, bits, T, scale):
    """The bound is wider than a bucket there, and a boundary in the next bucket within it.  One value of a block that is not far out: else
    another one's doubt has the whole block repeated."""
    import torch
    from triebwerk_amd import kvcache as kvc
    Hk = 8
    r = gen.rng(9150 + bits)
    rot, k = _far_rows(r, T, Hk)
    rot = (scale * rot.astype(np.float32)).astype(np.float16)
    v = r.standard_normal((T, Hk * D)).astype(np.float16)
    kv_dim, msl = Hk * D, T + 1
    pos = np.arange(T, dtype=np.int32)
    want = [(np.zeros((msl, kv_dim * bits // 8), np.uint8), np.zeros((msl, Hk), np.float16)) for _ in range(2)]
    got = [tuple(dev(x) for x in w) for w in want]
    for s, (c, n) in zip((k, v), want):
        oracle.turbo_kv_quantize(c, n, s, rot, pos, msl, T, Hk, D, kv_dim, bits)
    kvc.tw_turbo_kv_append_tokens(*got[0], *got[1], dev(k), dev(v), dev(rot), dev(pos), msl, T, Hk, D, kv_dim, bits)
    torch.cuda.synchronize()
    for g, w in zip(got, want):
        for a, b, what in zip(g, w, ("codes", "norms")):
            assert_bytes_equal(host(a), b, what)
