"""The append of many rows in tiles shared by a workgroup (append_tokens_kernel) and the producers 16 lanes to a vector
(producer_rows_kernel): the oracle's bytes at the edges of tiles, of tile runs per workgroup and of the choice between kernels,
and where a pointer or a stride does not admit 16-byte accesses."""
import numpy as np
import pytest

import gen

pytestmark = pytest.mark.gpu
D = 128


def dev(a, offset=0):
    """On the GPU, `offset` elements into its allocation (offset = 1: not on a 16-byte boundary)."""
    import torch
    t = torch.from_numpy(np.ascontiguousarray(a))
    out = torch.empty(t.numel() + offset, dtype=t.dtype, device="cuda")[offset:].view(t.shape)
    return out.copy_(t)


def same_bytes(got, want):
    assert np.array_equal(got.cpu().numpy().view(np.uint8), want.view(np.uint8))


@pytest.mark.parametrize("bits,T,Hk", [(4, 3, 8), (4, 4, 8), (4, 33, 1), (4, 129, 3), (4, 1500, 8), (4, 4111, 8), (4, 700, 20),
                                       (2, 63, 8), (2, 64, 8), (2, 171, 3), (2, 3001, 8)])
def test_append_tokens(oracle, rotation_fixture, bits, T, Hk):
    import torch
    from triebwerk_amd import kvcache as kv
    r = gen.rng(7000 + bits + T)
    kv_dim, msl = Hk * D, T + 5
    k, v = gen.normal_f16(r, (T, kv_dim)), gen.normal_f16(r, (T, kv_dim))
    k[0, :D] = 0
    k[1] = (k[1].astype(np.float32) * 1e-4).astype(np.float16)
    v[2] = (v[2].astype(np.float32) * 300).astype(np.float16)
    v[T - 1, -D:] = np.float16(np.nan)            # the last vector of the last, partial tile
    k[T - 1, :D] = np.float16(np.inf)
    pos = r.permutation(msl)[:T].astype(np.int32)
    want = [np.zeros((msl, n), t) for n, t in ((kv_dim * bits // 8, np.uint8), (Hk, np.float16))] + \
           [np.zeros((msl, n), t) for n, t in ((kv_dim * bits // 8, np.uint8), (Hk, np.float16))]
    oracle.turbo_kv_quantize(want[0], want[1], k, rotation_fixture, pos, msl, T, Hk, D, kv_dim, bits)
    oracle.turbo_kv_quantize(want[2], want[3], v, rotation_fixture, pos, msl, T, Hk, D, kv_dim, bits)
    rot, dp = dev(rotation_fixture), dev(pos)
    got = [dev(np.zeros_like(w)) for w in want]
    kv.tw_turbo_kv_append_tokens(got[0], got[1], got[2], got[3], dev(k), dev(v), rot, dp, msl, T, Hk, D, kv_dim, bits)
    one = [dev(np.zeros_like(w)) for w in want[:2]]
    kv.launch_turbo_kv_quantize(one[0], one[1], dev(k), rot, dp, msl, T, Hk, D, kv_dim, bits)
    off = [dev(np.zeros_like(w)) for w in want[:2]]       # source rows off the 16-byte boundaries: the other kernel
    kv.launch_turbo_kv_quantize(off[0], off[1], dev(k, 1), rot, dp, msl, T, Hk, D, kv_dim, bits)
    torch.cuda.synchronize()
    for g, w in zip(got + one + off, want + want[:2] + want[:2]):
        if w.dtype == np.float16:                 # (a NaN's own bits are not part of the comparison)
            gn = g.cpu().numpy()
            assert np.array_equal(np.isnan(gn), np.isnan(w)) and np.array_equal(gn[~np.isnan(w)], w[~np.isnan(w)])
        else:
            same_bytes(g, w)


def test_append_many_sequences(oracle, rotation_fixture):
    """The batch layout (row g of sequence g) at a size that takes the tiles."""
    from triebwerk_amd import kvcache as kv
    r = gen.rng(7100)
    G, Hk, msl, bits = 160, 8, 7, 4
    kv_dim = Hk * D
    rows, pos = gen.normal_f16(r, (G, kv_dim)), r.integers(0, msl, G).astype(np.int32)
    cq, cn = np.zeros((G, msl, kv_dim // 2), np.uint8), np.zeros((G, msl, Hk), np.float16)
    oracle.turbo_kv_quantize_batch(cq, cn, rows, rotation_fixture, pos, msl, G, Hk, D, kv_dim, bits)
    gq, gn = dev(np.zeros_like(cq)), dev(np.zeros_like(cn))
    kv.launch_turbo_kv_quantize_batch(gq, gn, dev(rows), dev(rotation_fixture), dev(pos), msl, G, Hk, D, kv_dim, bits)
    same_bytes(gq, cq)
    same_bytes(gn, cn)


@pytest.mark.parametrize("bits,T,H,Hk,rope_dim,norm,offset", [
    (4, 1, 8, 8, 128, True, 0), (4, 50, 16, 8, 128, True, 0), (2, 37, 8, 2, 16, True, 0), (4, 65, 6, 3, 48, False, 0),
    (2, 130, 8, 8, 64, True, 0), (4, 31, 4, 1, 32, True, 1), (4, 2300, 16, 8, 128, True, 0), (2, 90, 8, 4, 0, True, 0)])
def test_prompt_step_with_producers(oracle, rotation_fixture, bits, T, H, Hk, rope_dim, norm, offset):
    """Queries and keys come back as the oracle's producers leave them, the cache has the oracle's bytes: queries beside the
    tiles (short prompts), in a launch of their own (2300 tokens), and rows off the 16-byte boundaries."""
    import torch
    from triebwerk_amd import kvcache as kv
    r = gen.rng(7200 + T)
    q_dim, kv_dim, msl = H * D, Hk * D, T + 3
    q, k, v = (gen.normal_f16(r, (T, n)) for n in (q_dim, kv_dim, kv_dim))
    qw, kw = ((1 + 0.2 * r.standard_normal(D)).astype(np.float16) for _ in range(2))
    pos = np.arange(T, dtype=np.int32)
    extra, biased = {}, T % 2 == 1
    d = [dev(x, offset) for x in (q, k, v)]
    if norm:
        extra.update(q_weight=dev(qw), k_weight=dev(kw), eps=1e-6, biased=biased)
        oracle.qk_norm_batch(q, k, qw, kw, H, Hk, D, T, 1e-6, q_dim, kv_dim, biased)
    if rope_dim:
        ct, st = oracle.rope_tables(msl, rope_dim, 1e6)
        extra.update(cos_table=dev(ct), sin_table=dev(st), rope_dim=rope_dim)
        oracle.rope_batch(q, k, ct, st, pos, msl, T, H, Hk, D, q_dim, kv_dim, rope_dim)
    want = [np.zeros((msl, kv_dim * bits // 8), np.uint8), np.zeros((msl, Hk), np.float16)] * 2
    want = [w.copy() for w in want]
    oracle.turbo_kv_quantize(want[0], want[1], k, rotation_fixture, pos, msl, T, Hk, D, kv_dim, bits)
    oracle.turbo_kv_quantize(want[2], want[3], v, rotation_fixture, pos, msl, T, Hk, D, kv_dim, bits)
    got = [dev(np.zeros_like(w)) for w in want]
    out = torch.zeros((T, q_dim), dtype=torch.float16, device="cuda")
    scratch = torch.zeros(T * H * max(T, 1024) if T < 500 else T * H * 264, dtype=torch.float32, device="cuda")
    kv.tw_layer_prompt_step(out, *d, dev(pos), msl, T, H, Hk, D, q_dim, kv_dim, got[0], got[2], scratch, kv_bits=bits,
                            k_norms=got[1], v_norms=got[3], rotation=dev(rotation_fixture), **extra)
    torch.cuda.synchronize()
    for g, w in zip(got, want):
        same_bytes(g, w)
    for g, w in zip(d, (q, k, v)):
        same_bytes(g, w)
