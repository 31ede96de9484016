"""The pair kernel as attention alone (launch_turbo_gqa_attention_batch) and as the whole step over pages
(tw_paged_turbo_append_attention_batch), at the edges of tiles, pages and parts, against the oracle: the appended rows bit for
bit, the outputs within the parity tolerance; and that short bounds take it and long ones do not."""
import numpy as np
import pytest

import gen
from test_gpu_parity import D, TOL, assert_bytes_equal, dev, host, rel_err

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def kv():
    from triebwerk_amd import kvcache
    return kvcache


def _case(bits, H, Hk, lens, msl, seed):
    r = gen.rng(seed)
    G, kvp = len(lens), Hk * D * bits // 8
    c = [r.integers(0, 256, (G, msl, kvp), dtype=np.uint8) for _ in range(2)]
    c += [(11.3 + 0.7 * r.standard_normal((G, msl, Hk))).astype(np.float16) for _ in range(2)]
    q = gen.normal_f16(r, (G, H * D)); k = gen.normal_f16(r, (G, Hk * D)); v = gen.normal_f16(r, (G, Hk * D))
    return c, q, k, v, np.array([n - 1 for n in lens], np.int32), r


SHAPES = [
    (4, 16, 8, [1, 2, 15, 16, 17, 31, 32, 33, 64, 65], 272), (2, 16, 8, [1, 31, 32, 33, 255, 256, 257], 272),
    (4, 8, 8, [500, 511, 512], 512), (2, 8, 4, [129] * 70, 272), (4, 32, 8, [100, 1], 288), (2, 32, 8, [63] * 33, 272),
    (4, 4, 2, [300, 17], 304), (2, 12, 12, [48, 49], 272),
]


@pytest.mark.parametrize("bits,H,Hk,lens,msl", SHAPES)
def test_attention_alone(kv, oracle, rotation_fixture, bits, H, Hk, lens, msl):
    import torch
    G = len(lens)
    c, q, _, _, pos, _ = _case(bits, H, Hk, lens, msl, 5100 + bits + H + G)
    want = np.zeros((G, H * D), np.float16)
    oracle.turbo_gqa_attention_batch(want, q, *c, rotation_fixture, pos, msl, G, H, Hk, D, H * D, Hk * D, bits)
    d = [dev(x) for x in c]
    out = torch.zeros((G, H * D), dtype=torch.float16, device="cuda")
    scratch = torch.zeros(G * H * msl, dtype=torch.float32, device="cuda")
    kv.launch_turbo_gqa_attention_batch(out, dev(q), *d, dev(rotation_fixture), scratch, dev(pos), msl, G, H, Hk, D, H * D, Hk * D, bits)
    torch.cuda.synchronize()
    assert "attention alone" in kv.last_scan_kernel(), kv.last_scan_kernel()
    assert rel_err(host(out), want) <= TOL


@pytest.mark.parametrize("bits", [4, 2])
@pytest.mark.parametrize("room", ["256 rows", "none", "unaligned", "noalloc, 256 rows"])
def test_attention_alone_without_room_for_partials_stays_in_fp32(kv, oracle, rotation_fixture, bits, room):
    """No scratch for partials and the rotated query: the kernel that keeps p * norm in fp32 runs, and V norms past 65504 / 2^5, which
    an fp16 value + remainder does not hold, give the oracle's output.  One K direction for all tokens, its norm rising tile by tile
    in the second half of the context: among 16 heads and 8 tiles some p lie between 2^4 and 2^5, where a running maximum stays."""
    import torch
    H, Hk = 16, 8
    msl = 256 if "256" in room else 512
    lens = [msl, 33, 1]
    G = len(lens)
    c, q, _, _, pos, _ = _case(bits, H, Hk, lens, msl, 5400 + bits)
    c[0][:] = c[0][:, :1]
    c[2][:] = (5 + 16 * np.maximum(np.arange(msl) // 32 - 7, 0))[None, :, None]
    c[3] = (c[3].astype(np.float32) * 350).astype(np.float16)              # V norms of 3300 to 5000
    want = np.zeros((G, H * D), np.float16)
    oracle.turbo_gqa_attention_batch(want, q, *c, rotation_fixture, pos, msl, G, H, Hk, D, H * D, Hk * D, bits)
    out = torch.zeros((G, H * D), dtype=torch.float16, device="cuda")
    flat = torch.zeros(G * H * msl + 1, dtype=torch.float32, device="cuda")
    scratch = None if room == "none" else flat[1:] if room == "unaligned" else flat[:-1]
    head, tail = (out, dev(q), *[dev(x) for x in c], dev(rotation_fixture)), (dev(pos), msl, G, H, Hk, D, H * D, Hk * D, bits)
    if "noalloc" in room: kv.tw_turbo_gqa_attention_batch_noalloc(*head, *tail)
    else: kv.launch_turbo_gqa_attention_batch(*head, scratch, *tail)
    torch.cuda.synchronize()
    assert rel_err(host(out), want) <= TOL
    assert kv.last_scan_kernel() == "attention_valu_kernel"


@pytest.mark.parametrize("bits", [4, 2])
@pytest.mark.parametrize("room", ["none", "unaligned"])
def test_paged_step_without_a_workspace_stays_in_fp32(kv, oracle, rotation_fixture, bits, room):
    import torch
    H, Hk, lens = 16, 8, [200, 33, 1]
    G, msl = len(lens), 256
    c, q, k, v, pos, r = _case(bits, H, Hk, lens, msl, 5500 + bits)
    table = np.arange(G * msl // 16, dtype=np.int32).reshape(G, msl // 16)
    d = [dev(x.reshape(-1, 16, x.shape[2])) for x in c]
    out = torch.zeros((G, H * D), dtype=torch.float16, device="cuda")
    flat = torch.zeros(kv.attention_workspace_floats(G, H, msl) + 1, dtype=torch.float32, device="cuda")
    kv.tw_paged_turbo_append_attention_batch(out, dev(q), dev(k), dev(v), *d, dev(rotation_fixture), None if room == "none" else flat[1:], dev(pos),
                                             dev(table), msl // 16, msl, G, H, Hk, D, H * D, Hk * D, bits)
    torch.cuda.synchronize()
    oracle.turbo_kv_quantize_batch(c[0], c[2], k, rotation_fixture, pos, msl, G, Hk, D, Hk * D, bits)
    oracle.turbo_kv_quantize_batch(c[1], c[3], v, rotation_fixture, pos, msl, G, Hk, D, Hk * D, bits)
    want = np.zeros((G, H * D), np.float16)
    oracle.turbo_gqa_attention_batch(want, q, *c, rotation_fixture, pos, msl, G, H, Hk, D, H * D, Hk * D, bits)
    assert rel_err(host(out), want) <= TOL
    assert kv.last_scan_kernel() == "attention_valu_kernel"


@pytest.mark.parametrize("bits,H,Hk,lens,msl", SHAPES)
def test_paged_step(kv, oracle, rotation_fixture, bits, H, Hk, lens, msl):
    import torch
    G, pages = len(lens), msl // 16
    c, q, k, v, pos, r = _case(bits, H, Hk, lens, msl, 5200 + bits + H + G)
    table = r.permutation(G * pages).astype(np.int32).reshape(G, pages)
    # the same rows, page by page where the table puts them
    d = []
    for x in c:
        p = np.zeros((G * pages, 16, x.shape[2]), x.dtype)
        p[table.reshape(-1)] = x.reshape(G * pages, 16, x.shape[2])
        d.append(dev(p))
    out = torch.zeros((G, H * D), dtype=torch.float16, device="cuda")
    ws = torch.zeros(kv.attention_workspace_floats(G, H, msl), dtype=torch.float32, device="cuda")
    kv.tw_paged_turbo_append_attention_batch(out, dev(q), dev(k), dev(v), *d, dev(rotation_fixture), ws, dev(pos), dev(table), pages, msl,
                                             G, H, Hk, D, H * D, Hk * D, bits)
    torch.cuda.synchronize()
    assert kv.last_scan_kernel().endswith("paged"), kv.last_scan_kernel()
    oracle.turbo_kv_quantize_batch(c[0], c[2], k, rotation_fixture, pos, msl, G, Hk, D, Hk * D, bits)
    oracle.turbo_kv_quantize_batch(c[1], c[3], v, rotation_fixture, pos, msl, G, Hk, D, Hk * D, bits)
    want = np.zeros((G, H * D), np.float16)
    oracle.turbo_gqa_attention_batch(want, q, *c, rotation_fixture, pos, msl, G, H, Hk, D, H * D, Hk * D, bits)
    assert rel_err(host(out), want) <= TOL
    for got, x in zip(d, c):
        back = host(got).reshape(G * pages, 16, x.shape[2])[table.reshape(-1)].reshape(x.shape)
        assert_bytes_equal(back, x, "pages")


def test_long_bounds_keep_three_launches(kv, oracle, rotation_fixture):
    """Room for 8192 tokens of 18 sequences: the walk shares a sequence between workgroups, one launch would not."""
    import torch
    bits, H, Hk, msl = 4, 16, 8, 8192
    lens = [40, 700, 33] * 6
    G = len(lens)
    c, q, _, _, pos, _ = _case(bits, H, Hk, lens, msl, 5300)
    want = np.zeros((G, H * D), np.float16)
    oracle.turbo_gqa_attention_batch(want, q, *c, rotation_fixture, pos, msl, G, H, Hk, D, H * D, Hk * D, bits)
    out = torch.zeros((G, H * D), dtype=torch.float16, device="cuda")
    scratch = torch.zeros(G * H * msl, dtype=torch.float32, device="cuda")
    kv.launch_turbo_gqa_attention_batch(out, dev(q), *[dev(x) for x in c], dev(rotation_fixture), scratch, dev(pos), msl, G, H, Hk, D,
                                        H * D, Hk * D, bits)
    torch.cuda.synchronize()
    assert kv.last_scan_kernel() == "attention_pair_kernel"
    assert rel_err(host(out), want) <= TOL
