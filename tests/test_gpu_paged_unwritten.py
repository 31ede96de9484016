"""Pages whose slots past a sequence's end were never written: norms and fp16 rows there may be any bits, NaN and infinities among
them, and so may pages of the pool that no table entry names.  Every form of a paged step against the oracle on the rows that exist."""
import numpy as np
import pytest

import gen
from test_gpu_parity import D, TOL, dev, host, rel_err

pytestmark = pytest.mark.gpu

LENS = [1, 15, 16, 17, 31, 32, 33, 65]
POISON = [np.nan, np.inf, -np.inf]


def _pages(x, table, pages, lens, poison):
    """(G, msl, w) rows into a pool with one page more per sequence than the tables name; slots past the length hold `poison`."""
    G, msl, w = x.shape
    x = x.copy()
    if poison is not None:
        for g, n in enumerate(lens):
            x[g, n:] = poison
    pool = np.zeros((G * (pages + 1), 16, w), x.dtype)
    if poison is not None:
        pool[:] = poison
    pool[table.reshape(-1)] = x.reshape(G * pages, 16, w)
    return dev(pool)


@pytest.mark.parametrize("poison", POISON)
@pytest.mark.parametrize("form", ["one launch", "three launches", "one head per wave", "attention call", "vector ALU"])
@pytest.mark.parametrize("bits,H,Hk", [(4, 16, 8), (2, 16, 8), (4, 6, 3), (2, 8, 8), (4, 32, 8)])
def test_unwritten_norms_do_not_reach_the_output(oracle, rotation_fixture, bits, H, Hk, form, poison):
    import torch
    from triebwerk_amd import kvcache as kv
    G, pages = len(LENS), 6
    msl = 16 * pages
    r = gen.rng(6100 + bits + H + Hk)
    c = [r.integers(0, 256, (G, msl, Hk * D * bits // 8), dtype=np.uint8) for _ in range(2)]
    c += [(11.3 + 0.7 * r.standard_normal((G, msl, Hk))).astype(np.float16) for _ in range(2)]
    q = gen.normal_f16(r, (G, H * D)); k = gen.normal_f16(r, (G, Hk * D)); v = gen.normal_f16(r, (G, Hk * D))
    pos = np.array([n - 1 for n in LENS], np.int32)
    table = r.permutation(G * (pages + 1))[:G * pages].astype(np.int32).reshape(G, pages)
    d = [_pages(x, table, pages, LENS, poison if i >= 2 else None) for i, x in enumerate(c)]
    out = torch.zeros((G, H * D), dtype=torch.float16, device="cuda")
    ws = torch.zeros(kv.attention_workspace_floats(G, H, msl), dtype=torch.float32, device="cuda")
    tail = [dev(rotation_fixture), ws, dev(pos), dev(table), pages, msl, G, H, Hk, D, H * D, Hk * D, bits]
    try:
        if form == "three launches": kv.set_decode_fused(2)
        if form == "one head per wave": kv.set_attention_variant(3)
        if form == "vector ALU": kv.set_attention_variant(1)
        if form == "attention call":
            kv.tw_paged_turbo_gqa_attention_batch(out, dev(q), *d, *tail)
        else:
            kv.tw_paged_turbo_append_attention_batch(out, dev(q), dev(k), dev(v), *d, *tail)
        torch.cuda.synchronize()
    finally:
        kv.set_decode_fused(0)
        kv.set_attention_variant(0)
    if form == "one launch" and Hk % 2 == 0: assert kv.last_scan_kernel().endswith("paged"), kv.last_scan_kernel()
    if form == "one head per wave": assert kv.last_scan_kernel() == "attention_mfma_kernel"
    if form != "attention call":
        oracle.turbo_kv_quantize_batch(c[0], c[2], k, rotation_fixture, pos, msl, G, Hk, D, Hk * D, bits)
        oracle.turbo_kv_quantize_batch(c[1], c[3], v, rotation_fixture, pos, msl, G, Hk, D, Hk * D, bits)
    want = np.zeros((G, H * D), np.float16)
    oracle.turbo_gqa_attention_batch(want, q, *c, rotation_fixture, pos, msl, G, H, Hk, D, H * D, Hk * D, bits)
    got = host(out)
    assert np.isfinite(got).all(), f"{form}: sequences {sorted(set(np.argwhere(~np.isfinite(got))[:, 0].tolist()))}"
    assert rel_err(got, want) <= TOL


@pytest.mark.parametrize("poison", POISON)
@pytest.mark.parametrize("H,Hk", [(16, 8), (4, 1), (32, 8)])
def test_unwritten_fp16_rows_do_not_reach_the_output(oracle, H, Hk, poison):
    import torch
    from triebwerk_amd import kvcache as kv
    G, pages = len(LENS), 6
    msl = 16 * pages
    r = gen.rng(6200 + H + Hk)
    ck, cv = gen.normal_f16(r, (G, msl, Hk * D)), gen.normal_f16(r, (G, msl, Hk * D))
    q = gen.normal_f16(r, (G, H * D))
    pos = np.array([n - 1 for n in LENS], np.int32)
    table = r.permutation(G * (pages + 1))[:G * pages].astype(np.int32).reshape(G, pages)
    out = torch.zeros((G, H * D), dtype=torch.float16, device="cuda")
    ws = torch.zeros(kv.attention_workspace_floats(G, H, msl), dtype=torch.float32, device="cuda")
    kv.tw_paged_gqa_attention_batch(out, dev(q), _pages(ck, table, pages, LENS, poison), _pages(cv, table, pages, LENS, poison), ws, dev(pos),
                                    dev(table), pages, msl, G, H, Hk, D, H * D, Hk * D)
    torch.cuda.synchronize()
    want = np.zeros((G, H * D), np.float16)
    oracle.gqa_attention_batch(want, q, ck, cv, pos, msl, G, H, Hk, D, H * D, Hk * D)
    assert np.isfinite(host(out)).all() and rel_err(host(out), want) <= TOL
