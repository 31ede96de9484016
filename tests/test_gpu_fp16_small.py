"""Small fp16 batches (attention_valu_kernel and attention_merge_kernel): the appended token at the first, a middle and the last place
of a step of 32 tokens and alone in its chunk, one token in all, query heads in tiles of 1, 2 and 4, up to 64 partials (one group
of threads merges up to 8 of them, four merge more of up to 1024 heads), a query buffer that is not 16-byte aligned, gates.  Against the oracle."""
import numpy as np
import pytest

import gen
from test_gpu_parity import D, TOL, assert_bytes_equal, dev, host, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("aligned", [True, False])
@pytest.mark.parametrize("H,Hk,lens,msl,splits", [
    (16, 8, [1, 2, 32, 33], 256, 0), (16, 8, [1], 64, 0), (8, 8, [64, 65, 31], 1200, 8), (16, 8, [129, 257], 2048, 9),
    (32, 8, [300, 1], 4096, 30), (16, 8, [1025], 8704, 64), (4, 1, [97, 161, 3], 1500, 0), (6, 2, [200], 1500, 10), (16, 4, [2049], 4096, 0),
    (16, 8, [700] + [40] * 63, 1408, 9), (16, 8, [700] + [40] * 64, 1408, 9), (32, 8, [300, 17] * 20, 2176, 16),
])
def test_append_and_attention(oracle, H, Hk, lens, msl, splits, aligned):
    import torch
    from triebwerk_amd import kvcache as kv
    r = gen.rng(7000 + H + Hk + len(lens) + msl)
    G, kd, qd = len(lens), Hk * D, H * D
    ck, cv = gen.normal_f16(r, (G, msl, kd)), gen.normal_f16(r, (G, msl, kd))
    q, k, v = gen.normal_f16(r, (G, qd)), gen.normal_f16(r, (G, kd)), gen.normal_f16(r, (G, kd))
    pos = np.array([n - 1 for n in lens], np.int32)
    d_ck, d_cv = dev(ck), dev(cv)
    flat = torch.zeros(G * qd + 1, dtype=torch.float16, device="cuda")
    d_q = flat[:G * qd] if aligned else flat[1:]
    d_q.copy_(dev(q).view(-1))
    out = torch.zeros((G, qd), dtype=torch.float16, device="cuda")
    scratch = torch.full((G * H * msl,), float("nan"), dtype=torch.float32, device="cuda")     # what no workgroup writes is not used
    kv.set_num_splits(splits)
    try:
        kv.tw_append_attention_batch(out, d_q, dev(k), dev(v), d_ck, d_cv, scratch, dev(pos), msl, G, H, Hk, D, qd, kd)
        torch.cuda.synchronize()
    finally:
        kv.set_num_splits(0)
    assert kv.last_scan_kernel() in ("attention_valu_kernel", "attention_rows_kernel")
    oracle.kv_cache_write_batch(ck, cv, k, v, pos, msl, G, kd)
    want = np.zeros((G, qd), np.float16)
    oracle.gqa_attention_batch(want, q, ck, cv, pos, msl, G, H, Hk, D, qd, kd)
    assert rel_err(host(out), want) <= TOL
    assert_bytes_equal(host(d_ck), ck, "K"); assert_bytes_equal(host(d_cv), cv, "V")
