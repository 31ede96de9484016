"""Small fp16 steps whose chunks merge in the launch that scans them (tickets): few chunks and 64, chunks without a token, query
heads in tiles of 1, 2 and 4, the tickets left zero for the next step; an output exactly over the queries, and one over k, whose rows are in
the cache by then.  A step without tickets, heads in several tiles, and an output that lies over other heads' queries take the merge as a
launch of its own.  Against the oracle."""
import numpy as np
import pytest

import gen
from test_gpu_parity import D, TOL, assert_bytes_equal, dev, host, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("how", ["tickets", "none", "over q", "over k", "a head after q", "a head before q"])
@pytest.mark.parametrize("H,Hk,lens,msl,splits", [
    (16, 8, [1, 2, 32, 33], 2048, 2), (8, 8, [64, 65, 31], 2048, 8), (16, 8, [129, 257, 3], 2048, 9), (32, 8, [300, 1], 4096, 30),
    (4, 1, [97, 161, 3], 1500, 0), (6, 2, [200], 1500, 10), (16, 4, [2049], 16384, 64), (32, 8, [33, 8000], 16384, 64), (3, 3, [500, 1], 2048, 3),
])
def test_chunks_merge_themselves(oracle, H, Hk, lens, msl, splits, how):
    import torch
    from triebwerk_amd import kvcache as kv
    r = gen.rng(9400 + H + Hk + len(lens) + msl)
    G, kd, qd = len(lens), Hk * D, H * D
    ck, cv = gen.normal_f16(r, (G, msl, kd)), gen.normal_f16(r, (G, msl, kd))
    d_ck, d_cv = dev(ck), dev(cv)
    scratch = torch.full((G * H * msl,), float("nan"), dtype=torch.float32, device="cuda")     # what no workgroup writes is not used
    tickets = torch.zeros(G * Hk, dtype=torch.int32, device="cuda")
    kv.set_num_splits(splits)
    try:
        for step in range(3):
            q, k, v = gen.normal_f16(r, (G, qd)), gen.normal_f16(r, (G, kd)), gen.normal_f16(r, (G, kd))
            pos = np.array([n - 1 + step for n in lens], np.int32)
            d_q, d_k = dev(q), dev(k)
            out = torch.zeros((G, qd), dtype=torch.float16, device="cuda")
            if how == "over q": out = d_q
            if how in ("a head after q", "a head before q"):
                both = torch.zeros(G * qd + D, dtype=torch.float16, device="cuda")
                first, second = both[:G * qd].view(G, qd), both[D:].view(G, qd)
                d_q, out = (first, second) if how == "a head after q" else (second, first)
                d_q.copy_(dev(q))
            if how == "over k":                                # the rows' beginnings, a row apart
                both = torch.zeros(G * qd + G * kd, dtype=torch.float16, device="cuda")
                out, d_k = both[:G * qd].view(G, qd), both[G * qd - kd:G * qd + (G - 1) * kd].view(G, kd)
                d_k.copy_(dev(k))
            kv.tw_layer_attention_step(out, d_q, d_k, dev(v), dev(pos), msl, G, H, Hk, D, qd, kd, d_ck, d_cv, scratch, kv_bits=0,
                                       tickets=None if how == "none" else tickets)
            torch.cuda.synchronize()
            # heads in one tile to a KV head: else their workgroups share no ticket
            merged = how in ("tickets", "over q", "over k") and H // Hk in (1, 2, 4)
            assert kv.last_scan_kernel() == "attention_valu_kernel" + (", chunks merged in the launch" if merged else "")
            oracle.kv_cache_write_batch(ck, cv, k, v, pos, msl, G, kd)
            want = np.zeros((G, qd), np.float16)
            oracle.gqa_attention_batch(want, q, ck, cv, pos, msl, G, H, Hk, D, qd, kd)
            got = host(out)
            assert max(rel_err(got[g], want[g]) for g in range(G)) <= TOL, f"step {step}"
            assert not host(tickets).any(), "tickets were not left zero"
    finally:
        kv.set_num_splits(0)
    assert_bytes_equal(host(d_ck), ck, "K"); assert_bytes_equal(host(d_cv), cv, "V")
