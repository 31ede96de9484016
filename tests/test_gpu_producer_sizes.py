"""RMSNorm and rotary embedding of q and k on both sides of the number of vectors where the launch changes from a wave to a
vector to 16 lanes to a vector (16, 20 and 24 vectors per compute unit): the oracle's bytes, in place and into the fp16 cache."""
import numpy as np
import pytest

import gen

pytestmark = pytest.mark.gpu
D = 128


def dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def same_bytes(got, want):
    assert np.array_equal(got.cpu().numpy().view(np.uint8), want.view(np.uint8))


@pytest.mark.parametrize("kind", ["norm", "rope", "both"])
@pytest.mark.parametrize("H,Hk", [(16, 8), (4, 1)])
@pytest.mark.parametrize("past", [-1, 0, 1])
def test_both_mappings(oracle, kind, H, Hk, past):
    import torch
    from triebwerk_amd import kvcache as kv
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    edge = {"norm": 16, "rope": 20, "both": 24}[kind] * cus
    per_row = H + Hk * (2 if kind == "both" else 1)
    G = edge // per_row + past                  # edge itself where per_row divides it: still a wave to a vector
    r = gen.rng(7300 + G)
    q_dim, kv_dim, msl = H * D, Hk * D, G + 1
    q, k, v = (gen.normal_f16(r, (G, n)) for n in (q_dim, kv_dim, kv_dim))
    qw, kw = ((1 + 0.2 * r.standard_normal(D)).astype(np.float16) for _ in range(2))
    ct, st = oracle.rope_tables(msl, 128, 1e6)
    pos = np.arange(G, dtype=np.int32)
    dq, dk, dp = dev(q), dev(k), dev(pos)
    if kind == "both":                          # a prompt's producers: q in place, K and V straight into the cache
        ck, cv = (torch.zeros((msl, kv_dim), dtype=torch.float16, device="cuda") for _ in range(2))
        out = torch.zeros((G, q_dim), dtype=torch.float16, device="cuda")
        kv.tw_layer_prompt_step(out, dq, dk, dev(v), dp, msl, G, H, Hk, D, q_dim, kv_dim, ck, cv, None, kv_bits=0, q_weight=dev(qw),
                                k_weight=dev(kw), eps=1e-6, cos_table=dev(ct), sin_table=dev(st), rope_dim=128)
    elif kind == "norm":
        kv.launch_qk_norm_batch(dq, dk, dev(qw), dev(kw), H, Hk, D, G, 1e-6, q_dim, kv_dim)
    else:
        kv.launch_rope_batch(dq, dk, dev(ct), dev(st), dp, msl, G, H, Hk, D, q_dim, kv_dim, 128)
    torch.cuda.synchronize()
    if kind != "rope":
        oracle.qk_norm_batch(q, k, qw, kw, H, Hk, D, G, 1e-6, q_dim, kv_dim, False)
    if kind != "norm":
        oracle.rope_batch(q, k, ct, st, pos, msl, G, H, Hk, D, q_dim, kv_dim, 128)
    same_bytes(dq, q)
    if kind == "both":
        same_bytes(ck[:G], k)
        same_bytes(cv[:G], v)
    else:
        same_bytes(dk, k)
