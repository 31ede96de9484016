"""Outputs over inputs of the same call: launches one after the other have consumed k and v (and rotated q) before an output is stored,
a launch whose workgroups read and store in no order has not.  Every step that may be one launch, `out` over k, over v and over q a
head further on, with many more workgroups than the GPU runs at once, against the oracle; over q itself as it is."""
import numpy as np
import pytest

import gen
from test_gpu_parity import D, TOL, assert_bytes_equal, dev, host, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("over", ["k", "v", "q, a head on", "q"])
@pytest.mark.parametrize("call,bits", [("step", 4), ("step", 2), ("step", 0), ("paged", 4), ("paged", 2), ("attend", 4)])
def test_outputs_over_inputs(oracle, rotation_fixture, call, bits, over):
    import torch
    from triebwerk_amd import kvcache as kv
    if call == "attend" and over in "kv": pytest.skip("no k and v")
    if bits == 0 and over.startswith("q"): pytest.skip("fp16 attention reads q where it stores, as the reference's does")
    H, Hk, G, msl = 16, 8, 400, 272
    qd, kd = H * D, Hk * D
    r = gen.rng(5700 + bits + len(over))
    pos = r.integers(0, 40, G).astype(np.int32)
    width = kd * bits // 8 if bits else kd
    c = [r.integers(0, 256, (G, msl, width), dtype=np.uint8) if bits else gen.normal_f16(r, (G, msl, width)) for _ in range(2)]
    if bits: c += [(11.3 + 0.7 * r.standard_normal((G, msl, Hk))).astype(np.float16) for _ in range(2)]
    q, k, v = (gen.normal_f16(r, (G, n)) for n in (qd, kd, kd))
    # one buffer; every input as near its start as the outputs', which begin D halves in
    flat = torch.zeros(G * qd + 2 * D, dtype=torch.float16, device="cuda")
    d_in = {"q": dev(q).view(-1), "k": dev(k).view(-1), "v": dev(v).view(-1)}
    out = flat[D:D + G * qd]
    name = over[0]
    n = d_in[name].numel()
    at = 0 if "head" in over else D
    flat[at:at + n].copy_(d_in[name])
    d_in[name] = flat[at:at + n]
    d = [dev(x) for x in c]
    scratch = torch.zeros(max(G * H * msl, kv.attention_workspace_floats(G, H, msl)), dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    rot, p = dev(rotation_fixture), dev(pos)
    kv.set_fused_shape(2, 0)             # two KV heads to a workgroup, 1600 of them
    try:
        if call == "paged":
            table = dev(np.arange(G * msl // 16, dtype=np.int32))
            kv.tw_paged_turbo_append_attention_batch(out, d_in["q"], d_in["k"], d_in["v"], *d, rot, scratch, p, table, msl // 16, msl, G, H, Hk, D, qd, kd, bits)
        elif call == "attend":
            kv.launch_turbo_gqa_attention_batch(out, d_in["q"], *d, rot, scratch, p, msl, G, H, Hk, D, qd, kd, bits)
        elif bits:
            kv.tw_turbo_append_attention_batch(out, d_in["q"], d_in["k"], d_in["v"], *d, rot, scratch, p, msl, G, H, Hk, D, qd, kd, bits)
        else:
            kv.tw_append_attention_batch(out, d_in["q"], d_in["k"], d_in["v"], *d, scratch, p, msl, G, H, Hk, D, qd, kd)
    finally:
        kv.set_fused_shape(0, 0)
    torch.cuda.synchronize()
    want = np.zeros((G, qd), np.float16)
    if bits == 0:
        oracle.kv_cache_write_batch(c[0], c[1], k, v, pos, msl, G, kd)
        oracle.gqa_attention_batch(want, q, *c, pos, msl, G, H, Hk, D, qd, kd)
    else:
        if call != "attend":
            oracle.turbo_kv_quantize_batch(c[0], c[2], k, rotation_fixture, pos, msl, G, Hk, D, kd, bits)
            oracle.turbo_kv_quantize_batch(c[1], c[3], v, rotation_fixture, pos, msl, G, Hk, D, kd, bits)
        oracle.turbo_gqa_attention_batch(want, q, *c, rotation_fixture, pos, msl, G, H, Hk, D, qd, kd, bits)
    for got, x, what in zip(d, c, ("K", "V", "K norms", "V norms")):
        assert_bytes_equal(host(got), x, what)
    assert rel_err(host(out), want) <= TOL
    if over == "q" and bits: assert "decode_fused_kernel" in kv.last_scan_kernel()
