"""The one-launch decode step with a sequence's context shared by 16 to 64 workgroups: shares that hold one tile or none,
merge slots that take one share, several, or more than eight each, and the rule that picks the form for small batches."""
import numpy as np
import pytest

import gen
from test_gpu_parity import D, TOL, assert_bytes_equal, build_turbo_cache, dev, host, kv, rel_err  # noqa: F401


@pytest.mark.gpu
@pytest.mark.parametrize("bits,H,Hk,G", [(4, 16, 8, 2), (2, 32, 8, 2), (4, 4, 4, 3), (4, 12, 3, 2)])
@pytest.mark.parametrize("hkw,shares", [(1, 16), (1, 64), (2, 32), (2, 64), (4, 16), (8, 64)])
def test_many_shares_against_the_oracle(kv, oracle, rotation_fixture, bits, H, Hk, G, hkw, shares):  # noqa: F811
    import torch
    if Hk % hkw:
        pytest.skip("heads per workgroup must divide the KV heads")
    msl = 8704
    kv_dim, q_dim = Hk * D, H * D
    r = gen.rng(7700 + 10 * bits + H + hkw + shares)
    lens = [msl - 5, 31, 2047][:G] if (hkw + shares) % 3 else [64 * 32 - 1, 5000, 0][:G]
    ck, cv, kn, vn = build_turbo_cache(oracle, rotation_fixture, r, G, Hk, msl, lens, bits)
    d_c = [dev(x) for x in (ck, cv, kn, vn)]
    scratch = torch.full((G * H * msl,), float("nan"), dtype=torch.float32, device="cuda")
    tickets = torch.zeros(G * Hk, dtype=torch.int32, device="cuda")
    pos = np.array(lens, np.int32)
    kv.set_decode_fused(1)
    kv.set_fused_shape(hkw, shares)
    try:
        for step in range(2):
            q = gen.normal_f16(r, (G, q_dim)); k = gen.kv_rows_with_outliers(r, (G, kv_dim), kv_dim)[0]; v = gen.normal_f16(r, (G, kv_dim))
            out = torch.zeros((G, q_dim), dtype=torch.float16, device="cuda")
            kv.tw_layer_attention_step(out, dev(q), dev(k), dev(v), dev(pos), msl, G, H, Hk, D, q_dim, kv_dim, d_c[0], d_c[1],
                                       scratch, kv_bits=bits, k_norms=d_c[2], v_norms=d_c[3], rotation=dev(rotation_fixture), tickets=tickets)
            assert "context shared" in kv.last_scan_kernel()
            oracle.turbo_kv_quantize_batch(ck, kn, k, rotation_fixture, pos, msl, G, Hk, D, kv_dim, bits)
            oracle.turbo_kv_quantize_batch(cv, vn, v, rotation_fixture, pos, msl, G, Hk, D, kv_dim, bits)
            want = np.zeros((G, q_dim), np.float16)
            oracle.turbo_gqa_attention_batch(want, q, ck, cv, kn, vn, rotation_fixture, pos, msl, G, H, Hk, D, q_dim, kv_dim, bits)
            got = host(out)
            assert max(rel_err(got[g], want[g]) for g in range(G)) <= TOL
            assert not host(tickets).any(), "tickets were not left zero"
            pos = pos + 1
    finally:
        kv.set_fused_shape(0, 0)
        kv.set_decode_fused(0)
    for got, want_arr, what in zip(d_c, (ck, cv, kn, vn), ("K codes", "V codes", "K norms", "V norms")):
        assert_bytes_equal(host(got), want_arr, what)


def test_small_ragged_batches_share_their_longest_sequence():
    """With tickets a small ragged batch takes one launch (its longest sequence shared by workgroups); without them, or when
    the batch fills the compute units by itself, it stays on the balanced walk."""
    from triebwerk_amd import _lib
    plan2 = _lib.load().tw_kv_decode_step_plan2
    assert plan2(4, 16, 8, 4, 8448, 512, 8192, 1) == 1 and plan2(4, 16, 8, 4, 8448, 512, 8192, 0) == 0
    assert plan2(1, 16, 8, 4, 16384, 16001, 16001, 1) == 1
    assert plan2(48, 16, 8, 2, 8448, 300, 8000, 1) == 0
