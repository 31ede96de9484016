"""The prompt kernels' forms with two groups of waves (2 and 3), whose groups take turns with the context's tiles and add up
their sums at the end, and the eight-wave forms without mirrored pairs (7 and 8), against the oracle."""
import numpy as np
import pytest

import gen
from test_gpu_parity import D, TOL, build_fp16_cache, build_turbo_cache, dev, host, kv, rel_err  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", [2, 3, 7, 8])
@pytest.mark.parametrize("R,T", [(2, 1), (2, 16), (2, 31), (2, 32), (2, 33), (2, 48), (2, 64), (2, 65), (1, 127), (1, 129), (4, 97), (4, 160), (2, 515)])
@pytest.mark.parametrize("bits", [0, 4, 2])
def test_groups_of_waves_and_unpaired_blocks(kv, oracle, rotation_fixture, bits, R, T, form):  # noqa: F811
    """Lengths around the tiles of 32 tokens: a group may have no tile at all, one whose tokens all lie behind some of its
    queries, or one tile less than the other; blocks may be ragged."""
    import torch
    Hk = 2
    H = Hk * R
    r = gen.rng(2100 + 13 * R + T + bits)
    msl = T + 3
    kv_dim, q_dim = Hk * D, H * D
    q = gen.normal_f16(r, (T, q_dim))
    want = np.zeros((T, q_dim), np.float16)
    out = torch.zeros((T, q_dim), dtype=torch.float16, device="cuda")
    kv.set_prefill_form(form)
    try:
        if bits:
            ck, cv, kn, vn = build_turbo_cache(oracle, rotation_fixture, r, 1, Hk, msl, [T], bits)
            oracle.turbo_gqa_prefill_attention(want, q, ck[0], cv[0], kn[0], vn[0], rotation_fixture, T, msl, H, Hk, D, q_dim, kv_dim, bits)
            kv.launch_turbo_gqa_prefill_attention(out, dev(q), dev(ck[0]), dev(cv[0]), dev(kn[0]), dev(vn[0]),
                                                  dev(rotation_fixture), None, T, msl, H, Hk, D, q_dim, kv_dim, bits)
        else:
            ck, cv = build_fp16_cache(r, 1, msl, kv_dim)
            oracle.gqa_prefill_attention(want, q, ck[0], cv[0], T, msl, H, Hk, D, q_dim, kv_dim)
            kv.launch_gqa_prefill_attention(out, dev(q), dev(ck[0]), dev(cv[0]), None, T, msl, H, Hk, D, q_dim, kv_dim)
    finally:
        kv.set_prefill_form(0)
    assert rel_err(host(out), want) <= TOL
