"""The compressed append on both sides of the number of vectors where the launch changes from rotate_kernel to tiles shared by a
workgroup (3 vectors per compute unit at 4 bit, 8 at 2 bit), one stream and two, token list and batch: the oracle's bytes."""
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


@pytest.mark.parametrize("bits", [4, 2])
@pytest.mark.parametrize("Hk,streams,batch", [(8, 2, False), (8, 1, False), (1, 1, True), (3, 2, True)])
@pytest.mark.parametrize("past", [0, 1])
def test_both_kernels(oracle, rotation_fixture, bits, Hk, streams, batch, past):
    import torch
    from triebwerk_amd import kvcache as kv
    per_row = Hk * streams
    N = (3 if bits == 4 else 8) * torch.cuda.get_device_properties(0).multi_processor_count // per_row + past
    r = gen.rng(7400 + N)
    kv_dim = Hk * D
    src = [gen.kv_rows_with_outliers(r, (N, kv_dim), kv_dim)[0] for _ in range(streams)]
    lead, msl = ((N, 2), 2) if batch else ((N + 3,), N + 3)
    pos = r.integers(0, 2, N).astype(np.int32) if batch else r.permutation(msl)[:N].astype(np.int32)
    want = [(np.zeros((*lead, kv_dim * bits // 8), np.uint8), np.zeros((*lead, Hk), np.float16)) for _ in range(streams)]
    got = [tuple(dev(x) for x in w) for w in want]
    for s, (c, n) in zip(src, want):
        if batch:
            oracle.turbo_kv_quantize_batch(c, n, s, rotation_fixture, pos, msl, N, Hk, D, kv_dim, bits)
        else:
            oracle.turbo_kv_quantize(c, n, s, rotation_fixture, pos, msl, N, Hk, D, kv_dim, bits)
    rot, dp, d = dev(rotation_fixture), dev(pos), [dev(s) for s in src]
    if streams == 2:
        call = kv.tw_turbo_kv_append_batch if batch else kv.tw_turbo_kv_append_tokens
        call(*got[0], *got[1], d[0], d[1], rot, dp, msl, N, Hk, D, kv_dim, bits)
    elif batch:
        kv.launch_turbo_kv_quantize_batch(*got[0], d[0], rot, dp, msl, N, Hk, D, kv_dim, bits)
    else:
        kv.launch_turbo_kv_quantize(*got[0], d[0], rot, dp, msl, N, Hk, D, kv_dim, bits)
    torch.cuda.synchronize()
    for g, w in zip(got, want):
        for a, b in zip(g, w):
            same_bytes(a, b)


@pytest.mark.parametrize("bits,T,Hk", [(4, 1366, 8), (2, 2303, 8), (4, 3500, 8), (4, 4097, 8), (2, 5001, 8)])
def test_tiles_per_workgroup(oracle, rotation_fixture, bits, T, Hk):
    """Sizes that give a workgroup 2, 3, 2, 3 and 4 tiles on 256 compute units, the last run ragged."""
    from triebwerk_amd import kvcache as kv
    r = gen.rng(7500 + T)
    kv_dim, msl = Hk * D, T + 1
    k, v = (gen.normal_f16(r, (T, kv_dim)) for _ in range(2))
    pos = r.permutation(msl)[:T].astype(np.int32)
    want = [(np.zeros((msl, kv_dim * bits // 8), np.uint8), np.zeros((msl, Hk), np.float16)) for _ in range(2)]
    got = [tuple(dev(x) for x in w) for w in want]
    for s, (c, n) in zip((k, v), want):
        oracle.turbo_kv_quantize(c, n, s, rotation_fixture, pos, msl, T, Hk, D, kv_dim, bits)
    kv.tw_turbo_kv_append_tokens(*got[0], *got[1], dev(k), dev(v), dev(rotation_fixture), dev(pos), msl, T, Hk, D, kv_dim, bits)
    for g, w in zip(got, want):
        for a, b in zip(g, w):
            same_bytes(a, b)
