"""A decode step captured at a short context and replayed as the context grows: the captured step must hold the launches
that the context at hand asks for -- the heads per workgroup and the number of workgroups that share a sequence, not only
one launch against three -- so a replay gives the very bits of the eager step, which chooses anew every time."""
import pytest

pytestmark = pytest.mark.gpu

D = 128


@pytest.mark.parametrize("bits,H,Hk,G", [(4, 16, 8, 1), (4, 16, 8, 4), (2, 32, 8, 2), (4, 16, 8, 24)])
def test_replay_is_the_eager_step_at_every_length(layers_apart, bits, H, Hk, G):
    import torch
    from triebwerk_amd import Engine, _lib, kvcache
    lib = _lib.load()
    L, msl = 2, 16384
    eng = Engine(max_seq_len=msl, kv_bits=bits)
    eng.set_shape(L, H, Hk, D)
    eng.alloc_batch(G, msl)
    gt = torch.Generator(device="cuda"); gt.manual_seed(19)
    for l in range(L):
        c = eng.cache(l)
        for i in range(2):
            c[i].copy_(torch.randint(0, 256, c[i].shape, generator=gt, device="cuda", dtype=torch.uint8))
        for i in (2, 3):
            c[i].copy_((11.3 + 0.7 * torch.randn(c[i].shape, generator=gt, device="cuda")).to(torch.float16))
    q = 2 * torch.randn((L, G, H * D), generator=gt, device="cuda", dtype=torch.float16)
    k, v = (torch.randn((L, G, Hk * D), generator=gt, device="cuda", dtype=torch.float16) for _ in range(2))
    out = torch.zeros_like(q)
    forms = set()
    for ctx in (500, 501, 3000, 4097, 8193, 16000, 16001, 500):
        eng.set_positions([ctx - 1] * G)
        recorded = lib.tw_kv_decode_fused_launches()
        eng.decode_step(q, k, v, out, use_graph=True)
        recorded = lib.tw_kv_decode_fused_launches() - recorded
        assert eng.graph_state() == 1
        if ctx in (501, 16001):
            assert recorded == 0, "a step one token on was captured again"
        replayed = out.clone()
        eng.set_positions([ctx - 1] * G)
        eng.decode_step(q, k, v, out, use_graph=False)
        torch.cuda.synchronize()
        forms.add(kvcache.last_scan_kernel())
        assert torch.equal(replayed, out), f"context {ctx}: the replayed step is not the eager step's form"
    assert len(forms) > 1 and not any("decode_layers_kernel" in f for f in forms), forms
    assert G > 4 or any("context shared" in f for f in forms), forms


@pytest.mark.parametrize("bits,H,Hk,G,L", [(4, 16, 8, 1, 28), (2, 16, 8, 5, 28)])
def test_every_layer_in_one_launch_is_captured_again_only_for_another_launch(bits, H, Hk, G, L):
    """While every layer goes into the same one launch, what a layer by itself would take does not matter to the fixed step: nothing is planned
    or counted anew for it (a launch needs no capture), and it gives the very bits of the eager step."""
    import torch
    from triebwerk_amd import Engine, _lib, kvcache
    lib = _lib.load()
    msl = 4096
    eng = Engine(max_seq_len=msl, kv_bits=bits)
    eng.set_shape(L, H, Hk, D)
    eng.alloc_batch(G, msl)
    q = torch.randn((L, G, H * D), device="cuda").half()
    k, v = (torch.randn((L, G, Hk * D), device="cuda").half() for _ in range(2))
    out = torch.zeros_like(q)
    torch.cuda.synchronize()
    last, same = None, 0
    for ctx in range(40, 4000, 33):
        eng.set_positions([ctx - 1] * G)
        eng.decode_step(q, k, v, out, use_graph=False)
        name = kvcache.last_scan_kernel()
        eager = out.clone()
        out.zero_()
        eng.set_positions([ctx - 1] * G)
        recorded = lib.tw_kv_decode_fused_launches()
        eng.decode_step(q, k, v, out, use_graph=True)
        recorded = lib.tw_kv_decode_fused_launches() - recorded
        assert eng.graph_state() == 1
        assert kvcache.last_scan_kernel() == name and torch.equal(eager, out), f"context {ctx}: the fixed step is not the eager one"
        if name == last and "decode_layers_kernel" in name:
            same += 1
            assert recorded == 0, f"context {ctx}: {name} fixed again"
        last = name
    torch.cuda.synchronize()
    assert same > 20
