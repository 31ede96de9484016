"""Engine.broadcast_prefix over every layer at once: the rows of each layer reach every destination and nothing else changes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kv_bits,Hk,L,G,src,dst,T", [
    (4, 8, 3, 19, 5, (0, 19), 37),      # more destinations than a thread's group of eight, source among them
    (4, 1, 2, 10, 0, (1, 10), 5),       # norm rows of two bytes: the narrow copy
    (2, 2, 4, 9, 8, (0, 8), 64),        # exactly one group
    (0, 2, 1, 18, 17, (0, 17), 3),      # one layer, 16-byte rows
    (4, 8, 2, 3, 1, (0, 3), 1000),      # more bytes than the grid covers in one pass
])
def test_every_layer_and_destination(kv_bits, Hk, L, G, src, dst, T):
    import torch
    from triebwerk_amd import Engine
    msl = T + 3
    eng = Engine(max_seq_len=msl, kv_bits=kv_bits)
    eng.set_shape(L, Hk, Hk)
    eng.alloc_batch(G, msl)
    g = torch.Generator(device="cuda"); g.manual_seed(5)
    want = []
    for l in range(L):
        for t in eng.cache(l):
            if t is None:
                continue
            flat = t.view(-1).view(torch.uint8)
            flat.copy_(torch.randint(0, 256, flat.shape, generator=g, device="cuda", dtype=torch.uint8))
            w = t.view(torch.uint8).cpu().numpy().reshape(G, msl, -1).copy()
            w[dst[0]:dst[1], :T] = w[src, :T]
            want.append((t, w))
    eng.broadcast_prefix(src, dst[0], dst[1], T)
    torch.cuda.synchronize()
    for t, w in want:
        assert np.array_equal(t.view(torch.uint8).cpu().numpy().reshape(w.shape), w)
