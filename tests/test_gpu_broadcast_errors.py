"""What Engine.broadcast_prefix reports: a bad range with the library's message, nothing for an empty broadcast, and not the error
that some other HIP call left on the thread."""
import pytest

pytestmark = pytest.mark.gpu


def test_broadcast_reports_its_own_errors():
    import torch
    from triebwerk_amd import Engine, _lib
    lib = _lib.load()
    eng = Engine(max_seq_len=8, kv_bits=4)
    eng.set_shape(2, 2, 2)
    eng.alloc_batch(4, 8)
    lib.tw_kv_clear_error()
    h = eng._h
    assert lib.tw_engine_broadcast_prefix(h, 0, 3, 1, 4, None) == -2
    assert lib.tw_kv_last_error() != 0 and b"destinations 3 to 1" in lib.tw_kv_last_error_string()
    lib.tw_kv_clear_error()
    with pytest.raises(RuntimeError, match="destinations 3 to 1"):
        eng.broadcast_prefix(0, 3, 1, 4)
    assert lib.tw_kv_last_error() == 0
    # an earlier call's HIP error (a device that does not exist: refused by the runtime) is not this call's failure
    for src, lo, hi, T in ((0, 1, 4, 4), (0, 1, 4, 0), (1, 1, 2, 4)):
        assert lib.hipSetDevice(99) != 0
        assert lib.tw_engine_broadcast_prefix(h, src, lo, hi, T, None) == 0
        lib.tw_kv_clear_error()
    lib.hipGetLastError()
    torch.cuda.synchronize()
