"""dtattn_prefill_masked called through the C ABI: what it must refuse (on the host, before any launch), and one call
with and without its workspace against the operator."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

BF16, FP16, FP8, FP32, BOOL = 0, 1, 2, 3, 4
INVALID, UNSUPPORTED = 1, 2


class Mask(ctypes.Structure):
    _fields_ = [("data", ctypes.c_void_p), ("stride", ctypes.c_int64 * 3), ("dtype", ctypes.c_int32)]


def _lib():
    from dtorch_amd import _lib as L
    lib = L.cabi()
    lib.dtattn_last_error.restype = ctypes.c_char_p
    lib.dtattn_prefill_masked.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p]
    lib.dtattn_prefill_masked_workspace_size.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
    lib.dtattn_prefill_masked_workspace_size.restype = ctypes.c_size_t
    return lib


def _call(B, H, L, S, D, seed=0):
    from dtorch_amd._lib import PrefillArgs
    g = torch.Generator(device="cuda").manual_seed(seed)
    q, k, v = (torch.randn(B, H, n, D, device="cuda", generator=g).to(torch.bfloat16) for n in (L, S, S))
    o, lse = torch.zeros_like(q), torch.zeros(B, H, L, device="cuda")
    keep = torch.ones(B, 1, 1, S, dtype=torch.bool, device="cuda")
    keep[0, ..., : S // 3] = False
    a = PrefillArgs()
    a.q, a.k, a.v, a.o, a.lse = (t.data_ptr() for t in (q, k, v, o, lse))
    a.B, a.Hq, a.Hkv, a.Sq, a.Sk, a.D, a.Dv = B, H, H, L, S, D, D
    for dst, t in ((a.q_stride, q), (a.k_stride, k), (a.v_stride, v), (a.o_stride, o)):
        dst[:] = [t.stride(0), t.stride(1), t.stride(2)]
    a.lse_stride[:] = [H * L, L]
    m = Mask(keep.data_ptr(), (ctypes.c_int64 * 3)(S, 0, 0), BOOL)
    return a, m, (q, k, v, keep, o, lse)


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


@pytest.mark.parametrize("what,status,text", [
    ("two masks", INVALID, b"two masks"), ("null data", INVALID, b"null"), ("off its elements", INVALID, b"aligned"),
    ("dtype", UNSUPPORTED, b"mask dtype"), ("fp8 inputs", UNSUPPORTED, b"fp8"), ("head dim", UNSUPPORTED, b"128"),
    ("negative stride", UNSUPPORTED, b"negative"), ("slab", UNSUPPORTED, b"4 GB"),
])
def test_refused(what, status, text):
    lib = _lib()
    a, m, keep_alive = _call(1, 2, 40, 50, 136 if what == "head dim" else 64)
    if what == "two masks":
        a.mask = keep_alive[5].data_ptr()
    elif what == "null data":
        m.data = None
    elif what == "off its elements":
        m.dtype, m.data = FP32, m.data + 2
    elif what == "dtype":
        m.dtype = 7
    elif what == "fp8 inputs":
        a.dtype = FP8
    elif what == "negative stride":
        m.stride[2] = -50
    elif what == "slab":
        m.stride[2] = 1 << 31
    assert lib.dtattn_prefill_masked(ctypes.byref(a), ctypes.byref(m), _stream()) == status
    assert text in lib.dtattn_last_error()
    torch.cuda.synchronize()
    assert not keep_alive[4].any() and not keep_alive[5].any()  # nothing ran


def test_workspace_is_optional():
    import dtorch_amd.nn.functional as F
    lib = _lib()
    a, m, (q, k, v, keep, o, lse) = _call(4, 4, 2048, 2048, 128)
    ro, rl = F.scaled_dot_product_attention_with_lse(q, k, v, attn_mask=keep)
    need = lib.dtattn_prefill_masked_workspace_size(ctypes.byref(a), ctypes.byref(m))
    assert need > 0
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    for given in (need, need - 1, 0):
        a.workspace, a.workspace_bytes = (ws.data_ptr(), given) if given else (None, 0)
        assert lib.dtattn_prefill_masked(ctypes.byref(a), ctypes.byref(m), _stream()) == 0, lib.dtattn_last_error()
        torch.cuda.synchronize()
        if given == need:
            assert torch.equal(o, ro) and torch.equal(lse, rl)  # as the operator runs it
        # without spans the key tiles of batch 0 start elsewhere: P and O round differently (as test_gpu_mask_spans.py)
        assert (o.float() - ro.float()).abs().max() <= 8e-3 and (lse - rl).abs().max() <= 1e-4
        assert torch.equal(o[1:], ro[1:]) or given != need
        o.zero_(), lse.zero_()
