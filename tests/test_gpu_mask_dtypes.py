"""Masks read as stored (bool, bf16, fp16, fp32; any row pitch and start) against the fp32 mask of the same values.

A mask's values are exact in fp32 and enter the scores by the same arithmetic whichever type they are read from,
so the outputs are the same bits; the fp32 form itself is compared with the oracle.
"""
import numpy as np
import pytest
import torch

from oracle import sdpa as orc
from tests.attn_cases import LSE_TOL, O_TOL_BF16, host, lse_rel, max_abs, randn, rounded, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,L,S,D,causal,start,pitch", [
    (torch.bfloat16, 77, 77, 64, False, 0, 77),     # odd pitch: rows start at every byte of a word
    (torch.float16, 130, 65, 64, True, 3, 67),      # one key past a tile, unaligned start
    (torch.bfloat16, 64, 128, 128, False, 1, 129),
    (torch.float16, 33, 31, 128, True, 2, 31),      # fewer keys than a tile
    (torch.bfloat16, 90, 200, 48, False, 5, 203),   # padded head dim
    (torch.float32, 77, 77, 64, False, 1, 77),
    (torch.float32, 200, 97, 128, True, 0, 101),
    (torch.float32, 20, 260, 36, False, 3, 261),
])
def test_mask_dtypes(dtype, L, S, D, causal, start, pitch):
    import dtorch_amd.nn.functional as F
    rng = np.random.default_rng(L * S)
    B, Hq, Hkv = 2, 4, 2
    q, k, v = randn(rng, (B, Hq, L, D)), randn(rng, (B, Hkv, S, D)), randn(rng, (B, Hkv, S, D))
    tq, tk, tv = to_dev(q, dtype), to_dev(k, dtype), to_dev(v, dtype)

    def run(m):
        o, lse = F.scaled_dot_product_attention_with_lse(tq, tk, tv, is_causal=causal, enable_gqa=True, attn_mask=m)
        torch.cuda.synchronize()
        return o, lse

    def placed(m, t):
        """m [B, 1, L, S] as a view of a flat buffer: rows `pitch` apart, first element at `start`."""
        buf = torch.zeros(start + B * L * pitch + S, dtype=t, device="cuda")
        w = torch.as_strided(buf, (B, 1, L, S), (L * pitch, L * pitch, pitch, 1), start)
        w.copy_(m)
        return w

    keep = torch.from_numpy(rng.random((B, 1, L, S)) < 0.6).cuda()
    keep[:, :, L // 2] = False  # a hidden row
    hide = torch.zeros(B, 1, L, S, device="cuda").masked_fill_(~keep, float("-inf"))
    o, lse = run(hide)
    for got in (run(placed(keep, torch.bool)), run(placed(hide, torch.float32))):
        assert torch.equal(got[0], o) and torch.equal(got[1], lse)
    ro, rl = orc.sdpa_fwd(rounded(q, dtype), rounded(k, dtype), rounded(v, dtype), attn_mask=keep.cpu().numpy(),
                          is_causal=causal, enable_gqa=True)
    assert max_abs(host(o), ro) <= (1e-5 if dtype == torch.float32 else O_TOL_BF16)
    assert lse_rel(host(lse), rl) <= (1e-5 if dtype == torch.float32 else LSE_TOL)
    for t in (torch.bfloat16, torch.float16):
        add = torch.from_numpy(rng.standard_normal((B, 1, L, S)).astype(np.float32)).cuda().to(t)
        add.masked_fill_(~keep, torch.finfo(t).min)
        o, lse = run(add.float())
        got = run(placed(add, t))
        assert torch.equal(got[0], o) and torch.equal(got[1], lse)
    # one row for all queries and heads; a mask without a unit key stride; one value for all keys
    row = keep[:, :, :1]
    o, lse = run(row.expand(B, Hq, L, S).contiguous())
    for m in (row, row.transpose(2, 3).contiguous().transpose(2, 3), row.double().log()):
        got = run(m)
        assert torch.equal(got[0], o) and torch.equal(got[1], lse)
    o, lse = run(keep[:, :, :, :1].expand(B, 1, L, S).contiguous())
    got = run(keep[:, :, :, :1])
    assert torch.equal(got[0], o) and torch.equal(got[1], lse)


@pytest.mark.parametrize("dtype,B,Hq,L,S,D,causal", [
    (torch.bfloat16, 2, 4, 130, 97, 64, True),
    (torch.float16, 2, 4, 77, 200, 128, False),
    (torch.bfloat16, 8, 8, 1024, 1501, 128, True),   # one row for all queries: read once into fp32 rows
    (torch.float16, 8, 8, 1024, 1501, 128, False),
    (torch.bfloat16, 16, 8, 1024, 1501, 64, False),  # a large row without spans: converted first
    (torch.bfloat16, 1, 2, 33, 70, 256, False),      # wide heads: likewise
    (torch.float32, 1, 2, 90, 100, 64, False),       # key-split fp32 form
    (torch.float32, 4, 192, 200, 300, 64, True),     # 128-row fp32 form
])
def test_bool_bytes(dtype, B, Hq, L, S, D, causal):
    """Bytes of a bool mask other than 0 and 1 (a uint8 tensor viewed as bool): any non-zero byte keeps its key."""
    import dtorch_amd.nn.functional as F
    g = torch.Generator(device="cuda").manual_seed(L + S)
    q, k, v = (torch.randn(B, h, n, D, device="cuda", generator=g).to(dtype) for h, n in ((Hq, L), (Hq // 2, S), (Hq // 2, S)))
    rows = 1 if L == 1024 else L
    at = torch.randint(0, 7, (B, 1, rows, S), device="cuda", generator=g)
    raw = torch.tensor([0, 1, 2, 4, 128, 254, 255], dtype=torch.uint8, device="cuda")[at]
    raw[0, :, 0, :64] = 255   # a tile that every byte keeps
    kw = dict(is_causal=causal, enable_gqa=True)
    o, lse = F.scaled_dot_product_attention_with_lse(q, k, v, attn_mask=raw.view(torch.bool), **kw)
    ro, rl = F.scaled_dot_product_attention_with_lse(q, k, v, attn_mask=raw != 0, **kw)
    torch.cuda.synchronize()
    assert torch.equal(o, ro) and torch.equal(lse, rl)


@pytest.mark.parametrize("heads", [1, 16])
def test_large_mask_of_a_row_per_query(heads):
    """Not causal at D = 128 from 2^27 pairs on: a mask that the heads share is converted first, one per head is not."""
    import dtorch_amd.nn.functional as F
    g = torch.Generator(device="cuda").manual_seed(heads)
    H, S = 16, 2900
    assert H * S * S >= 2 ** 27
    q, k, v = (torch.randn(1, h, S, 128, device="cuda", generator=g).to(torch.bfloat16) for h in (H, 4, 4))
    m = torch.randn(1, heads, S, S, device="cuda", generator=g).to(torch.bfloat16)
    m.masked_fill_(torch.rand(m.shape, device="cuda", generator=g) < 0.2, float("-inf"))
    o, lse = F.scaled_dot_product_attention_with_lse(q, k, v, attn_mask=m, enable_gqa=True)
    ro, rl = F.scaled_dot_product_attention_with_lse(q, k, v, attn_mask=m.float(), enable_gqa=True)
    torch.cuda.synchronize()
    assert torch.equal(o, ro) and torch.equal(lse, rl)
