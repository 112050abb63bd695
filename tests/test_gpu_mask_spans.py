"""Large calls with one mask row for all queries (padding masks): key spans against the same mask spelled out per query.

The spelled-out mask runs on prefill_fwd_kernel tile by tile; the row form finds each batch's span of visible keys
and runs it as a shorter call, whose key tiles start elsewhere.  Both round P and O to the input type, so they agree
within the bound the stream-K tests use (8e-3 on O of unit normals, 1e-5 on the LSE); batches without a span run
the same kernel on the same values and must agree bit for bit.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,Hq,Hkv,D,causal,q_off,kind", [
    (torch.bfloat16, 8, 2, 128, True, 0, "bool"),    # persistent grouped-query form
    (torch.float16, 8, 4, 128, True, 300, "float"),  # row form, diagonal moved
    (torch.bfloat16, 8, 2, 128, False, 0, "same"),
    (torch.float16, 8, 8, 128, False, 0, "bool"),
    (torch.bfloat16, 16, 4, 64, True, 0, "bool"),    # no span form at this head dim: the row mask in fp32
    (torch.float16, 8, 2, 96, False, 0, "bool"),     # padded head dim: likewise
])
def test_spans(dtype, Hq, Hkv, D, causal, q_off, kind):
    import dtorch_amd.nn.functional as F
    B, L, S = 8, 1024, 1501
    if D < 128:
        B = 16
    g = torch.Generator(device="cuda").manual_seed(Hq * D + causal)
    q = torch.randn(B, L, Hq, D, device="cuda", generator=g).to(dtype).transpose(1, 2)
    k = torch.randn(B, Hkv, S, D, device="cuda", generator=g).to(dtype)
    v = torch.randn(B, Hkv, S, D, device="cuda", generator=g).to(dtype)
    keep = torch.ones(B, 1, 1, S, dtype=torch.bool, device="cuda")
    keep[0, ..., :37] = False                # left padding
    keep[1, ..., 1000:] = False              # right padding
    keep[2, ..., :700] = keep[2, ..., 703:] = False
    keep[3] = False                          # nothing visible
    keep[4, ..., 64] = False                 # a hole: no span
    keep[5, ..., 0] = keep[5, ..., -1] = False
    keep[6, ..., ::2] = False
    whole = [4, 6]                           # batches without a span
    m = keep
    if kind != "bool":
        m = torch.zeros(B, 1, 1, S, device="cuda", dtype=torch.float32 if kind == "float" else dtype)
        m.masked_fill_(~keep, float("-inf"))
        m[7, ..., 5] = 0.5                   # a bias: no span
        whole.append(7)
    kw = dict(is_causal=causal, enable_gqa=True, q_offset=q_off)
    o, lse = F.scaled_dot_product_attention_with_lse(q, k, v, attn_mask=m, **kw)
    dense = (m if kind != "bool" else torch.zeros(m.shape, device="cuda").masked_fill_(~m, float("-inf"))).float()
    ro, rl = F.scaled_dot_product_attention_with_lse(q, k, v, attn_mask=dense.expand(B, 1, L, S).contiguous(), **kw)
    torch.cuda.synchronize()
    assert torch.equal(torch.isneginf(lse), torch.isneginf(rl))
    assert torch.isneginf(rl[3]).all() and (o[3] == 0).all()
    fin = ~torch.isneginf(rl)
    assert ((lse - rl)[fin].abs() / rl[fin].abs().clamp(min=1)).max() <= 1e-5
    assert (o.float() - ro.float()).abs().max() <= 8e-3
    for b in whole:
        assert torch.equal(o[b], ro[b]) and torch.equal(lse[b], rl[b])
    if D < 128:
        assert torch.equal(o, ro) and torch.equal(lse, rl)
