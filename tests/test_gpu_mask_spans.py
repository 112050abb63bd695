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


@pytest.mark.parametrize("dtype,D,causal,kind,batches,heads,S", [
    (torch.bfloat16, 128, True, "bool", 8, 1, 2049),   # one key past a round of the span search
    (torch.float16, 128, False, "float", 8, 1, 2049),
    (torch.bfloat16, 128, True, "same", 8, 1, 4097),
    (torch.float16, 128, True, "bool", 1, 1, 4097),    # one row for the batch
    (torch.bfloat16, 128, True, "bool", 8, 8, 1501),   # a row per head: no spans
    (torch.float16, 128, False, "same", 1, 8, 1501),
    (torch.bfloat16, 64, True, "same", 8, 8, 1501),
    (torch.bfloat16, 64, False, "bool", 8, 8, 2049),
    (torch.float16, 96, False, "same", 8, 1, 1501),
])
def test_long_rows_and_rows_per_head(dtype, D, causal, kind, batches, heads, S):
    """Row masks whose spans end on either side of the 2048 keys that the span search reads at once, and row masks
    that differ by head (as stored, or converted first): as above, against the mask spelled out per query.  Rows with a
    few visible keys have |O| up to that of a unit normal (4), whose rounding to bf16 moves it by up to 2^-7 of its size:
    that is added to the bound of O below 1."""
    import dtorch_amd.nn.functional as F
    B, H, L = 8, 8, 1024
    g = torch.Generator(device="cuda").manual_seed(S * D + heads)
    q, k, v = (torch.randn(B, h, n, D, device="cuda", generator=g).to(dtype) for h, n in ((H, L), (2, S), (2, S)))
    edges = [x for x in (0, 1, 63, 64, 65, 2046, 2047, 2048, 2049, 4095, 4096) if x < S]
    keep = torch.ones(batches, heads, 1, S, dtype=torch.bool, device="cuda")
    for i, row in enumerate(keep.flatten(0, 2)):
        row[:edges[i % len(edges)]] = False
        if i % 3 == 1:
            row[edges[-1 - i % 4] + 1:] = False
        if i % 5 == 4:
            row[edges[-1]] = False  # a hole, unless the span ends before it
    m = keep
    if kind != "bool":
        m = torch.zeros(keep.shape, device="cuda", dtype=torch.float32 if kind == "float" else dtype).masked_fill_(~keep, float("-inf"))
        if batches > 1:
            m[batches - 1, ..., 5:9] = 0.5  # a bias: no span
    kw = dict(is_causal=causal, enable_gqa=True, q_offset=S - L if causal else 0)
    o, lse = F.scaled_dot_product_attention_with_lse(q, k, v, attn_mask=m, **kw)
    dense = (m if kind != "bool" else torch.zeros(m.shape, device="cuda").masked_fill_(~m, float("-inf"))).float()
    ro, rl = F.scaled_dot_product_attention_with_lse(q, k, v, attn_mask=dense.expand(batches, heads, L, S).contiguous(), **kw)
    torch.cuda.synchronize()
    assert torch.equal(torch.isneginf(lse), torch.isneginf(rl))
    fin = ~torch.isneginf(rl)
    assert ((lse - rl)[fin].abs() / rl[fin].abs().clamp(min=1)).max() <= 1e-5
    assert ((o.float() - ro.float()).abs() - 2.0 ** -7 * ro.float().abs()).max() <= 8e-3
    if heads > 1 or D < 128:
        assert torch.equal(o, ro) and torch.equal(lse, rl)
