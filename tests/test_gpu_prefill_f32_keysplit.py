"""The key-split form of the fp32 prefill (small grids) against the 128-row form (large grids) and the oracle.

The same rows run once as a small grid and once repeated over a batch large enough for the 128-row form.  Both
sum in fp32, in different orders: |O| is an average of unit normals, and reordering the <= 700 terms of its sums
moves it by at most a few hundred roundings of 2^-24 relative to sums of O(1), i.e. below 1e-5 (the bar of
the fp32 tests).
"""
import numpy as np
import pytest
import torch

from oracle import sdpa as orc
from tests.attn_cases import host, lse_rel, max_abs, randn

pytestmark = pytest.mark.gpu

TOL = 1e-5


@pytest.mark.parametrize("Sq,Sk,D,Dv,causal,q_off,k_off,masked", [
    (1, 1, 64, 64, False, 0, 0, False),        # one key: three waves without a tile
    (33, 97, 64, 64, False, 0, 0, False),      # one key past a tile and past a round of four tiles
    (31, 128, 128, 128, False, 0, 0, False),
    (300, 300, 64, 64, True, 0, 0, False),
    (129, 255, 128, 128, True, 40, 0, False),  # diagonal inside the keys
    (200, 70, 64, 64, True, 0, 30, False),     # rows 0..29 see nothing
    (65, 160, 48, 36, True, 0, 0, False),      # padded head dims
    (77, 77, 100, 128, False, 0, 0, True),
    (130, 700, 64, 64, True, 570, 0, True),
    (64, 513, 128, 128, True, 449, 0, True),
])
def test_key_split_against_128_row_form(Sq, Sk, D, Dv, causal, q_off, k_off, masked):
    import dtorch_amd.nn.functional as F
    rng = np.random.default_rng(Sq * 1000 + Sk)
    H = 2
    q, k, v = randn(rng, (1, H, Sq, D)), randn(rng, (1, 1, Sk, D)), randn(rng, (1, 1, Sk, Dv))
    m = None
    if masked:
        m = np.where(rng.random((1, 1, Sq, Sk)) < 0.3, -np.inf, rng.standard_normal((1, 1, Sq, Sk)))
        m[..., 0, :] = -np.inf  # a row without a key
        m = m.astype(np.float32)
    ro, rl = orc.sdpa_fwd(q.astype(np.float64), k.astype(np.float64), v.astype(np.float64),
                          attn_mask=None if m is None else m.astype(np.float64), is_causal=causal, enable_gqa=True,
                          q_offset=q_off, k_offset=k_off)
    tq, tk, tv = (torch.from_numpy(x).cuda() for x in (q, k, v))
    tm = None if m is None else torch.from_numpy(m).cuda()
    kw = dict(is_causal=causal, enable_gqa=True, q_offset=q_off, k_offset=k_off)
    n = 4096 * 128 // (H * 128) + 1  # more than 8 blocks of 128 rows per CU whatever Sq is
    o, lse = F.scaled_dot_product_attention_with_lse(tq, tk, tv, attn_mask=tm, **kw)
    ob, lb = F.scaled_dot_product_attention_with_lse(tq.expand(n, -1, -1, -1), tk.expand(n, -1, -1, -1),
                                                     tv.expand(n, -1, -1, -1),
                                                     attn_mask=tm, **kw)
    torch.cuda.synchronize()
    assert max_abs(host(o), ro) <= TOL and lse_rel(host(lse), rl) <= TOL
    assert max_abs(host(o[0]), host(ob[n - 1])) <= TOL and lse_rel(host(lse[0]), host(lb[n - 1])) <= TOL


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("r", [0.4, 0.9, 1.5, 2.5, 9])
def test_forms_by_grid(r, D, causal):
    """Grids of r 128-row items per CU, through every branch of the rule that picks a form: some heads against the oracle."""
    import dtorch_amd.nn.functional as F
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    rng = np.random.default_rng(int(10 * r) + D)
    S, H = 200, int(r * cus) // 2  # two items a head
    q, k, v = randn(rng, (1, H, S, D)), randn(rng, (1, 1, S + 40, D)), randn(rng, (1, 1, S + 40, D))
    kw = dict(is_causal=causal, enable_gqa=True, q_offset=40)
    o, lse = F.scaled_dot_product_attention_with_lse(*(torch.from_numpy(x).cuda() for x in (q, k, v)), **kw)
    torch.cuda.synchronize()
    for h in (0, H // 2, H - 1):
        ro, rl = orc.sdpa_fwd(*(x.astype(np.float64) for x in (q[:, h:h + 1], k, v)), is_causal=causal, q_offset=40)
        assert max_abs(host(o[:, h:h + 1]), ro) <= TOL and lse_rel(host(lse[:, h:h + 1]), rl) <= TOL
