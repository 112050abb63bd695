"""The prefill forms of small grids (two key groups per workgroup, or one) against the oracle and against the same
rows inside a batch that fills the chip.

A grid of at most one 128-row workgroup per CU takes two key groups from 8 key tiles of 64 on, and one group below;
the sizes sit around the ends of tiles, of a round of two tiles and of that rule.  Both forms sum in fp32 and round
P and O to the input type; the groups' merge reorders sums only, so they differ by O's rounding (2^-8 of |O| < 4 in
bf16, 2^-11 in fp16) and, where a running max differs, by P's.
"""
import numpy as np
import pytest
import torch

from oracle import sdpa as orc
from tests.attn_cases import LSE_TOL, O_TOL_BF16, host, lse_rel, max_abs, randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Sq,Sk,D,causal,q_off,k_off,scale,peak", [
    (1, 449, 128, False, 0, 0, None, 1.0),       # 8 tiles, the last of one key
    (130, 448, 128, False, 0, 0, None, 1.0),     # 7 tiles: one group
    (200, 577, 128, False, 0, 0, None, 1.0),     # 10 tiles: as many for both groups
    (777, 777, 128, True, 0, 0, None, 1.0),
    (129, 640, 128, True, 511, 0, None, 1.0),    # diagonal in the last tiles
    (600, 600, 128, True, 0, 70, None, 1.0),     # rows 0..69 see nothing, and the second group nothing for more
    (450, 1000, 128, True, 0, 0, -0.1, 1.0),     # negative scale
    (450, 1000, 128, True, 0, 0, None, 30.0),    # peaked scores: rescales, and groups far apart
    (512, 512, 64, False, 0, 0, None, 1.0),
    (513, 705, 64, True, 0, 0, None, 1.0),
    (300, 1100, 64, False, 0, 0, None, 30.0),
    (600, 600, 64, True, 0, 70, None, 1.0),
])
def test_small_grids(Sq, Sk, D, causal, q_off, k_off, scale, peak, dtype):
    import dtorch_amd.nn.functional as F
    rng = np.random.default_rng(Sq * 1000 + Sk)
    H = 2
    q, k, v = peak * randn(rng, (1, H, Sq, D)), randn(rng, (1, 1, Sk, D)), randn(rng, (1, 1, Sk, D))
    tq, tk, tv = (torch.from_numpy(x).to(dtype).cuda() for x in (q, k, v))
    ro, rl = orc.sdpa_fwd(*(host(t).astype(np.float64) for t in (tq, tk, tv)), is_causal=causal, scale=scale,
                          enable_gqa=True, q_offset=q_off, k_offset=k_off)
    kw = dict(is_causal=causal, scale=scale, enable_gqa=True, q_offset=q_off, k_offset=k_off)
    o, lse = F.scaled_dot_product_attention_with_lse(tq, tk, tv, **kw)
    n = 600 // (H * ((Sq + 127) // 128)) + 1  # more than two 128-row workgroups per CU
    ob, lb = F.scaled_dot_product_attention_with_lse(tq.expand(n, -1, -1, -1), tk.expand(n, -1, -1, -1),
                                                     tv.expand(n, -1, -1, -1), **kw)
    torch.cuda.synchronize()
    assert max_abs(host(o), ro) <= O_TOL_BF16 and lse_rel(host(lse), rl) <= LSE_TOL
    assert max_abs(host(o[0]), host(ob[n - 1])) <= O_TOL_BF16 and lse_rel(host(lse[0]), host(lb[n - 1])) <= 1e-5


@pytest.mark.parametrize("D,Sq,before,r", [
    (128, 300, 900, 1.5), (128, 300, 800, 1.5),      # either side of the rule: 15 and 16 tiles in the first block
    (128, 1536, 1000, 1.2), (128, 1536, 3000, 1.2),  # two key groups, and the 64-row kernel
    (64, 300, 1000, 1.5),
])
def test_prompts_that_continue_a_context(D, Sq, before, r):
    """Causal with the diagonal behind `before` keys, on grids of r 128-row workgroups per CU: some heads against the oracle."""
    import dtorch_amd.nn.functional as F
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    rng = np.random.default_rng(Sq + before)
    H, Sk = int(r * cus) // ((Sq + 127) // 128) // 4 * 4, Sq + before
    q, k, v = randn(rng, (1, H, Sq, D)), randn(rng, (1, H // 4, Sk, D)), randn(rng, (1, H // 4, Sk, D))
    tq, tk, tv = (torch.from_numpy(x).to(torch.bfloat16).cuda() for x in (q, k, v))
    o, lse = F.scaled_dot_product_attention_with_lse(tq, tk, tv, is_causal=True, enable_gqa=True, q_offset=before)
    torch.cuda.synchronize()
    for h in (0, H - 1):
        ro, rl = orc.sdpa_fwd(*(host(t).astype(np.float64) for t in (tq[:, h:h + 1], tk[:, h // 4:h // 4 + 1], tv[:, h // 4:h // 4 + 1])),
                              is_causal=True, q_offset=before)
        assert max_abs(host(o[:, h:h + 1]), ro) <= O_TOL_BF16 and lse_rel(host(lse[:, h:h + 1]), rl) <= LSE_TOL
