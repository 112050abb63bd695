"""Head dim 64, non-causal, no mask: the row max moves only when a lane's sum of P passes its limit.

The keys are laid out so that the scores of one row group rise from tile to tile by a set step (in log2 units): steps
that never reach the limit, ones where a single P does, ones where only the sum of many does, and jumps past what
fp16 could hold; then the same falling.  Against the oracle, at the tolerances of the prefill tests.
"""
import numpy as np
import pytest
import torch

from oracle import sdpa as orc
from tests.attn_cases import LSE_TOL, O_TOL_BF16, host, lse_rel, max_abs, randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("step", [0.0, 0.3, 4.0, 6.0, 7.9, 9.0, 20.0, 200.0, -9.0])
@pytest.mark.parametrize("Sq,Sk", [(70, 64 * 5 + 1), (300, 64 * 9)])
def test_rising_scores(Sq, Sk, step, dtype):
    import dtorch_amd.nn.functional as F
    rng = np.random.default_rng(int(10 * step) + Sk)
    q, k, v = randn(rng, (1, 2, Sq, 64)), 0.3 * randn(rng, (1, 2, Sk, 64)), randn(rng, (1, 2, Sk, 64))
    # score = q.k / 8; the first coordinate of q alternates between rising, falling and neither by rows
    q[..., 0] = np.resize([1.0, -1.0, 0.0], Sq)
    k[..., 0] = (np.arange(Sk) // 64) * step * np.log(2.0) * 8.0
    tq, tk, tv = (torch.from_numpy(x).to(dtype).cuda() for x in (q, k, v))
    ro, rl = orc.sdpa_fwd(*(host(t).astype(np.float64) for t in (tq, tk, tv)))
    o, lse = F.scaled_dot_product_attention_with_lse(tq, tk, tv)
    torch.cuda.synchronize()
    assert max_abs(host(o), ro) <= O_TOL_BF16 and lse_rel(host(lse), rl) <= LSE_TOL


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("r,Sk", [(0.9, 300), (1.5, 256), (1.5, 257), (2.5, 320), (3.2, 600), (3.8, 600), (3.8, 200), (4.5, 129)])
def test_forms_by_grid(r, Sk, dtype):
    """Grids of r workgroups per CU, on each side of the lines between the form that checks the sums and the one that
    takes the row max first: the scores of the test above (steps of 4), some heads against the oracle."""
    import dtorch_amd.nn.functional as F
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    rng = np.random.default_rng(Sk + int(10 * r))
    Sq, H = 130, int(r * cus) // 2  # two workgroups a head
    q, k, v = randn(rng, (1, H, Sq, 64)), 0.3 * randn(rng, (1, 1, Sk, 64)), randn(rng, (1, 1, Sk, 64))
    q[..., 0] = np.resize([1.0, -1.0, 0.0], Sq)
    k[..., 0] = (np.arange(Sk) // 64) * 4.0 * np.log(2.0) * 8.0
    tq, tk, tv = (torch.from_numpy(x).to(dtype).cuda() for x in (q, k, v))
    o, lse = F.scaled_dot_product_attention_with_lse(tq, tk, tv, enable_gqa=True)
    torch.cuda.synchronize()
    for h in (0, H // 2, H - 1):
        ro, rl = orc.sdpa_fwd(*(host(t).astype(np.float64) for t in (tq[:, h:h + 1], tk, tv)))
        assert max_abs(host(o[:, h:h + 1]), ro) <= O_TOL_BF16 and lse_rel(host(lse[:, h:h + 1]), rl) <= LSE_TOL
