"""KV-cache append in one launch (few tokens per sequence) and in two (more): the caches and the lengths against a
plain indexing loop.  Whole numbers and copied rows: everything is compared exactly."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_new", [1, 3, 16, 17])  # 16: the most 2048 chunks of 16 bytes hold; 17: two launches
@pytest.mark.parametrize("page", [0, 16])
def test_append_one_and_two_launches(n_new, page):
    import dtorch_amd.nn.functional as F
    B, Hkv, D, cap = 6, 8, 128, 64
    g = torch.Generator(device="cuda").manual_seed(n_new)
    kn, vn = (torch.randn(B, n_new, Hkv, D, device="cuda", generator=g).to(torch.bfloat16).transpose(1, 2) for _ in range(2))
    # empty, inside, ending at the capacity, running past it, full, negative (counts as empty)
    start = [0, 17, cap - n_new, cap - 1, cap, -3]
    lengths = torch.tensor(start, dtype=torch.int32, device="cuda")
    pages = B * (cap // page) if page else 0
    table = torch.randperm(pages, device="cuda", generator=g).view(B, -1).to(torch.int32) if page else None
    shape = (pages, Hkv, page, D) if page else (B, Hkv, cap, D)
    k, v = (torch.randn(*shape, device="cuda", generator=g).to(torch.bfloat16) for _ in range(2))
    if page:
        table[1, 1] = -1  # an unassigned slot: tokens 16 .. 31 of sequence 1 are dropped
    wk, wv = k.clone(), v.clone()
    for b in range(B):
        for j in range(n_new):
            t = max(start[b], 0) + j
            if t >= cap:
                continue
            if page:
                p = int(table[b, t // page])
                if p < 0:
                    continue
                wk[p, :, t % page], wv[p, :, t % page] = kn[b, :, j], vn[b, :, j]
            else:
                wk[b, :, t], wv[b, :, t] = kn[b, :, j], vn[b, :, j]
    if page:
        F.kv_cache_append_paged(k, v, table, lengths, kn, vn)
    else:
        F.kv_cache_append(k, v, lengths, kn, vn)
    torch.cuda.synchronize()
    assert torch.equal(k, wk) and torch.equal(v, wv)
    assert lengths.tolist() == [min(max(s, 0) + n_new, cap) for s in start]
