"""The streaming decode (decode_stream.hip: larger bf16 / fp16 batches at head dim 128) against the split form and the
oracle.

An explicit chunk selects the split form, so both run on the same inputs.  Both keep scores, sums and partial outputs
in fp32 and round P and O to the input type, over different splits: their O differ by those roundings (2^-9 of P and
of |O| < 3 in bf16), the LSE by fp32 ones.  Lengths sit at the ends of a 32-token unit, of the 64 sequences a wave's
prefix covers at once, and at zero; rows of the caches past a length hold NaN.
"""
import numpy as np
import pytest
import torch

from oracle import sdpa as orc
from tests.attn_cases import LSE_TOL, O_TOL_BF16, host, lse_rel, max_abs

pytestmark = pytest.mark.gpu


def _lengths(kind, B, cap, rng):
    edge = [0, 1, 31, 32, 33, 63, 64, 65, cap - 1, cap]
    if kind == "mixed":
        n = np.concatenate([edge, rng.integers(0, cap + 1, B - len(edge))])
        return rng.permutation(n)
    if kind == "short":  # a share spans many sequences
        return rng.integers(0, 40, B)
    if kind == "one":  # every wave cuts the same sequence; the others are empty
        return np.where(np.arange(B) == B - 1, cap, 0)
    return np.ones(B, dtype=int)


@pytest.mark.parametrize("B,Hq,Hkv,cap,page,kind,dtype,scale", [
    (70, 8, 2, 1024, 0, "mixed", torch.bfloat16, None),
    (70, 8, 2, 1024, 16, "mixed", torch.float16, None),
    (70, 14, 2, 1024, 32, "mixed", torch.bfloat16, None),    # groups of 7
    (130, 16, 2, 512, 64, "short", torch.bfloat16, -0.1),    # groups of 8, a negative scale
    (33, 32, 32, 1024, 256, "mixed", torch.bfloat16, None),  # groups of 1
    (70, 8, 2, 1024, 16, "one", torch.bfloat16, None),
    (70, 8, 2, 1024, 0, "ones", torch.bfloat16, None),
    (2, 10, 2, 16384, 0, "one", torch.float16, None),        # groups of 5; merged by four waves a head
])
def test_stream_against_split_and_oracle(B, Hq, Hkv, cap, page, kind, dtype, scale):
    import dtorch_amd.nn.functional as F
    D = 128
    rng = np.random.default_rng(B + cap + page)
    lens = _lengths(kind, B, cap, rng)
    g = torch.Generator(device="cuda").manual_seed(B)
    q = torch.randn(B, Hkv, Hq // Hkv, D, device="cuda", generator=g).to(dtype).flatten(1, 2)[:, :, None]
    # [B, S, H, D] storage: rows of a head are not contiguous
    k, v = (torch.randn(B, cap, Hkv, D, device="cuda", generator=g).to(dtype).transpose(1, 2) for _ in range(2))
    past = torch.arange(cap, device="cuda")[None, :] >= torch.tensor(lens, device="cuda")[:, None]
    for t in (k, v):
        t.masked_fill_(past[:, None, :, None], float("nan"))
    tl = torch.tensor(lens, dtype=torch.int32, device="cuda")
    if page:
        per = cap // page
        table = torch.randperm(B * per, device="cuda", generator=g).view(B, per)
        pages = []
        for t in (k, v):
            pool = torch.empty(B * per, Hkv, page, D, dtype=dtype, device="cuda")
            pool[table.flatten()] = t.unflatten(2, (per, page)).transpose(1, 2).flatten(0, 1)
            pages.append(pool)
        run = lambda chunk: F.decode_attention_paged(q, *pages, table.to(torch.int32), tl, scale=scale, chunk=chunk)
    else:
        run = lambda chunk: F.decode_attention(q, k, v, tl, scale=scale, chunk=chunk)
    o, lse = run(0)
    o2, lse2 = run(0)
    os_, ls = run(384)
    torch.cuda.synchronize()
    assert torch.equal(o, o2) and torch.equal(lse, lse2)
    assert max_abs(host(o), host(os_)) <= O_TOL_BF16 and lse_rel(host(lse), host(ls)) <= 1e-5
    for b in np.unique(np.concatenate([[0, B - 1], rng.integers(0, B, 6), np.flatnonzero(lens == lens.max())[:1]])):
        n = int(lens[b])
        if n == 0:
            assert not o[b].any() and torch.isneginf(lse[b]).all()
            continue
        ro, rl = orc.sdpa_fwd(host(q[b:b + 1]), host(k[b:b + 1, :, :n]), host(v[b:b + 1, :, :n]), scale=scale, enable_gqa=True)
        assert max_abs(host(o[b:b + 1]), ro) <= O_TOL_BF16 and lse_rel(host(lse[b:b + 1]), rl[:, :, 0]) <= LSE_TOL


@pytest.mark.parametrize("B,S", [(1, 4000), (70, 1024)])  # below and above the streaming form's line
def test_smaller_workspace_is_still_accepted(B, S):
    """chunk 0 with the workspace of 384-token splits, as 0 picked for these calls before it also picked 128."""
    import ctypes
    from tests.test_zz_no_alloc import BF16, _args, _case
    from tests.test_zz_no_alloc import _lib as bound
    lib = bound()
    q, k, v, lengths = _case(B, 8, 2, S, 128, torch.bfloat16, B)
    lengths.fill_(S - 3)
    outs = []
    for chunk in (0, 384):
        o, lse = torch.empty_like(q), torch.empty(B, 8, device="cuda")
        ws = torch.empty(lib.dtattn_decode_workspace_size(B, 8, S, 128, 384), dtype=torch.uint8, device="cuda")
        a = _args(q, k, v, lengths, o, lse, BF16, chunk, ws)
        stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        assert lib.dtattn_decode_splitkv(ctypes.byref(a), stream) == 0, lib.dtattn_last_error()
        outs.append((host(o), host(lse)))
    torch.cuda.synchronize()
    assert max_abs(outs[0][0], outs[1][0]) <= O_TOL_BF16 and lse_rel(outs[0][1], outs[1][1]) <= 1e-5


@pytest.mark.parametrize("chunk", [0, 128, 384])  # streaming form, then splits
@pytest.mark.parametrize("page", [0, 16])
def test_parts_whose_scores_are_all_minus_infinity(page, chunk):
    """Keys of -inf in a coordinate where every query is positive have a score of -inf, hence no weight, also where a
    whole share or split holds nothing else; a part without weight adds nothing to the merge."""
    import dtorch_amd.nn.functional as F
    B, Hq, Hkv, cap, D, dtype = 70, 8, 2, 1024, 128, torch.bfloat16
    g = torch.Generator(device="cuda").manual_seed(page + chunk)
    q = torch.randn(B, Hq, 1, D, device="cuda", generator=g).to(dtype)
    q[..., 0] = 1.5
    k, v = (torch.randn(B, Hkv, cap, D, device="cuda", generator=g).to(dtype) for _ in range(2))
    k[::2, :, 128:900, 0] = float("-inf")
    lens = torch.full((B,), cap, dtype=torch.int32, device="cuda")
    lens[::4] = 700  # ends among them
    if page:
        per = cap // page
        table = torch.arange(B * per, device="cuda", dtype=torch.int32).view(B, per)
        kp, vp = (t.unflatten(2, (per, page)).transpose(1, 2).flatten(0, 1).contiguous() for t in (k, v))
        o, lse = F.decode_attention_paged(q, kp, vp, table, lens, chunk=chunk)
    else:
        o, lse = F.decode_attention(q, k, v, lens, chunk=chunk)
    torch.cuda.synchronize()
    for b in (0, 1, 2, 3, B - 2, B - 1):
        at = [t for t in range(int(lens[b])) if b % 2 or not 128 <= t < 900]
        ro, rl = orc.sdpa_fwd(host(q[b:b + 1]), host(k[b:b + 1, :, at]), host(v[b:b + 1, :, at]), enable_gqa=True)
        assert max_abs(host(o[b:b + 1]), ro) <= O_TOL_BF16 and lse_rel(host(lse[b:b + 1]), rl[:, :, 0]) <= LSE_TOL


@pytest.mark.parametrize("which", ["q", "o"])
def test_pointers_off_their_alignment_keep_the_split_form(which):
    """The C ABI checks strides, not pointers: a query or output 4 elements into a buffer of a call large enough for the
    streaming form takes the splits that chunk 0 picks beside it, bit for bit."""
    import ctypes
    from tests.test_zz_no_alloc import BF16, _args, _case
    from tests.test_zz_no_alloc import _lib as bound
    lib = bound()
    B, S = 70, 1024
    q, k, v, lengths = _case(B, 8, 2, S, 128, torch.bfloat16, B)
    lengths.fill_(S - 3)

    def moved(t, by):
        return torch.empty(t.numel() + 8, dtype=t.dtype, device="cuda")[by:by + t.numel()].view(t.shape)

    q = moved(q, 4 if which == "q" else 0).copy_(q)
    outs = []
    for chunk in (0, 384):
        o, lse = moved(q, 2 if which == "o" else 0), torch.empty(B, 8, device="cuda")
        ws = torch.empty(lib.dtattn_decode_workspace_size(B, 8, S, 128, 0), dtype=torch.uint8, device="cuda")
        a = _args(q, k, v, lengths, o, lse, BF16, chunk, ws)
        stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        assert lib.dtattn_decode_splitkv(ctypes.byref(a), stream) == 0, lib.dtattn_last_error()
        outs.append((o, lse))
    torch.cuda.synchronize()
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])


# units of 32 tokens per CU from which a group of query heads takes the streaming form (1: paged caches only)
LINE = {1: 124, 2: 124, 3: 15, 4: 15, 5: 12, 6: 12, 7: 6, 8: 7}


@pytest.mark.parametrize("group", sorted(LINE))
@pytest.mark.parametrize("page", [0, 16])
@pytest.mark.parametrize("B", [2, 67])  # merged by four waves a head, and by one
def test_every_group_on_both_sides_of_its_line(group, page, B):
    """The streaming form from its line on, and the splits that chunk 0 picks just below it, against splits of 256 and
    the oracle.  Forms differ in the last bits of some LSE, so a chunk 0 that matches neither split length ran the
    streaming kernel."""
    import dtorch_amd.nn.functional as F
    D, dtype = 128, torch.bfloat16
    Hkv = 8 if group <= 2 else 4
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    units = LINE[group] * cus // (B * Hkv) + 1  # a sequence
    g = torch.Generator(device="cuda").manual_seed(group + page)
    q = torch.randn(B, Hkv * group, 1, D, device="cuda", generator=g).to(dtype)
    for u in (units, units - 2):
        cap = 32 * u
        streams = B * Hkv * u >= LINE[group] * cus and (group > 1 or page > 0)
        assert streams == (u == units and (group > 1 or page > 0))
        k, v = (torch.randn(B, Hkv, cap, D, device="cuda", generator=g).to(dtype) for _ in range(2))
        lens = torch.randint(0, cap + 1, (B,), device="cuda", generator=g, dtype=torch.int32)
        lens[0], lens[B - 1] = cap - 1, cap
        if page:
            per = cap // page
            table = torch.randperm(B * per, device="cuda", generator=g).view(B, per)
            pages = []
            for t in (k, v):
                pool = torch.empty(B * per, Hkv, page, D, dtype=dtype, device="cuda")
                pool[table.flatten()] = t.unflatten(2, (per, page)).transpose(1, 2).flatten(0, 1)
                pages.append(pool)
            run = lambda chunk: F.decode_attention_paged(q, *pages, table.to(torch.int32), lens, chunk=chunk)
        else:
            run = lambda chunk: F.decode_attention(q, k, v, lens, chunk=chunk)
        o, lse = run(0)
        os_, ls = run(256)
        same = [torch.equal(lse, run(c)[1]) for c in (128, 384)]
        torch.cuda.synchronize()
        assert any(same) != streams
        assert max_abs(host(o), host(os_)) <= O_TOL_BF16
        fin = ~torch.isneginf(ls)
        assert torch.equal(fin, ~torch.isneginf(lse)) and lse_rel(host(lse[fin]), host(ls[fin])) <= 1e-5
        for b in (0, B - 1):
            n = int(lens[b])
            ro, rl = orc.sdpa_fwd(host(q[b:b + 1]), host(k[b:b + 1, :, :n]), host(v[b:b + 1, :, :n]), enable_gqa=True)
            assert max_abs(host(o[b:b + 1]), ro) <= O_TOL_BF16 and lse_rel(host(lse[b:b + 1]), rl[:, :, 0]) <= LSE_TOL


@pytest.mark.parametrize("group", [3, 4, 5, 6, 8])
@pytest.mark.parametrize("B,cap", [(1, 128), (1, 129), (1, 384), (1, 385), (20, 384), (1, 1536), (1, 1537), (2, 2560), (2, 2561), (1, 3073),
                                   (1, 8193), (9, 600)])
def test_split_lengths_of_smaller_calls(group, B, cap):
    """The bounds between splits of 128 and of 384 tokens (one split, a merge or none) against splits of 256."""
    import dtorch_amd.nn.functional as F
    Hkv, D, dtype = 8, 128, torch.float16
    g = torch.Generator(device="cuda").manual_seed(group + cap)
    q = torch.randn(B, Hkv * group, 1, D, device="cuda", generator=g).to(dtype)
    k, v = (torch.randn(B, Hkv, cap, D, device="cuda", generator=g).to(dtype) for _ in range(2))
    for n in (cap, cap - 1, 1, 0):
        lens = torch.full((B,), n, dtype=torch.int32, device="cuda")
        o, lse = F.decode_attention(q, k, v, lens)
        ro, rl = F.decode_attention(q, k, v, lens, chunk=256)
        torch.cuda.synchronize()
        if n == 0:
            assert not o.any() and torch.isneginf(lse).all()
            continue
        assert max_abs(host(o), host(ro)) <= O_TOL_BF16 and lse_rel(host(lse), host(rl)) <= 1e-5


def test_table_entries_outside_the_pool():
    """Entries of the block table past a sequence's last page hold anything; one inside its length that is not a page of
    the pool reads some page of it, and no other sequence notices."""
    import dtorch_amd.nn.functional as F
    B, Hq, Hkv, page, per, D = 70, 8, 2, 16, 64, 128
    g = torch.Generator(device="cuda").manual_seed(5)
    q = torch.randn(B, Hq, 1, D, device="cuda", generator=g).to(torch.bfloat16)
    kp, vp = (torch.randn(B * per, Hkv, page, D, device="cuda", generator=g).to(torch.bfloat16) for _ in range(2))
    table = torch.randperm(B * per, device="cuda", generator=g).view(B, per).to(torch.int32)
    lens = torch.randint(1, per * page + 1, (B,), device="cuda", generator=g, dtype=torch.int32)
    lens[0] = 100
    o, lse = F.decode_attention_paged(q, kp, vp, table, lens)
    bad = table.clone()
    past = torch.arange(per, device="cuda")[None] * page >= lens[:, None]
    junk = torch.tensor([-1, -2 ** 31, B * per, 2 ** 31 - 1], dtype=torch.int32, device="cuda")
    bad[past] = junk[torch.randint(0, 4, (int(past.sum()),), device="cuda", generator=g)]
    o2, l2 = F.decode_attention_paged(q, kp, vp, bad, lens)
    bad[0, 2] = 2 ** 31 - 1
    o3, l3 = F.decode_attention_paged(q, kp, vp, bad, lens)
    torch.cuda.synchronize()
    assert torch.equal(o2, o) and torch.equal(l2, lse)
    assert torch.equal(o3[1:], o[1:]) and torch.equal(l3[1:], lse[1:]) and o3.isfinite().all()
