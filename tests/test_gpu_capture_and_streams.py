"""The calls that keep something in a workspace between two launches, or pick a form by the grid, under graph capture
and on concurrent streams: streaming decode (records, merge), key spans of padding masks (spans, fp32 rows, two attention
kernels), row masks converted first, two key groups, the key-split fp32 form.  Every replay and every stream must equal
the eager serial call bit for bit; inputs, lengths and masks change between replays.
"""
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = ["decode_stream", "decode_stream_paged", "decode_splits", "spans_causal", "spans_rows", "row_converted",
         "key_groups", "fp32_key_split"]


def _case(name, seed):
    """(tensors of one call, the call on such tensors)."""
    import dtorch_amd.nn.functional as F
    g = torch.Generator(device="cuda").manual_seed(seed)
    r = lambda *s, dtype=torch.bfloat16: torch.randn(*s, device="cuda", generator=g).to(dtype)
    if name.startswith("decode"):
        B, Hq, Hkv, cap, page = (70, 8, 2, 1024, 16) if name != "decode_splits" else (2, 8, 2, 1000, 0)
        lens = torch.randint(0, cap + 1, (B,), device="cuda", generator=g, dtype=torch.int32)
        q = r(B, Hq, 1, 128)
        if name == "decode_stream_paged":
            per = cap // page
            table = torch.randperm(B * per, device="cuda", generator=g).view(B, per).to(torch.int32)
            pool = [r(B * per, Hkv, page, 128) for _ in range(2)]
            return [q, *pool, table, lens], lambda q, k, v, t, n: F.decode_attention_paged(q, k, v, t, n)
        return [q, r(B, Hkv, cap, 128), r(B, Hkv, cap, 128), lens], lambda q, k, v, n: F.decode_attention(q, k, v, n)
    kw = dict(enable_gqa=True, is_causal=name in ("spans_causal", "key_groups", "fp32_key_split"))
    if name in ("key_groups", "fp32_key_split"):
        t = torch.float32 if name == "fp32_key_split" else torch.bfloat16
        x = [r(1, h, 600, 64 if t == torch.float32 else 128, dtype=t) for h in (4, 2, 2)]
        return x, lambda q, k, v: F.scaled_dot_product_attention_with_lse(q, k, v, **kw)
    B, L, S, D = 8, 1024, 1501, 64 if name == "row_converted" else 128
    x = [r(B, h, n, D) for h, n in ((8, L), (2, S), (2, S))]
    first = torch.randint(0, S, (B,), device="cuda", generator=g)
    hole = torch.randint(0, S, (B,), device="cuda", generator=g)
    at = torch.arange(S, device="cuda")[None]
    keep = (at >= first[:, None]) & ((at != hole[:, None]) | (torch.arange(B, device="cuda")[:, None] % 2 == 0))
    m = keep[:, None, None]
    if name != "spans_causal":
        m = torch.zeros(B, 1, 1, S, device="cuda", dtype=torch.bfloat16).masked_fill_(~m, float("-inf"))
    return x + [m], lambda q, k, v, m: F.scaled_dot_product_attention_with_lse(q, k, v, attn_mask=m, **kw)


@pytest.mark.parametrize("name", CASES)
def test_graph_replays_match_eager(name):
    inputs = [_case(name, 10 + i)[0] for i in range(3)]
    static, call = _case(name, 9)
    ref = [tuple(t.clone() for t in call(*x)) for x in inputs]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call(*static)
    torch.cuda.synchronize()
    for n in (0, 1, 2, 0):
        for dst, src in zip(static, inputs[n]):
            dst.copy_(src)
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(out, ref[n])), (name, n)
        torch.ones(1000, device="cuda").sum().item()  # eager work between the replays
        assert all(torch.equal(a, b) for a, b in zip(call(*inputs[1]), ref[1]))


def test_concurrent_streams_match_serial():
    work = [_case(name, 20 + i) for i, name in enumerate(CASES)]
    serial = [tuple(t.clone() for t in call(*x)) for x, call in work]
    torch.cuda.synchronize()
    results, errors = [None] * 4, []
    start = threading.Barrier(4)

    def worker(i):
        try:
            s = torch.cuda.Stream()  # default priority
            with torch.cuda.stream(s):
                start.wait()
                for _ in range(6):
                    got = [call(*x) for x, call in work[i:] + work[:i]]
                s.synchronize()
                results[i] = got
        except Exception as e:  # surfaced in the main thread
            errors.append((i, repr(e)))

    threads = [threading.Thread(target=worker, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=60)
    assert not any(t.is_alive() for t in threads) and not errors, errors
    torch.cuda.synchronize()
    for i, got in enumerate(results):
        for o, want in zip(got, serial[i:] + serial[:i]):
            assert all(torch.equal(a, b) for a, b in zip(o, want)), i
