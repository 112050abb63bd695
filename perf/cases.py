"""Performance cases of the attention path: the calls that the model ports make of it, through dtorch_amd.nn.functional.

A case is a dict with a "kind" (which call, in which model's role) and its sizes; `listed()` holds one or two
of each kind, `draw()` gives more over the same ranges.  Sizes, heads and layouts are those of the models the
package names: Llama (32 query / 8 kv heads of 128), the Flux and SD3 joint attentions (24 heads of 128 / 64),
the CLIP text encoders (12 or 20 heads of 64, 77 tokens) and the VAE's one head of 512.  Inputs are unit
normals, which is what projections behind a norm layer give.
"""
import math

import torch

from dtorch_amd.nn import functional as F

_DT = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_SIZE = {"bf16": 2, "fp16": 2, "fp32": 4}


def listed():
    return [
        # CLIP text encoder layer of one prompt pair: 77 tokens, the causal-and-padding mask as an additive tensor
        dict(name="text_encoder", kind="text_encoder", B=2, H=12, S=77, D=64, dtype="fp16"),
        # one short chat prompt: causal attention, then its keys and values into 16-token pages
        dict(name="prompt", kind="prompt", B=1, Hq=32, Hkv=8, S=777, D=128, page=16, dtype="bf16"),
        # a batch of equal prompts with the per-row LSE (the headline shape)
        dict(name="prefill", kind="prefill", B=4, Hq=32, Hkv=8, S=2048, D=128, dtype="bf16"),
        # a left-padded batch of prompts of different lengths: causal plus a boolean key mask
        dict(name="padded_prompts", kind="padded_prompts", B=4, Hq=32, Hkv=8, S=2000, D=128, dtype="bf16"),
        # Flux joint attention at 1024 x 1024: 512 text and 4096 image tokens
        dict(name="flux_joint", kind="joint", B=1, H=24, S=4608, D=128, dtype="bf16"),
        # SD3 joint attention at 1024 x 1024 with guidance (two samples): 333 text and 4096 image tokens
        dict(name="sd3_joint", kind="joint", B=2, H=24, S=4429, D=64, dtype="fp16"),
        # the same Flux attention on the native fp8 path, quantization included
        dict(name="flux_fp8", kind="joint_fp8", B=1, H=24, S=4608, D=128, dtype="bf16"),
        # VAE mid-block attention of a 1024 x 1024 image: one head of 512
        dict(name="vae_mid", kind="vae", B=1, S=16384, D=512, dtype="bf16"),
        # a full-precision layer
        dict(name="fp32_layer", kind="fp32_layer", B=2, H=16, S=1000, D=64, causal=True, dtype="fp32"),
        # one device's share of causal ring attention: three full blocks, the diagonal one, and their merge
        dict(name="ring", kind="ring", B=1, Hq=32, Hkv=8, S=4096, D=128, chunks=4, dtype="bf16"),
        # one token of one sequence: append to the cache, then attend over it
        dict(name="decode_step", kind="decode_step", B=1, Hq=32, Hkv=8, S=4000, D=128, dtype="bf16"),
        # one token of a serving batch of mixed lengths (512 to 8192) over a paged cache
        dict(name="decode_paged", kind="decode_paged", B=64, Hq=32, Hkv=8, lo=512, hi=8192, D=128, page=16, dtype="bf16"),
    ]


# Rates (operations a second, bytes a second) by which draw() bounds a case's cost; the most it may cost is
# that of the listed ring step.
_RATE = {"fp32": 0.06e15, "text_encoder": 0.1e15, "padded_prompts": 0.35e15, "joint64": 0.8e15, "vae": 0.7e15}
_MOST_S = 0.8e-3


def _cost(c):
    rate = _RATE.get(c["dtype"]) or _RATE.get(c["kind"] + ("64" if c["D"] == 64 else "")) or _RATE.get(c["kind"]) or 1.0e15
    w = work(c)
    return w["flops"] / rate + w["bytes"] / 4.5e12


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _drawn(rng):
    kind = rng.choice(["text_encoder", "prompt", "prefill", "padded_prompts", "joint", "joint_fp8", "vae", "fp32_layer",
                       "ring", "decode_step", "decode_paged"])
    half = rng.choice(["bf16", "bf16", "fp16"])
    hq, hkv = rng.choice([(32, 8), (32, 8), (32, 32), (64, 8), (28, 4)])
    if kind == "text_encoder":
        s = 77 if rng.random() < 0.5 else rng.randint(16, 512)
        return dict(kind=kind, B=_log(rng, 1, 64), H=rng.choice([12, 20]), S=s, D=64, dtype=rng.choice(["fp16", "bf16", "fp32"]))
    if kind == "prompt":
        return dict(kind=kind, B=_log(rng, 1, 8), Hq=hq, Hkv=hkv, S=_log(rng, 16, 8192), D=128, page=rng.choice([16, 32, 64]), dtype=half)
    if kind == "prefill":
        return dict(kind=kind, B=_log(rng, 1, 16), Hq=hq, Hkv=hkv, S=_log(rng, 128, 8192), D=rng.choice([128, 128, 64]), dtype=half)
    if kind == "padded_prompts":
        return dict(kind=kind, B=_log(rng, 2, 16), Hq=hq, Hkv=hkv, S=_log(rng, 64, 4096), D=128, dtype=half)
    if kind in ("joint", "joint_fp8"):
        d = 128 if kind == "joint_fp8" else rng.choice([64, 128])
        # image tokens of 256 x 256 to 1536 x 1536 pixels behind 77 to 512 text tokens
        return dict(kind=kind, B=rng.choice([1, 1, 2, 4]), H=24, S=(rng.randint(16, 96) * rng.randint(16, 96)) + rng.choice([77, 256, 333, 512]),
                    D=d, dtype=half)
    if kind == "vae":
        return dict(kind=kind, B=rng.choice([1, 1, 2]), S=rng.randint(24, 128) * rng.randint(24, 128), D=512, dtype=half)
    if kind == "fp32_layer":
        return dict(kind=kind, B=rng.choice([1, 2, 4]), H=rng.choice([8, 12, 16]), S=_log(rng, 64, 4096), D=rng.choice([64, 64, 128]),
                    causal=rng.random() < 0.5, dtype="fp32")
    if kind == "ring":
        return dict(kind=kind, B=rng.choice([1, 1, 2]), Hq=hq, Hkv=hkv, S=_log(rng, 256, 4096), D=128, chunks=rng.randint(2, 8), dtype=half)
    if kind == "decode_step":
        return dict(kind=kind, B=_log(rng, 1, 16), Hq=hq, Hkv=hkv, S=_log(rng, 64, 32768), D=rng.choice([128, 128, 64]),
                    dtype=rng.choice(["bf16", "bf16", "fp16", "fp32"]))
    hi = _log(rng, 512, 16384)
    return dict(kind=kind, B=_log(rng, 4, 128), Hq=hq, Hkv=hkv, lo=max(1, hi // rng.choice([2, 8, 16])), hi=hi, D=128,
                page=rng.choice([16, 32, 64, 256]), dtype=half)


def draw(rng):
    while True:
        c = _drawn(rng)
        if _cost(c) <= _MOST_S:
            return c


def _lengths(c):
    """Cached tokens of each sequence of a decode batch, spread evenly over [lo, hi]."""
    n = c["B"]
    return [c["lo"] + (c["hi"] - c["lo"]) * i // max(n - 1, 1) for i in range(n)]


def _padding(c):
    """Left padding of each prompt of a batch: none for the first, up to half of S for the last."""
    return [(c["S"] // 2) * b // max(c["B"] - 1, 1) for b in range(c["B"])]


def _pairs(c):
    """Visible (query, key) pairs of one query head, over the batch."""
    s, b = c.get("S"), c["B"]
    kind = c["kind"]
    tri = lambda n: n * (n + 1) // 2  # noqa: E731
    if kind in ("text_encoder", "prompt", "prefill"):
        return b * tri(s)
    if kind == "padded_prompts":
        return sum(tri(s - p) for p in _padding(c))
    if kind == "ring":
        return b * ((c["chunks"] - 1) * s * s + tri(s))
    if kind == "decode_step":
        return b * s
    if kind == "decode_paged":
        return sum(_lengths(c))
    return b * (tri(s) if c.get("causal") else s * s)


def work(c):
    e, d, kind = _SIZE[c["dtype"]], c["D"], c["kind"]
    heads = 1 if kind == "vae" else c.get("H") or c["Hq"]
    kv = 1 if kind == "vae" else c.get("H") or c["Hkv"]
    flops = 4 * heads * d * _pairs(c)
    if kind in ("decode_step", "decode_paged"):
        tokens = _pairs(c)
        data = 2 * kv * tokens * d * e + 2 * c["B"] * heads * d * e + 4 * c["B"] * heads
        data += 4 * kv * c["B"] * d * e if kind == "decode_step" else 4 * (tokens // c["page"])
        return {"bytes": data, "flops": flops}
    rows = c["B"] * c["S"]
    blocks = c.get("chunks", 1)
    data = 2 * rows * heads * d * e + 2 * blocks * rows * kv * d * e
    if kind in ("prefill", "ring"):
        data += 4 * rows * heads
    if kind == "prompt":  # the pages are written
        data += 2 * rows * kv * d * e
    if kind == "text_encoder":
        data += c["B"] * c["S"] * c["S"] * e
    if kind == "padded_prompts":
        data += rows
    return {"bytes": data, "flops": flops}


def tolerance(c):
    # Outputs are rounded to the input's type and so are the probabilities before the second product; the
    # fp8 path rounds the probabilities to e4m3.
    if c["kind"] == "joint_fp8":
        return {"rel": 4e-2}
    return {"rel": {"bf16": 1e-2, "fp16": 1.5e-3, "fp32": 1e-5}[c["dtype"]]}


def _normal(g, *shape, dtype):
    return torch.randn(*shape, device="cuda", generator=g).to(dtype)


def _tokens(g, b, s, h, d, dtype):
    """[B, H, S, D] view of a projection's [B, S, H, D] output."""
    return _normal(g, b, s, h, d, dtype=dtype).transpose(1, 2)


def prepare(c, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    t, kind, b, s, d = _DT[c["dtype"]], c["kind"], c["B"], c.get("S"), c["D"]
    st = {"case": c}
    if kind in ("text_encoder", "joint", "joint_fp8", "fp32_layer"):
        for n in "qkv":
            st[n] = _tokens(g, b, s, c["H"], d, t)
    elif kind == "vae":
        for n in "qkv":
            st[n] = _normal(g, b, 1, s, d, dtype=t)
    elif kind in ("prompt", "padded_prompts"):
        for n, h in (("q", c["Hq"]), ("k", c["Hkv"]), ("v", c["Hkv"])):
            st[n] = _tokens(g, b, s, h, d, t)
    elif kind == "prefill":
        for n, h in (("q", c["Hq"]), ("k", c["Hkv"]), ("v", c["Hkv"])):
            st[n] = _normal(g, b, h, s, d, dtype=t)
    elif kind == "ring":
        st["q"] = _normal(g, b, c["Hq"], s, d, dtype=t)
        for n in "kv":
            st[n] = [_normal(g, b, c["Hkv"], s, d, dtype=t) for _ in range(c["chunks"])]
    else:
        st["q"] = _normal(g, b, c["Hq"], 1, d, dtype=t)
    if kind == "text_encoder":
        # causal and padding parts, each filled with the type's lowest value, as the encoders build it
        low = torch.finfo(t).min
        keep = torch.tensor([max(3, s - s * i // (2 * b)) for i in range(b)], device="cuda")
        at = torch.arange(s, device="cuda")
        hidden = (at[None, None, :] > at[None, :, None]) | (at[None, None, :] >= keep[:, None, None])
        hidden &= ~torch.eye(s, dtype=torch.bool, device="cuda")
        st["mask"] = torch.zeros(b, 1, s, s, dtype=t, device="cuda").masked_fill_(hidden[:, None], low)
    if kind == "padded_prompts":
        pad = torch.tensor(_padding(c), device="cuda")
        st["mask"] = (torch.arange(s, device="cuda")[None, :] >= pad[:, None])[:, None, None, :]
    if kind == "prompt":
        per = -(-s // c["page"])
        for n in ("kp", "vp"):
            st[n] = torch.zeros(b * per, c["Hkv"], c["page"], d, dtype=t, device="cuda")
        st["table"] = torch.randperm(b * per, device="cuda", generator=g).view(b, per).to(torch.int32)
        st["lengths"] = torch.zeros(b, dtype=torch.int32, device="cuda")
    if kind == "decode_step":
        room = -(-s // 256) * 256
        for n in ("kc", "vc"):
            st[n] = _normal(g, b, c["Hkv"], room, d, dtype=t)
        for n in ("k", "v"):
            st[n] = _tokens(g, b, 1, c["Hkv"], d, t)
        st["before"] = torch.full((b,), s - 1, dtype=torch.int32, device="cuda")
        st["lengths"] = st["before"].clone()
    if kind == "decode_paged":
        per = -(-c["hi"] // c["page"])
        for n in ("kp", "vp"):
            st[n] = _normal(g, b * per, c["Hkv"], c["page"], d, dtype=t)
        st["table"] = torch.randperm(b * per, device="cuda", generator=g).view(b, per).to(torch.int32)
        order = torch.randperm(b, device="cuda", generator=g)
        st["lengths"] = torch.tensor(_lengths(c), dtype=torch.int32, device="cuda")[order]
    return st


def run(st):
    c = st["case"]
    kind = c["kind"]
    if kind == "text_encoder":
        return F.scaled_dot_product_attention(st["q"], st["k"], st["v"], attn_mask=st["mask"])
    if kind in ("joint", "vae"):
        return F.scaled_dot_product_attention(st["q"], st["k"], st["v"])
    if kind == "fp32_layer":
        return F.scaled_dot_product_attention(st["q"], st["k"], st["v"], is_causal=c["causal"])
    if kind == "joint_fp8":
        return F.scaled_dot_product_attention(st["q"], st["k"], st["v"], sdpa_option=F.SdpaOption(sage_attn_type="native_fp8"))
    if kind == "padded_prompts":
        return F.scaled_dot_product_attention(st["q"], st["k"], st["v"], attn_mask=st["mask"], is_causal=True, enable_gqa=True)
    if kind == "prefill":
        return F.scaled_dot_product_attention_with_lse(st["q"], st["k"], st["v"], is_causal=True, enable_gqa=True)
    if kind == "ring":
        return F.ring_attention_step(st["q"], st["k"], st["v"], c["chunks"] - 1)
    if kind == "prompt":
        o = F.scaled_dot_product_attention(st["q"], st["k"], st["v"], is_causal=True, enable_gqa=True)
        st["lengths"].zero_()  # a new request takes the slot
        F.kv_cache_append_paged(st["kp"], st["vp"], st["table"], st["lengths"], st["k"], st["v"])
        return o, st["kp"], st["vp"], st["lengths"]
    if kind == "decode_step":
        st["lengths"].copy_(st["before"])  # the scheduler's lengths of this step
        F.kv_cache_append(st["kc"], st["vc"], st["lengths"], st["k"], st["v"])
        n = c["S"]
        o, lse = F.decode_attention(st["q"], st["kc"][:, :, :n], st["vc"][:, :, :n], st["lengths"])
        return o, lse, st["kc"], st["vc"], st["lengths"]
    return F.decode_attention_paged(st["q"], st["kp"], st["vp"], st["table"], st["lengths"])


def _attend64(q, k, v, offset=None, bias=None):
    """(O, LSE) of one head in 64 bits: q [L, D], k and v [S, D]; with `offset`, key j is visible to query i iff
    j <= i + offset; `bias` [L or 1, S] is added.  Rows without a visible key give 0."""
    q, k, v = q.double(), k.double(), v.double()
    kt, os, ls = k.t().contiguous(), [], []
    at = torch.arange(k.shape[0], device=q.device)
    for r in range(0, q.shape[0], 4096):
        x = (q[r:r + 4096] @ kt) / math.sqrt(q.shape[1])
        if bias is not None:
            x += bias[r:r + 4096] if bias.shape[0] > 1 else bias
        if offset is not None:
            x.masked_fill_(at[None, :] > torch.arange(r, r + x.shape[0], device=q.device)[:, None] + offset, -math.inf)
        lse = torch.logsumexp(x, -1)
        os.append(torch.exp(x - torch.where(lse == -math.inf, 0.0, lse)[:, None]) @ v)
        ls.append(lse)
    return torch.cat(os), torch.cat(ls)


def _heads64(st, q, k, v, offset=None, bias=None):
    B, H, L, _ = q.shape
    group = H // k.shape[1]
    o = torch.empty(*q.shape, dtype=torch.float64, device=q.device)
    lse = torch.empty(B, H, L, dtype=torch.float64, device=q.device)
    for b in range(B):
        m = None if bias is None else bias[b]
        for h in range(H):
            o[b, h], lse[b, h] = _attend64(q[b, h], k[b, h // group], v[b, h // group], offset, m)
    return o, lse


def exact(c, seed):
    st = prepare(c, seed)
    kind = c["kind"]
    if kind == "text_encoder":
        return _heads64(st, st["q"], st["k"], st["v"], bias=st["mask"][:, 0].double())[0]
    if kind in ("joint", "joint_fp8", "vae", "fp32_layer"):
        return _heads64(st, st["q"], st["k"], st["v"], offset=0 if c.get("causal") else None)[0]
    if kind == "padded_prompts":
        bias = torch.zeros(c["B"], 1, c["S"], dtype=torch.float64, device="cuda").masked_fill_(~st["mask"][:, 0], -math.inf)
        return _heads64(st, st["q"], st["k"], st["v"], offset=0, bias=bias)[0]
    if kind == "prefill":
        return _heads64(st, st["q"], st["k"], st["v"], offset=0)
    if kind == "ring":
        n = c["chunks"]
        return _heads64(st, st["q"], torch.cat(st["k"], 2), torch.cat(st["v"], 2), offset=(n - 1) * c["S"])
    if kind == "prompt":
        o = _heads64(st, st["q"], st["k"], st["v"], offset=0)[0]
        kp, vp, at = st["kp"], st["vp"], torch.arange(c["S"], device="cuda")
        for b in range(c["B"]):
            page = st["table"][b].long()[at // c["page"]]
            kp[page, :, at % c["page"]] = st["k"][b].transpose(0, 1)
            vp[page, :, at % c["page"]] = st["v"][b].transpose(0, 1)
        return o, kp, vp, torch.full_like(st["lengths"], c["S"])
    if kind == "decode_step":
        n = c["S"]
        st["kc"][:, :, n - 1:n] = st["k"]
        st["vc"][:, :, n - 1:n] = st["v"]
        o, lse = _heads64(st, st["q"], st["kc"][:, :, :n], st["vc"][:, :, :n])
        return o, lse[:, :, 0], st["kc"], st["vc"], st["before"] + 1
    o, ls = [], []
    for b, n in enumerate(st["lengths"].tolist()):
        pages = st["table"][b, :-(-n // c["page"])].long()
        k, v = (st[x][pages].transpose(0, 1).flatten(1, 2)[None, :, :n] for x in ("kp", "vp"))
        x, y = _heads64(st, st["q"][b:b + 1], k, v)
        o.append(x)
        ls.append(y[:, :, 0])
    return torch.cat(o), torch.cat(ls)
