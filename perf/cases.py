"""The calls whose speed this framework is judged by: what a serving program has it do, one attention
layer at a time, through the public entry points, with inputs made from a seed.

Kinds of case (``kind``):
  layer    one layer's step over a ``QuantizedKVCache``: the new keys are rotated, quantized and
           appended in one call, then the queries attend to the cache through the dispatcher that
           model code calls, and the new rows are trimmed again (as a rejected draft or a replayed
           prefix is), so that a pass can be repeated. L = 1 is a decode step, a few rows a
           speculative verification, hundreds a prefill chunk, L = S a whole prompt.
  decode   a prepared decode call (``kernels.prepare_attention``), the form a serving loop keeps.
  paged    a batch of sequences of unequal lengths over a paged pool (``PagedRadixKVCache``).
  dense    attention over an unquantized cache (a plain cache before it is quantized, or the rows of
           a sliding-window cache), causal, with a window or without.
  masked   a prompt batch padded on the left, whose boolean mask the caller built.
  append   the quantize-and-append of a prefill chunk alone.
"""

import math

import torch

from myinfer_amd import attention, kernels
from myinfer_amd.cache import QuantizedKVCache
from myinfer_amd.paged import PAGE_ROWS, PagedRadixKVCache

_DT = {"fp16": torch.float16, "bf16": torch.bfloat16}
_ROPE_BASE = 1000000.0


def _case(name, kind, B, Hq, Hkv, D, L, S, bits, G, dtype, window=0):
    return dict(name=name, kind=kind, B=B, Hq=Hq, Hkv=Hkv, D=D, L=L, S=S, bits=bits, G=G, dtype=dtype, window=window)


def listed():
    return [
        # a decode step of a small model (16 / 8 heads of 128) after 4096 tokens: launches and latency
        _case("step-4k", "layer", 1, 16, 8, 128, 1, 4097, 8, 64, "fp16"),
        # a large model's decode step at 32K tokens, one user: the cache is read once
        _case("decode-32k", "decode", 1, 64, 8, 128, 1, 32768, 8, 64, "fp16"),
        # long context in 4 bits: 128K tokens
        _case("decode-131k-4bit", "decode", 1, 64, 8, 128, 1, 131072, 4, 64, "fp16"),
        # eight users of unequal lengths up to 32K tokens over a paged pool
        _case("paged-8-users", "paged", 8, 64, 8, 128, 1, 32768, 8, 64, "bf16"),
        # five drafted tokens verified for two users
        _case("verify-5", "layer", 2, 32, 4, 128, 5, 9006, 8, 64, "bf16"),
        # the last 512-token chunk of a 16K prompt
        _case("chunk-16k", "layer", 1, 32, 4, 128, 512, 16384, 8, 64, "bf16"),
        # a whole prompt over a plain cache, heads of 64
        _case("prompt-d64-dense", "dense", 1, 32, 8, 64, 1999, 1999, 16, 64, "fp16"),
        # a sliding-window layer's chunk, four users
        _case("window-chunk-dense", "dense", 4, 32, 16, 128, 2048, 3071, 16, 64, "bf16", 1024),
        # a whole prompt of a model with heads of 96 (their groups are 32 wide)
        _case("prompt-d96", "layer", 1, 32, 32, 96, 1999, 1999, 8, 32, "fp16"),
        # a chunk of a model with heads of 256
        _case("chunk-d256", "layer", 1, 16, 8, 256, 2048, 8192, 8, 64, "bf16"),
        # four prompts of unequal lengths padded on the left, 4-bit cache
        _case("prompts-left-padded", "masked", 4, 32, 8, 128, 1023, 1023, 4, 64, "fp16"),
        # the cache update of four users' 2048-token chunk
        _case("append-chunk", "append", 4, 16, 16, 128, 2048, 8192, 8, 64, "bf16"),
    ]


def _pick(rng, lo, hi):
    """A size from lo to hi, even over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


# (query heads, KV heads)
_HEADS = ((16, 8), (64, 8), (32, 4), (32, 16), (32, 8), (32, 32), (16, 16), (8, 1))
_MAX_FLOPS = 2.2e11
_MAX_BYTES = 5e8


def draw(rng):
    while True:
        kind = rng.choice(("step", "decode", "paged", "verify", "chunk", "prompt", "dense", "masked", "append"))
        Hq, Hkv = rng.choice(_HEADS)
        D = rng.choice((64, 128, 128, 256, 96))
        bits, dtype = rng.choice((8, 8, 4)), rng.choice(("fp16", "bf16"))
        B, L, window = 1, 1, 0
        if kind == "step":
            S = _pick(rng, 64, 16384)
        elif kind == "decode":
            B, S = rng.choice((1, 1, 2, 4)), _pick(rng, 1024, 131072)
        elif kind == "paged":
            B, S = rng.randint(2, 16), _pick(rng, 512, 32768)
            D = 128 if D == 96 else D
        elif kind == "verify":
            B, L = rng.choice((1, 2, 4)), rng.randint(2, 8)
            S = L + _pick(rng, 512, 32768)
        elif kind == "chunk":
            L = _pick(rng, 64, 2048)
            S = L + _pick(rng, 256, 16384)
        elif kind == "prompt":
            B, L = rng.choice((1, 1, 2)), _pick(rng, 100, 4096)
            S = L
        elif kind == "dense":
            B, D, bits = rng.choice((1, 2, 4)), rng.choice((64, 128, 128)), 16
            form = rng.choice(("step", "prompt", "window"))
            L = 1 if form == "step" else _pick(rng, 100, 4096 if form == "prompt" else 2048)
            S = _pick(rng, 256, 8192) if form == "step" else L
            if form == "window":
                window = rng.choice((512, 1024))
                S = L + window - 1
        elif kind == "masked":
            B, L = rng.choice((2, 4)), _pick(rng, 64, 1500)
            S = L
        else:
            B, L = rng.choice((1, 2, 4)), _pick(rng, 64, 4096)
            S = L + rng.randint(0, 4096)
        G = 64 if D != 96 else 32
        kind = {"step": "layer", "verify": "layer", "chunk": "layer", "prompt": "layer"}.get(kind, kind)
        case = dict(kind=kind, B=B, Hq=Hq, Hkv=Hkv, D=D, L=L, S=S, bits=bits, G=G, dtype=dtype, window=window)
        w = work(case)
        if w["flops"] <= _MAX_FLOPS and w["bytes"] <= _MAX_BYTES:
            return case


# ---- inputs

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _rows(g, B, H, n, D, dt):
    """K or V rows as projections give them: normal, each dim at a scale of its own within a factor of
    two or so."""
    dims = torch.exp(0.3 * torch.randn(1, 1, 1, D, generator=g, device="cuda"))
    return (torch.randn(B, H, n, D, generator=g, device="cuda") * dims).to(dt)


def _inputs(case, seed):
    """The tensors of a case, from its seed alone: queries, the K and V rows of the whole context (the
    last L of them are the call's own), and what the kind adds."""
    g, dt = _gen(seed), _DT[case["dtype"]]
    B, Hq, Hkv, D, L, S = (case[k] for k in ("B", "Hq", "Hkv", "D", "L", "S"))
    x = {"q": torch.randn(B, Hq, L, D, generator=g, device="cuda").to(dt),
         "k": _rows(g, B, Hkv, S, D, dt), "v": _rows(g, B, Hkv, S, D, dt)}
    if case["kind"] == "paged":
        x["lens"] = torch.randint(S // 2, S + 1, (B,), generator=g, device="cuda").to(torch.int32)
        pages = -(-S // PAGE_ROWS)
        x["table"] = torch.randperm(B * pages, generator=g, device="cuda").view(B, pages).to(torch.int32)
    if case["kind"] == "masked":
        pad = torch.randint(0, S // 2 + 1, (B,), generator=g, device="cuda")
        pad[0] = 0  # the longest prompt has none
        k = torch.arange(S, device="cuda")
        x["mask"] = ((k[None, :] <= k[:, None])[None] & (k[None, None, :] >= pad[:, None, None]))[:, None]
    return x


def _scale(case):
    return 1.0 / math.sqrt(case["D"])


def _rope(case):
    return kernels.Rope(dims=case["D"], base=_ROPE_BASE)


def _filled(case, k, v, rows, reserve):
    cache = QuantizedKVCache(group_size=case["G"], bits=case["bits"])
    cache.reserve(k, reserve)
    if rows:
        cache.update_and_fetch(k[:, :, :rows].contiguous(), v[:, :, :rows].contiguous())
    return cache


def prepare(case, seed):
    x = _inputs(case, seed)
    kind, L, S = case["kind"], case["L"], case["S"]
    st = {"case": case, "q": x["q"], "scale": _scale(case)}
    if kind in ("layer", "append"):
        st["cache"] = _filled(case, x["k"], x["v"], S - L, S)
        st["k"], st["v"] = x["k"][:, :, S - L:].contiguous(), x["v"][:, :, S - L:].contiguous()
        st["rope"] = _rope(case) if kind == "layer" else None
        st["mask"] = "causal" if L > 1 else None
    elif kind == "decode":
        st["cache"] = _filled(case, x["k"], x["v"], S, S)
        keys, values = st["cache"].fetch()
        st["call"] = kernels.prepare_attention(x["q"], keys, values, st["scale"], group_size=case["G"],
                                               bits=case["bits"])
    elif kind == "paged":
        B, pages = x["table"].shape
        pool = PagedRadixKVCache(1, case["Hkv"], case["D"], max_blocks=B * pages, bits=case["bits"],
                                 group_size=case["G"], dtype=_DT[case["dtype"]])
        pool.append(0, x["k"], x["v"], x["table"])
        st.update(pool=pool, table=x["table"], lens=x["lens"])
    elif kind == "dense":
        st["k"], st["v"] = x["k"], x["v"]
    else:
        keys, values = _filled(case, x["k"], x["v"], S, S).fetch()
        st.update(keys=keys, values=values, mask=x["mask"])
    return st


def run(state):
    case = state["case"]
    kind, L, S = case["kind"], case["L"], case["S"]
    if kind == "decode":
        return state["call"]()
    if kind == "paged":
        return state["pool"].attention(0, state["q"], state["table"], state["lens"], state["scale"], max_len=S)
    if kind == "dense":
        return attention.fast_scaled_dot_product_attention(state["q"], state["k"], state["v"], state["scale"],
                                                           "causal", window=case["window"])
    if kind == "masked":
        return attention.blocked_quantized_sdpa(state["q"], state["keys"], state["values"], state["scale"],
                                                state["mask"], case["G"], case["bits"])
    cache = state["cache"]
    keys, values = cache.update_and_fetch(state["k"], state["v"], rope=state["rope"])
    out = None
    if kind == "layer":
        out = attention.scaled_dot_product_attention(state["q"], keys, values, cache, state["scale"], state["mask"])
    cache.trim(L)
    new = [[t[:, :, S - L:].view(torch.int32) if t.dtype == torch.uint32 else t[:, :, S - L:] for t in tr]
           for tr in (keys, values)]
    return {"keys": new[0], "values": new[1]} if out is None else {"out": out, "keys": new[0], "values": new[1]}


# ---- what a pass cannot do without

def _pairs(case):
    """Visible (query, key) pairs of one query head, over the batch (lengths at their expectation)."""
    B, L, S, W = case["B"], case["L"], case["S"], case["window"]
    if case["kind"] == "paged":
        return B * 0.75 * S
    if case["kind"] == "masked":
        return L * (L + 1) / 2 + (B - 1) * 7 / 24 * L * L  # pads even over [0, S / 2]
    if W:
        return B * sum(min(S - L + i + 1, W) for i in range(L))
    return B * (L * (S - L) + L * (L + 1) / 2)


def work(case):
    B, Hq, Hkv, D, L, S, bits, G = (case[k] for k in ("B", "Hq", "Hkv", "D", "L", "S", "bits", "G"))
    row = 2 * 2 * D if bits == 16 else 2 * (D * bits // 8 + 2 * 2 * D // G)  # bytes of a key and its value
    new = 2 * 2 * D  # the same, as the call is given them
    if case["kind"] == "append":
        return {"bytes": B * Hkv * L * (new + row), "flops": 2.0 * B * Hkv * L * 2 * D}
    rows = B * S * (0.75 if case["kind"] == "paged" else 1.0)
    nbytes = rows * Hkv * row + 2 * B * Hq * L * D * 2
    if case["kind"] == "layer":
        nbytes += B * Hkv * L * new
    if case["kind"] == "masked":
        nbytes += B * L * S
    return {"bytes": nbytes, "flops": 4.0 * D * Hq * _pairs(case)}


def tolerance(case):
    """Appended codes, scales and biases are fixed to the bit. An attention output carries the rounding
    of its type and of the 16-bit operands of its products (against 64 bits: 2.6e-4 to 9e-4 in fp16, 2e-3
    to 2.4e-3 in bf16; at 4 bits up to 4.7e-3, where a large bias cancels in a long average); a key that
    was rotated may land on the neighbouring value of its type, and its code with it."""
    if case["kind"] == "append":
        return "exact"
    if case["bits"] == 4:
        rel = 1.5e-2
    elif case["dtype"] == "bf16":
        rel = 9e-3
    else:
        rel = 1.5e-3 if case["bits"] == 16 else 3.5e-3
    return {"rel": rel, "max": 16 * rel, "differ": 2e-3}


# ---- the same in plain torch and 64 bits

def _quantized(x, bits, G):
    """(codes, scales, biases) of MLX's affine quantizer, whose own definition is in 32 bits."""
    n = float(2 ** bits - 1)
    y = x.float().view(*x.shape[:-1], -1, G)
    lo, hi = y.amin(-1, keepdim=True), y.amax(-1, keepdim=True)
    low = lo.abs() > hi.abs()
    s = torch.clamp((hi - lo) / n, min=1e-7)
    s = torch.where(low, s, -s)
    edge = torch.where(low, lo, hi)
    q0 = torch.round(edge / s)
    s = torch.where(q0 != 0, edge / torch.where(q0 != 0, q0, torch.ones_like(q0)), s)
    b = torch.where(q0 != 0, edge, torch.zeros_like(edge))
    codes = torch.clamp(torch.round((y - b) / s), 0, n)
    return codes, s.to(x.dtype), b.to(x.dtype)


def _read_back(x, bits, G):
    codes, s, b = _quantized(x, bits, G)
    return (codes.double() * s.double() + b.double()).view(x.shape)


def _rotated(x, first):
    D = x.shape[-1]
    freq = 1.0 / _ROPE_BASE ** (torch.arange(0, D, 2, device=x.device, dtype=torch.float64) / D)
    a = torch.arange(first, first + x.shape[2], device=x.device, dtype=torch.float64)[:, None] * freq
    u, w = x.double().chunk(2, dim=-1)
    return torch.cat([u * a.cos() - w * a.sin(), w * a.cos() + u * a.sin()], dim=-1).to(x.dtype)


def _attend(q, k, v, scale, visible):
    """q [Hq, L, D], k and v [Hkv, S, D] in 64 bits, visible [L, S] or None."""
    Hkv, rep = k.shape[0], q.shape[0] // k.shape[0]
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    for h in range(Hkv):
        keys_t = k[h].t().contiguous()
        for r in range(rep):
            s = (q[h * rep + r].double() @ keys_t) * scale
            if visible is not None:
                s = s.masked_fill(~visible, -math.inf)
            p = torch.exp(s - s.amax(-1, keepdim=True).clamp(min=-1e300))
            out[h * rep + r] = (p @ v[h]) / p.sum(-1, keepdim=True).clamp(min=1e-300)
    return out


def exact(case, seed):
    x = _inputs(case, seed)
    kind, L, S, bits, G = (case[k] for k in ("kind", "L", "S", "bits", "G"))
    if kind == "append":
        new = [_quantized(x[n][:, :, S - L:], bits, G) for n in ("k", "v")]
        return {"keys": [None, *(t[..., 0].double() for t in new[0][1:])],
                "values": [None, *(t[..., 0].double() for t in new[1][1:])]}
    k, v = x["k"], x["v"]
    if kind == "layer":
        k = torch.cat([k[:, :, : S - L], _rotated(k[:, :, S - L:], S - L)], dim=2)
    outs = []
    for b in range(case["B"]):
        n = int(x["lens"][b]) if kind == "paged" else S
        kb, vb = (t[b, :, :n].double() if bits == 16 else _read_back(t[b, :, :n], bits, G) for t in (k, v))
        if kind == "masked":
            visible = x["mask"][b, 0]
        elif L == 1:
            visible = None
        else:
            pos, key = torch.arange(n - L, n, device="cuda")[:, None], torch.arange(n, device="cuda")[None]
            visible = key <= pos
            if case["window"]:
                visible &= key > pos - case["window"]
        outs.append(_attend(x["q"][b], kb, vb, _scale(case), visible))
    out = torch.stack(outs)
    if kind != "layer":
        return out
    return {"out": out, "keys": [None] * 3, "values": [None] * 3}
