"""General masks on the prefill kernel: tiles that no row, some rows or all rows see, left-padded batches,
per-head masks, rows at any byte offset, many splits and none, rows and whole sequences that see nothing,
against the exact fp64 oracle."""

import math

import pytest
import torch

from myinfer_amd import attention as A
from myinfer_amd import kernels
from oracle import attention as OA
from tests.helpers import assert_close, seeded_normal
from tests.test_gpu_decode import make_cache
from tests.test_gpu_masks import _exact

pytestmark = pytest.mark.gpu
DEV = "cuda"


def left_padded(B, L, S, pads):
    pos, k = torch.arange(S - L, S)[:, None], torch.arange(S)[None]
    return ((k <= pos)[None] & (k[None] >= torch.tensor(pads)[:, None, None]))[:, None]


@pytest.mark.parametrize("B,Hq,Hkv,L,S,D,bits,dtype,pads", [
    (2, 16, 4, 300, 300, 128, 8, torch.float16, [0, 141]),       # rows of 300 bytes: every alignment
    (4, 8, 8, 257, 257, 128, 4, torch.float16, [0, 1, 64, 256]),  # one query left; a second row block of one row
    (2, 8, 4, 600, 600, 64, 8, torch.float16, [600, 63]),        # a sequence that sees nothing: zeros
    (1, 8, 8, 400, 400, 96, 8, torch.float16, [37]),
    (1, 8, 2, 40, 9000, 128, 8, torch.float16, [5000]),          # 3 bitmap words, tiles skipped, many splits
])
def test_left_padded(B, Hq, Hkv, L, S, D, bits, dtype, pads):
    print(f"left padded {B} {Hq} {Hkv} L={L} S={S} D={D} bits={bits} {dtype} {pads}", flush=True)
    G = 32 if D == 96 else 64
    kt, vt = make_cache(B, Hkv, S, D, bits, dtype, 4700 + S, group=G)
    q = seeded_normal((B, Hq, L, D), 4701 + L, dtype, DEV)
    m = left_padded(B, L, S, pads)
    scale = 1.0 / math.sqrt(D)
    out = A.blocked_quantized_sdpa(q, kt, vt, scale, m.to(DEV), G, bits)
    assert_close(out, _exact(q, kt, vt, scale, bits, G, vis=m.numpy()), f"pads {pads}")
    assert torch.equal(out, A.blocked_quantized_sdpa(q, kt, vt, scale, m.to(DEV), G, bits))


@pytest.mark.parametrize("heads,dtype", [("kv", torch.bfloat16), ("query", torch.float16)])
def test_per_head_masks(heads, dtype):
    """A mask per KV head (its own tile classes) or per query head (256 mask rows a row block), block-sparse;
    the bf16 cache keeps range words."""
    from myinfer_amd.cache import QuantizedKVCache

    B, Hq, Hkv, L, S, D = 1, 16, 4, 260, 700, 128
    cache = QuantizedKVCache(64, 8)
    kt, vt = cache.update_and_fetch(*(seeded_normal((B, Hkv, S, D), 4800 + i, dtype, DEV) for i in range(2)))
    q = seeded_normal((B, Hq, L, D), 4802, dtype, DEV)
    g = torch.Generator().manual_seed(4803)
    H = Hkv if heads == "kv" else Hq
    m = (torch.rand(B, H, 5, 11, generator=g) < 0.4).repeat_interleave(52, 2).repeat_interleave(64, 3)[:, :, :L, :S]
    m = m & (torch.rand(B, H, L, S, generator=g) < 0.9)
    vis = m.repeat_interleave(Hq // H, 1).numpy()
    if heads == "kv":
        out = A.blocked_quantized_sdpa(q, kt, vt, 0.09, m.to(DEV), 64, 8)
    else:
        out = kernels.masked_attention(q, kt, vt, 0.09, m.to(DEV), layout="heads")
    assert_close(out, _exact(q, kt, vt, 0.09, 8, 64, vis=vis), f"{heads} heads")


@pytest.mark.parametrize("D,dtype,kind", [(128, torch.float16, "bool"), (64, torch.bfloat16, "bool"),
                                          (128, torch.bfloat16, "f32"), (64, torch.float16, "same"),
                                          (64, torch.float16, "lowest")])
def test_unquantized(D, dtype, kind):
    """Unquantized caches: boolean masks, additive masks in fp32 and in the cache's type (ALiBi-like slopes
    with a causal cut), and the type's lowest value as the cut."""
    B, Hq, Hkv, L, S = 2, 8, 2, 333, 501
    k, v = (seeded_normal((B, Hkv, S, D), 4900 + i, dtype, DEV) for i in range(2))
    q = seeded_normal((B, Hq, L, D), 4902, dtype, DEV)
    vis = left_padded(B, L, S, [0, 130 if kind != "lowest" else 230])  # (the first position is 168)
    if kind == "bool":
        mask, kw = vis, dict(vis=vis.numpy())
    else:
        slope = -0.01 * (torch.arange(S - L, S)[:, None] - torch.arange(S)[None]).abs().float() * torch.arange(1, 9)[:, None, None]
        mt = torch.float32 if kind == "f32" else dtype
        mask = slope.to(mt)[None].expand(B, 8, L, S).clone()
        cut = float("-inf") if kind != "lowest" else torch.finfo(mt).min
        mask = torch.where(vis, mask, torch.tensor(cut, dtype=mt))
        kw = dict(add=mask.double().numpy())
    out = A.fast_scaled_dot_product_attention(q, k, v, 0.1, mask.to(DEV))
    qn, kn, vn = (t.cpu().double().numpy() for t in (q, k, v))
    ref = OA.exact_attention(qn, kn, vn, 0.1, **kw)
    if kind == "lowest":
        # A row whose every key is cut: fp16's lowest value is finite, so the row attends by its scores; added to it
        # in fp32 they are rounded to 2^-7 (half of it either way, in log2 units), a probability by up to
        # 2^-8 ln 2 = 0.27% and an output, whose values' signs differ, by less. (fp32's and bf16's lowest values
        # are beyond fp32 in those units and hide the keys.)
        seen = vis.any(-1)[:, 0].numpy()
        o = out.transpose(1, 2)[torch.from_numpy(~seen).to(DEV)].cpu().double().numpy()
        r = ref.transpose(0, 2, 1, 3)[~seen]
        assert len(r) and OA.error_stats(o, r)["rel_l2"] <= 2.7e-3 + 1e-3
        out, ref = out.transpose(1, 2)[torch.from_numpy(seen).to(DEV)], ref.transpose(0, 2, 1, 3)[seen]
    assert_close(out, ref, f"{kind} D={D}")


def test_workspace_too_small():
    """A masked call that needs more than the stream's workspace gets a larger one and the same results."""
    B, Hq, Hkv, L, S, D = 1, 8, 2, 200, 3000, 128
    kt, vt = make_cache(B, Hkv, S, D, 8, torch.float16, 5100)
    q = seeded_normal((B, Hq, L, D), 5101, torch.float16, DEV)
    m = left_padded(B, L, S, [77]).to(DEV)
    ref = kernels.masked_attention(q, kt, vt, 0.1, m, layout="blocked")
    kernels._workspaces.clear()
    kernels.masked_attention(q[:, :, :1], kt, vt, 0.1, m[:, :, :1], layout="blocked")
    small = max(w.numel() for w in kernels._workspaces.values())
    assert torch.equal(kernels.masked_attention(q, kt, vt, 0.1, m, layout="blocked"), ref)
    assert max(w.numel() for w in kernels._workspaces.values()) > small
    with pytest.raises(ValueError):
        kernels.masked_attention(q, kt, vt, float("nan"), m, layout="blocked")
    with pytest.raises(NotImplementedError):
        kernels.masked_attention(q[:, :, :0], kt, vt, 0.1, m[:, :, :0], layout="blocked")


def test_mask_and_call_that_stay_on_decode():
    """The same left-padded mask as an additive one over a quantized cache, and into output rows the
    prefill kernel cannot store, give the boolean call's results within two roundings."""
    B, Hq, Hkv, L, S, D = 1, 16, 4, 300, 300, 128
    kt, vt = make_cache(B, Hkv, S, D, 8, torch.float16, 5000)
    q = seeded_normal((B, Hq, L, D), 5001, torch.float16, DEV)
    m = left_padded(B, L, S, [41])
    ref = _exact(q, kt, vt, 0.1, 8, 64, vis=m.numpy())
    add = torch.where(m, 0.0, float("-inf")).half().to(DEV)
    assert_close(A.blocked_quantized_sdpa(q, kt, vt, 0.1, add), ref, "additive")
    wide = torch.zeros((B, Hq, L, D + 8), dtype=torch.float16, device=DEV)
    out = kernels.masked_attention(q, kt, vt, 0.1, m.to(DEV), layout="blocked", out=wide[..., 4:4 + D])
    assert_close(out, ref, "rows at 8 bytes")
