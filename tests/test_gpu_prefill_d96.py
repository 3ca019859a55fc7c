"""The prefill kernel at head_dim 96 (quantized, groups of 32): 64-key tiles of rows that are 6 or 3
chunks long, three scale groups per row, 256-row blocks. Edges of its tiles and row blocks, caches
whose scale rows are only 2-byte aligned, and the calls it leaves to the decode kernel, against the
exact fp64 oracle at the usual bars."""

import math

import pytest
import torch

from myinfer_amd import kernels
from tests.helpers import assert_close, exact_reference, seeded_normal
from tests.test_gpu_decode import make_cache
from tests.test_gpu_paged import build

pytestmark = pytest.mark.gpu
DEV = "cuda"
D, G = 96, 32


@pytest.mark.parametrize("B,Hq,Hkv,L,S,bits,dtype,causal,window", [
    (1, 4, 4, 65, 65, 8, torch.float16, True, 0),        # the fewest rows, a ragged second tile
    (1, 2, 1, 33, 64, 4, torch.float16, True, 0),        # one whole tile
    (2, 2, 2, 255, 319, 8, torch.bfloat16, True, 0),     # one row short of a block
    (1, 2, 2, 256, 385, 4, torch.bfloat16, True, 0),
    (1, 8, 2, 65, 1027, 8, torch.float16, False, 0),     # a second row block of 4 rows, keys split
    (1, 3, 1, 301, 4200, 8, torch.float16, True, 0),     # positions cut by row blocks, many splits
    (1, 4, 1, 129, 700, 4, torch.float16, True, 100),    # a window over two tiles
])
def test_shapes(B, Hq, Hkv, L, S, bits, dtype, causal, window):
    print(f"prefill D=96 {B} {Hq} {Hkv} L={L} S={S} bits={bits} {dtype} causal={causal} window={window}", flush=True)
    kt, vt = make_cache(B, Hkv, S, D, bits, dtype, 3100 + S, group=G)
    q = seeded_normal((B, Hq, L, D), 3101 + L, dtype, DEV)
    scale = 1.0 / math.sqrt(D)
    kw = dict(causal=causal, window=window, group_size=G, bits=bits)
    ref = exact_reference(q, kt, vt, scale, **kw)
    assert_close(kernels.attention(q, kt, vt, scale, kernel="prefill", **kw), ref, f"L={L} S={S}")
    assert_close(kernels.attention(q, kt, vt, scale, kernel="decode", **kw), ref, "the decode kernel")


def test_odd_scale_strides_and_row_neighbours():
    """Scale rows at odd element offsets (a head stride that is odd), output rows inside wider ones
    (16-byte aligned: the prefill kernel; 8-byte aligned: the decode kernel), NaN past each sequence."""
    B, Hq, Hkv, L, S = 2, 4, 2, 70, 333
    kt, vt = make_cache(B, Hkv, S, D, 8, torch.float16, 3200, group=G)
    lens = torch.tensor([333, 200], dtype=torch.int32, device=DEV)

    def odd(t):  # the same rows, heads S * 3 + 2 elements apart, the first at an odd element
        per = S * 3 + 2
        buf = torch.full((B * Hkv * per + 1,), float("nan"), dtype=t.dtype, device=DEV)
        v = buf[1:].as_strided(t.shape, (Hkv * per, per, 3, 1), 1)
        v.copy_(t)
        v[1, :, 200:] = float("nan")
        return v

    ref = exact_reference(q := seeded_normal((B, Hq, L, D), 3201, torch.float16, DEV), kt, vt, 0.1, bits=8,
                          group_size=G, causal=True, seq_lens=lens)
    kt, vt = ((c, odd(s), odd(b)) for c, s, b in (kt, vt))
    for first in (0, 4):  # the rows' first element within 128
        wide = torch.full((B, Hq, L, 128), 7.0, dtype=torch.float16, device=DEV)
        out = kernels.attention(q, kt, vt, 0.1, causal=True, seq_lens=lens, group_size=G, bits=8,
                                out=wide[..., first:first + D])
        assert_close(out, ref, f"rows from element {first}")
        assert torch.all(wide[..., :first] == 7.0) and torch.all(wide[..., first + D:] == 7.0)


def test_bf16_beyond_fp16():
    """A bf16 cache with values past 65504: finite through the range exponent (one-shot calls compute
    it), and through the decode kernel where a prepared call has no word."""
    B, Hq, Hkv, L, S = 1, 2, 2, 80, 200
    v = seeded_normal((B, Hkv, S, D), 3301, torch.float32, DEV)
    v[..., 5] *= 1.6e5
    kt = kernels.quantize(seeded_normal((B, Hkv, S, D), 3300, torch.bfloat16, DEV), G, 8)
    vt = kernels.quantize(v.to(torch.bfloat16), G, 8)
    q = seeded_normal((B, Hq, L, D), 3302, torch.bfloat16, DEV)
    kw = dict(causal=True, group_size=G, bits=8)
    ref = exact_reference(q, kt, vt, 0.1, **kw)
    assert_close(kernels.attention(q, kt, vt, 0.1, **kw), ref, "one-shot")
    assert_close(kernels.prepare_attention(q, kt, vt, 0.1, **kw)(), ref, "prepared, no range word")


@pytest.mark.parametrize("paged", [False, True])
@pytest.mark.parametrize("B,Hq,Hkv,L,bits,dtype", [
    (1, 32, 4, 975, 8, torch.float16),   # 31 row blocks of 4 pairs
    (2, 8, 1, 1445, 4, torch.bfloat16),  # 46 of 2
    (4, 5, 1, 1275, 8, torch.float16),   # 25 of 4
    (1, 16, 4, 1600, 8, torch.bfloat16),
    (1, 12, 4, 1904, 4, torch.float16),
])
def test_prompts_of_few_pairs(B, Hq, Hkv, L, bits, dtype, paged):
    """Causal prompts of 2 or 4 (sequence, KV head) pairs, whose row blocks are dealt to the XCDs, at odd
    numbers of row blocks and splits: every row is written and nothing before or after the output."""
    print(f"prefill D=96 {B} {Hq} {Hkv} L={L} bits={bits} {dtype} paged={paged}", flush=True)
    q = seeded_normal((B, Hq, L, D), 3401 + L, dtype, DEV)
    scale = 1.0 / math.sqrt(D)
    kw = dict(causal=True, group_size=G, bits=bits)
    guard = 512 * D
    buf = torch.full((2 * guard + q.numel(),), 7.0, dtype=dtype, device=DEV)
    out = buf[guard:-guard].view(q.shape)
    out.fill_(float("nan"))
    if paged:
        _, table, kp, vp, kt, vt = build(B, Hkv, [L] * B, D, bits, dtype, 3400 + L, group=G)
        lens = torch.full((B,), L, dtype=torch.int32, device=DEV)
        kernels.paged_attention(q, kp, vp, table, lens, scale, max_len=L, out=out, **kw)
    else:
        kt, vt = make_cache(B, Hkv, L, D, bits, dtype, 3400 + L, group=G)
        kernels.attention(q, kt, vt, scale, out=out, **kw)
    assert torch.all(buf[:guard] == 7.0) and torch.all(buf[-guard:] == 7.0)
    assert_close(out, exact_reference(q, kt, vt, scale, **kw), f"L={L}")
