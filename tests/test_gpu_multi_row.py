"""Quantized decode over several passes' query rows (the MULTI kernels): row blocks at their edges, unit
counts that do not divide the grid, every width and group, contiguous and paged, against the exact
fp64 oracle; and the rounding of their value sums, which may not exceed the prefill kernels'."""

import math

import pytest
import torch

from myinfer_amd import kernels
from tests.helpers import assert_close, exact_reference, seeded_normal
from tests.test_gpu_decode import make_cache

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("B,Hq,Hkv,L,S,D,G,bits,dtype,window", [
    (1, 8, 4, 5, 700, 128, 64, 8, torch.float16, 0),     # 10 rows: the second row block has two
    (3, 8, 1, 3, 4100, 128, 64, 4, torch.bfloat16, 0),   # 9 units, splits merged by the combine launch
    (2, 12, 4, 7, 333, 128, 32, 8, torch.float16, 0),    # 4 rows a pass, 21 rows
    (1, 8, 2, 9, 1000, 128, 128, 4, torch.float16, 77),  # 16 rows a pass, a window over two tiles
    (2, 16, 2, 5, 515, 64, 64, 8, torch.float16, 0),     # 40 rows, 16 a pass
    (1, 6, 2, 11, 900, 64, 32, 4, torch.bfloat16, 200),
    (2, 8, 2, 4, 640, 256, 64, 8, torch.float16, 0),
    (1, 4, 1, 40, 40, 256, 128, 4, torch.bfloat16, 0),   # a whole short prompt
    (1, 8, 1, 64, 64, 128, 64, 8, torch.float16, 0),
])
def test_against_exact(B, Hq, Hkv, L, S, D, G, bits, dtype, window):
    print(f"multi-row {B} {Hq} {Hkv} L={L} S={S} D={D} G={G} bits={bits} {dtype} window={window}", flush=True)
    kt, vt = make_cache(B, Hkv, S, D, bits, dtype, 4000 + S, group=G)
    q = seeded_normal((B, Hq, L, D), 4001 + L, dtype, DEV)
    lens = torch.tensor([S] + [max(L, S - 37 * b) for b in range(1, B)], dtype=torch.int32, device=DEV)
    kw = dict(causal=True, window=window, seq_lens=lens, group_size=G, bits=bits)
    scale = 1.0 / math.sqrt(D)
    out = kernels.attention(q, kt, vt, scale, kernel="decode", **kw)
    assert_close(out, exact_reference(q, kt, vt, scale, **kw), f"rows={Hq // Hkv * L} S={S}")


@pytest.mark.parametrize("D,bits", [(128, 8), (128, 4), (64, 8), (256, 8)])
def test_rounding_is_no_larger_than_prefill(D, bits):
    """fp16 rel-L2 against 64 bits over 3000 keys. Bound: 4.0e-4, from the output's own rounding (an
    fp16 output: 2^-11 / sqrt(3) = 2.8e-4 at most) and as much again in quadrature for the rounding of
    p s with its codes centred; without the centring it measures 4.5e-4 to 5.6e-4."""
    B, Hq, Hkv, L, S = 1, 16, 2, 5, 3000
    kt, vt = make_cache(B, Hkv, S, D, bits, torch.float16, 4100 + D)
    q = seeded_normal((B, Hq, L, D), 4101, torch.float16, DEV)
    kw = dict(causal=True, group_size=64, bits=bits)
    ref = torch.from_numpy(exact_reference(q, kt, vt, D ** -0.5, **kw))

    def err(kernel):
        o = kernels.attention(q, kt, vt, D ** -0.5, kernel=kernel, **kw).cpu().double()
        return float((o - ref).norm() / ref.norm())

    multi, prefill = err("decode"), err("prefill")
    assert multi <= 4.0e-4 and multi <= prefill * 1.05, (multi, prefill)


@pytest.mark.parametrize("D,G,bits", [(128, 64, 8), (64, 64, 4), (256, 64, 8)])
def test_paged_equals_contiguous(D, G, bits):
    from tests.test_gpu_paged import build

    B, Hkv, Hq, L = 3, 2, 16, 5
    lens = [300, 64, 1500]
    _, tables, kp, vp, kc, vc = build(B, Hkv, lens, D, bits, torch.float16, 4200, group=G)
    seq = torch.tensor(lens, dtype=torch.int32, device=DEV)
    q = seeded_normal((B, Hq, L, D), 4201, torch.float16, DEV)
    kw = dict(causal=True, group_size=G, bits=bits, kernel="decode")
    out = kernels.paged_attention(q, kp, vp, tables, seq, 0.1, max_len=max(lens), **kw)
    assert torch.equal(out, kernels.attention(q, kc, vc, 0.1, seq_lens=seq, **kw))
