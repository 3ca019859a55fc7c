"""How prefill calls are cut into splits and merged: causal prompts whose row blocks take one to four
splits of equal length (numbered from the longest down, over one or several (sequence, KV head) pairs
per XCD), and calls of many splits, whose partials a launch of their own merges; against the exact fp64
oracle, and replayed from a graph."""

import math

import pytest
import torch

from myinfer_amd import kernels
from tests.helpers import assert_close, exact_reference, seeded_normal
from tests.test_gpu_decode import make_cache

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("B,Hq,Hkv,L,S,D,bits,dtype,lens", [
    (1, 8, 8, 1100, 1100, 128, 8, torch.float16, None),          # a pair per XCD, 5 row blocks of 1 to 4 splits
    (1, 8, 2, 520, 520, 128, 4, torch.bfloat16, None),           # 2 pairs
    (3, 4, 1, 700, 700, 64, 8, torch.float16, [700, 701 - 64, 700 - 250]),  # 3 pairs
    (1, 16, 16, 900, 900, 64, 8, torch.float16, None),           # two pairs per XCD
    (1, 4, 2, 70, 4096, 128, 8, torch.float16, None),            # 16 splits, a ragged row block
    (2, 2, 1, 300, 9000, 64, 4, torch.bfloat16, [9000, 310]),    # 64 splits for one sequence, two for the other
    (1, 8, 1, 40, 16500, 128, 8, torch.float16, None),           # 65 splits: more than one round of the merge
    (1, 2, 2, 100, 5000, 96, 8, torch.float16, None),
    (1, 2, 2, 1600, 1600, 128, 8, torch.float16, None),          # a prompt of 5 splits: a merge launch over 1 to 5
    (2, 1, 1, 1500, 1500, 64, 4, torch.float16, [1500, 700]),    # 6
])
def test_splits(B, Hq, Hkv, L, S, D, bits, dtype, lens):
    G = 32 if D == 96 else 64
    print(f"prefill splits {B} {Hq} {Hkv} L={L} S={S} D={D} bits={bits} {dtype} lens={lens}", flush=True)
    kt, vt = make_cache(B, Hkv, S, D, bits, dtype, 4400 + S, group=G)
    q = seeded_normal((B, Hq, L, D), 4401 + L, dtype, DEV)
    seq = None if lens is None else torch.tensor(lens, dtype=torch.int32, device=DEV)
    kw = dict(causal=True, seq_lens=seq, group_size=G, bits=bits)
    scale = 1.0 / math.sqrt(D)
    ref = exact_reference(q, kt, vt, scale, **kw)
    out = kernels.attention(q, kt, vt, scale, kernel="prefill", **kw)
    assert_close(out, ref, f"L={L} S={S}")
    assert torch.equal(out, kernels.attention(q, kt, vt, scale, kernel="prefill", **kw))


@pytest.mark.parametrize("form,B,Hq,Hkv,L,S,D,bits", [
    ("causal", 1, 2, 2, 100, 5000, 96, 8),    # many splits, merged by their own launch
    ("causal", 1, 4, 4, 900, 900, 96, 4),     # a few, merged by the last of them
    ("causal", 1, 8, 2, 100, 3000, 64, 16),
    ("causal", 1, 8, 4, 900, 900, 64, 16),
    ("masked", 1, 8, 2, 100, 5000, 128, 8),
    ("masked", 1, 8, 2, 160, 3000, 64, 4),
    ("masked", 1, 8, 2, 100, 5000, 128, 16),
    ("masked", 2, 8, 4, 130, 700, 96, 8),
])
def test_partials_in_fp32(form, B, Hq, Hkv, L, S, D, bits):
    """Zero queries over whole-number values: every probability and every sum is exact, so an output is the
    correctly rounded mean but for the last bits of one fp32 division (a share of about 2^-12 near a tie).
    Partial rows rounded to fp16 on the way would miss it in a quarter of the elements or so."""
    print(f"fp32 partials {form} {B} {Hq} {Hkv} L={L} S={S} D={D} bits={bits}", flush=True)
    G, top = (32 if D == 96 else 64), (255 if bits != 4 else 15)
    v = torch.randint(0, top + 1, (B, Hkv, S, D), generator=torch.Generator().manual_seed(4700 + S + D))
    v[..., ::32], v[..., 1::32] = 0, top  # the groups' extremes: scale -1, bias `top`
    k = seeded_normal((B, Hkv, S, D), 4701, torch.float16, DEV)
    vd = v.half().to(DEV)
    kt, vt = (k, vd) if bits == 16 else (kernels.quantize(k, G, bits), kernels.quantize(vd, G, bits))
    q = torch.zeros((B, Hq, L, D), dtype=torch.float16, device=DEV)
    visible = torch.ones((L, S), dtype=torch.bool).tril(S - L)
    if form == "masked":
        visible[:, ::3] = False  # (no structure that the causal kernels take)
        mask = visible.to(DEV)
        out = kernels.masked_attention(q, kt, vt, 0.1, mask, group_size=G, bits=bits if bits != 16 else 8)
    else:
        out = kernels.attention(q, kt, vt, 0.1, causal=True, group_size=G, bits=bits if bits != 16 else 8, kernel="prefill")
    mean = visible.double() @ v.double() / visible.double().sum(-1, keepdim=True)
    want = mean.half().repeat_interleave(Hq // Hkv, dim=1)
    off = (out.cpu() != want).double().mean().item()
    assert off < 0.005, off


def test_unquantized_d64_rows_of_8_bytes():
    """Unquantized head_dim-64 prefill into output rows that are only 8-byte aligned, many splits and none."""
    for L, S in ((100, 3000), (300, 300)):
        q = seeded_normal((1, 8, L, 64), 4500, torch.float16, DEV)
        k, v = (seeded_normal((1, 2, S, 64), 4501 + i, torch.float16, DEV) for i in range(2))
        wide = torch.full((1, 8, L, 72), 7.0, dtype=torch.float16, device=DEV)
        out = kernels.attention(q, k, v, 0.125, causal=True, out=wide[..., 4:68], kernel="prefill")
        assert torch.equal(out, kernels.attention(q, k, v, 0.125, causal=True, kernel="prefill"))
        assert torch.all(wide[..., :4] == 7.0) and torch.all(wide[..., 68:] == 7.0)


def test_merge_launch_in_a_graph():
    kt, vt = make_cache(1, 2, 6000, 128, 8, torch.float16, 4600)
    q = seeded_normal((1, 8, 90, 128), 4601, torch.float16, DEV)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        call = kernels.prepare_attention(q, kt, vt, 0.1, causal=True, kernel="prefill")
        eager = call().clone()
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            call()
    for i in range(3):
        call.out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(call.out, eager), f"replay {i}"
        torch.randn(1 << 20, device=DEV).sum().item()  # the program's own work between replays
