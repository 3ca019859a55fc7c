"""The native host path of a layer's step (csrc/host): the same results, bit for bit, as the prepared calls
it stands for, over the forms it takes, and the same errors for the forms it hands back."""

import ctypes
import subprocess
import threading

import pytest
import torch

from myinfer_amd import _lib
from myinfer_amd import attention as A
from myinfer_amd import kernels
from myinfer_amd.cache import QuantizedKVCache
from tests.helpers import seeded_normal
from tests.test_gpu_decode import make_cache

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("B,Hq,Hkv,L,S,cap,D,G,bits,dtype,window,lens", [
    (1, 16, 8, 1, 333, 512, 128, 64, 8, torch.float16, 0, None),       # a capacity view
    (2, 16, 2, 5, 700, None, 128, 64, 4, torch.float16, 0, [700, 41]),  # several row blocks, lengths
    (1, 8, 2, 1, 900, None, 256, 64, 8, torch.bfloat16, 100, None),    # a window
    (2, 4, 4, 90, 90, None, 64, 64, 8, torch.float16, 0, None),        # a prompt on the prefill kernel
    (1, 4, 4, 120, 300, None, 96, 32, 8, torch.float16, 0, None),
])
@pytest.mark.parametrize("int32_codes", [False, True])
def test_equals_the_prepared_call(B, Hq, Hkv, L, S, cap, D, G, bits, dtype, window, lens, int32_codes):
    kt, vt = make_cache(B, Hkv, S, D, bits, dtype, 5200 + S, cap=cap, group=G)
    if int32_codes:
        kt, vt = ((c.view(torch.int32), s, b) for c, s, b in (kt, vt))
    q = seeded_normal((B, Hq, L, D), 5201, dtype, DEV)
    seq = None if lens is None else torch.tensor(lens, dtype=torch.int32, device=DEV)
    kw = dict(causal=True, window=window, seq_lens=seq, group_size=G, bits=bits)
    ref = kernels.attention(q, kt, vt, 0.11, **kw)
    out = kernels.layer_attention(q, kt, vt, 0.11, **kw)
    assert out is not None and torch.equal(out, ref)
    assert torch.equal(A.blocked_quantized_sdpa(q, kt, vt, 0.11, "causal", G, bits, window=window, seq_lens=seq), ref)
    # forms it hands to the general path: queries to copy, triples as lists
    odd = torch.empty(B, Hq, L, D + 4, dtype=dtype, device=DEV)[..., :D].copy_(q)
    assert kernels.layer_attention(odd, kt, vt, 0.11, **kw) is None
    assert torch.equal(A.blocked_quantized_sdpa(odd, list(kt), list(vt), 0.11, "causal", G, bits, window=window,
                                                seq_lens=seq), ref)


def test_refusals_are_the_general_paths():
    kt, vt = make_cache(1, 2, 100, 128, 8, torch.float16, 5300)
    q = seeded_normal((1, 4, 1, 128), 5301, torch.float16, DEV)
    for args, kw in [((q.bfloat16(), kt, vt), {}), ((q, kt, (vt[0], vt[1][:, :, :50], vt[2])), {}),
                     ((q[:, :3], kt, vt), {}), ((q, kt, vt), dict(bits=4)), ((q.cpu(), kt, vt), {}),
                     ((q, kt, vt), dict(seq_lens=torch.tensor([100], device=DEV)))]:
        with pytest.raises((ValueError, NotImplementedError)):
            A.blocked_quantized_sdpa(*args, 0.1, None, **kw)
    with pytest.raises(ValueError):
        A.blocked_quantized_sdpa(q, kt, vt, float("nan"), None)


def test_bf16_prefill_reads_the_range_words():
    """Values past the fp16 range: through a cache (words) and over bare triples (the general path)."""
    k, v = (seeded_normal((1, 2, 200, 128), 5400 + i, torch.bfloat16, DEV) for i in range(2))
    v = v * 1e5
    q = seeded_normal((1, 4, 150, 128), 5402, torch.bfloat16, DEV)
    cache = QuantizedKVCache(64, 8)
    kt, vt = cache.update_and_fetch(k, v)
    out = A.blocked_quantized_sdpa(q, kt, vt, 0.1, "causal", 64, 8)
    assert torch.isfinite(out).all()
    assert torch.equal(out, kernels.attention(q, kt, vt, 0.1, causal=True, bits=8, kernel="prefill"))
    bare = [tuple(x.clone() for x in tr) for tr in (kt, vt)]
    assert kernels.layer_attention(q, *bare, 0.1, causal=True) is None
    assert torch.equal(A.blocked_quantized_sdpa(q, *bare, 0.1, "causal", 64, 8), out)


def test_append_forms_and_streams():
    """Appends through the native path, from views whose rows it reads in place and from ones it hands
    back, on two streams, equal quantize_append; a refused append changes nothing."""
    B, H, D = 2, 4, 128
    rows = seeded_normal((B, 9, H, D), 5500, torch.float16, DEV)  # projections: heads inside
    r = kernels.Rope(dims=128, base=1e6)
    ref = QuantizedKVCache(64, 8)
    ref.reserve(rows.transpose(1, 2), 256)
    kernels.quantize_append(rows.transpose(1, 2).contiguous(), ref.keys, rows.transpose(1, 2).contiguous(), ref.values,
                            0, rope=r)
    for stream in (torch.cuda.current_stream(), torch.cuda.Stream()):
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            cache = QuantizedKVCache(64, 8)
            cache.reserve(rows.transpose(1, 2), 256)
            for l0, l1 in ((0, 1), (1, 9)):
                x = rows[:, l0:l1].transpose(1, 2)
                got = cache.update_and_fetch(x, x, rope=r)
            with pytest.raises(ValueError):
                cache.update_and_fetch(rows[:, :2].transpose(1, 2).bfloat16(), rows[:, :2].transpose(1, 2).bfloat16())
            stream.synchronize()
        for a, b in zip(got[0] + got[1], ref.keys + ref.values):
            assert a.shape[2] == 9 and a.stride() == b.stride()
            assert torch.equal(a.view(torch.int16), b[:, :, :9].view(torch.int16))


STUBS = """
#include <unistd.h>
extern "C" {
volatile int go = 0, calls = 0, late = 0;
int waits() {  // until `go` is set, at most 3 s
  for (int i = 0; i < 3000 && !go; ++i) usleep(1000);
  late = !go;
  return 0;
}
int fails() { return ++calls, -4; }  // KVQ_ERR_HIP
size_t bytes() { return 256; }
}
"""


@pytest.fixture
def stubs(tmp_path):
    (tmp_path / "stubs.cpp").write_text(STUBS)
    subprocess.run(["g++", "-shared", "-fPIC", str(tmp_path / "stubs.cpp"), "-o", str(tmp_path / "stubs.so")], check=True)
    lib = ctypes.CDLL(str(tmp_path / "stubs.so"))
    lib.addr = lambda name: ctypes.cast(getattr(lib, name), ctypes.c_void_p).value
    lib.get = lambda name: ctypes.c_int.in_dll(lib, name)
    return lib


def test_other_threads_run_during_a_call(stubs):
    """A launch that waits (a full queue) does not hold the interpreter lock: here it waits for another thread."""
    kt, vt = make_cache(1, 2, 64, 128, 8, torch.float16, 5600)
    k = seeded_normal((1, 2, 1, 128), 5601, torch.float16, DEV)
    call = kernels.prepare_append(kt, vt)
    call._state.fn = stubs.addr("waits")
    threading.Timer(0.05, lambda: setattr(stubs.get("go"), "value", 1)).start()
    call(k, k, 0)
    assert stubs.get("late").value == 0


def test_a_failed_launch_raises_and_is_not_tried_again(stubs):
    kt, vt = make_cache(1, 2, 64, 128, 8, torch.float16, 5700)
    k = seeded_normal((1, 2, 1, 128), 5701, torch.float16, DEV)
    call = kernels.prepare_append(kt, vt)
    call._state.fn = stubs.addr("fails")
    with pytest.raises(RuntimeError, match="status -4"):
        call(k, k, 0)
    assert stubs.get("calls").value == 1
    h = _lib.host()
    try:
        _lib.bind_host(h, *(stubs.addr(n) for n in ("fails", "fails", "bytes", "bytes")))
        with pytest.raises(RuntimeError, match="status -4"):
            A.blocked_quantized_sdpa(k, kt, vt, 0.1, None)
    finally:
        _lib._host = None
        _lib.host()
    assert stubs.get("calls").value == 2
    A.blocked_quantized_sdpa(k, kt, vt, 0.1, None)
