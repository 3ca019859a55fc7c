"""The native path's cache views on the CPU: the slices Python would take, and what it hands back."""

import struct

import pytest
import torch

from myinfer_amd import _lib
from myinfer_amd.cache import QuantizedKVCache


def test_views_are_slices():
    h = _lib.host()
    tr = tuple(torch.arange(2 * 3 * 8 * w).view(2, 3, 8, w) for w in (4, 2, 2))
    for n in (0, 1, 5, 8):
        both = h.views(tr, tr, n)
        assert type(both) is tuple and len(both) == 2
        for got in both:
            for a, b in zip(got, tr):
                s = b[..., :n, :]
                assert torch.equal(a, s) and a.stride() == s.stride() and a.storage_offset() == s.storage_offset()
    both = h.views(tr, tr, 3)
    both[0][0].fill_(-1)  # a view, not a copy
    assert bool((tr[0][..., :3, :] == -1).all())


def test_handed_back():
    h = _lib.host()
    tr = tuple(torch.zeros(1, 1, 4, 2) for _ in range(3))
    assert h.views(list(tr), tr, 2) is None and h.views(tr, tr[:2], 2) is None
    assert h.views(tr, tr, 5) is None and h.views(tr, tr, -1) is None
    assert h.attention(tr[0], tr, tr, 0.1, 0, 0, None, 64, 8, 0, 0, 0, None, 0) is None  # CPU tensors
    assert h.append(0, tr[0], tr[0], 0, 0) is None


def test_another_build_is_refused(monkeypatch):
    h = _lib.host()
    for name, value in (("ABI_VERSION", _lib.ABI_VERSION + 1), ("AppendState", _lib.Rows)):
        with monkeypatch.context() as m:
            m.setattr(_lib, name, value)
            with pytest.raises(ImportError, match="rebuild"):
                _lib.bind_host(h, 0, 0, 0, 0)
    for version in ("2.1.0", "", torch.__version__.split("+")[0] + "1"):
        with monkeypatch.context() as m:
            m.setattr(torch, "__version__", version)
            with pytest.raises(ImportError, match="rebuild"):
                _lib.bind_host(h, 0, 0, 0, 0)
    assert _lib.lib() and h.attention(None) is None  # (bound as before)


def test_views_of_a_restored_cache_need_no_library(monkeypatch):
    def missing(*_):
        raise ImportError("no library")

    monkeypatch.setattr(_lib, "_host", None)
    monkeypatch.setattr(_lib, "lib", missing)
    c = QuantizedKVCache(group_size=64, bits=8)
    c.keys = c.values = tuple(torch.arange(2 * 8 * w).view(1, 2, 8, w) for w in (4, 2, 2))
    c.offset = 5
    for tr in c.fetch():
        assert all(torch.equal(a, b[..., :5, :]) for a, b in zip(tr, c.keys))


def test_module_has_no_thread_local_storage():
    """Loaded after torch, a library with a TLS segment slows every thread's access to tensors (see _build.py)."""
    _lib.host()
    elf = (_lib.LIB_PATH.parent / "_kvqhost.so").read_bytes()
    at, size, count = struct.unpack_from("<Q", elf, 32)[0], *struct.unpack_from("<HH", elf, 54)
    kinds = [struct.unpack_from("<I", elf, at + i * size)[0] for i in range(count)]
    assert 1 in kinds and 7 not in kinds  # PT_LOAD, PT_TLS
