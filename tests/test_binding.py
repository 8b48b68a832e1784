"""The binding of the hot calls, as far as it shows without a GPU."""
import os
import re
import sys
import types

import pytest
import torch

import aitherkvcache_amd
from aitherkvcache_amd import _lib
from aitherkvcache_amd.triattention import TriAttentionConfig
from aitherkvcache_amd.triattention.cache import SpectralKVCache

SOURCE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "aitherkvcache_amd", "csrc", "akv_binding.cpp")


def test_tensors_are_read_under_the_interpreters_lock():
    """Between giving up the lock and taking it again stands the library's function alone, with arguments by value."""
    text = re.sub(r"//[^\n]*", "", open(SOURCE).read())
    blocks = re.findall(r"Py_BEGIN_ALLOW_THREADS;?(.*?)Py_END_ALLOW_THREADS", text, re.S)
    assert [b.strip() for b in blocks] == ["rc = f(args...);"]
    assert re.search(r"template <class F, class\.\.\. Args>\s*int without_gil\(F f, Args\.\.\. args\)", text)
    assert len(re.findall(r"without_gil\(g_lib\.", text)) == len(re.findall(r"guarded<\w+>, METH_FASTCALL", text)) == len(re.findall(r"METH_FASTCALL", text)) - 1


@pytest.mark.parametrize("module", [None, types.SimpleNamespace(BUILT_FOR=("0.0.1", "3.10"))])
def test_without_a_binding_calls_go_the_long_way(monkeypatch, module):
    """A binding that is missing, or was built for another torch: a warning that names the make command, and the library works."""
    for name in ("_lib", "_calls"):
        monkeypatch.setattr(_lib, name, None)
    monkeypatch.setitem(sys.modules, "aitherkvcache_amd._binding", module)
    monkeypatch.delattr(aitherkvcache_amd, "_binding", raising=False)
    with pytest.warns(RuntimeWarning, match="make -C"):
        assert b"aitherkv" in _lib.lib().akv_version()
    assert _lib.calls().uniform_attention(1, 2, 3) is None


def test_without_a_library_a_call_is_checked_before_it_is_missed(monkeypatch):
    for name in ("_lib", "_calls"):
        monkeypatch.setattr(_lib, name, None)
    monkeypatch.setattr(_lib, "LIB_PATH", "/nonexistent/libaitherkv_hip.so")
    cache = SpectralKVCache(TriAttentionConfig(head_dim=64, num_freqs=8, coeff_bits=4, num_kv_heads=2, num_query_heads=4, block_size=16), max_blocks=2)
    x, slots = torch.zeros(3, 2, 64), torch.arange(3)
    with pytest.raises(ValueError, match="kv_heads"):
        cache.encode_and_store(x[:, :1], x[:, :1], slots)
    with pytest.raises(RuntimeError, match="HIP devices only"):
        cache.encode_and_store(x, x, slots)
