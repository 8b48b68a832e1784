"""The binding of the hot calls, as far as it shows without a GPU."""
import os
import re

SOURCE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "aitherkvcache_amd", "csrc", "akv_binding.cpp")


def test_tensors_are_read_under_the_interpreters_lock():
    """Between giving up the lock and taking it again stands the library's function alone, with arguments by value."""
    text = re.sub(r"//[^\n]*", "", open(SOURCE).read())
    blocks = re.findall(r"Py_BEGIN_ALLOW_THREADS;?(.*?)Py_END_ALLOW_THREADS", text, re.S)
    assert [b.strip() for b in blocks] == ["rc = f(args...);"]
    assert re.search(r"template <class F, class\.\.\. Args>\s*int without_gil\(F f, Args\.\.\. args\)", text)
    assert len(re.findall(r"without_gil\(g_lib\.", text)) == len(re.findall(r"guarded<\w+>, METH_FASTCALL", text)) == len(re.findall(r"METH_FASTCALL", text)) - 1
