"""The host side of the attention of many query tokens (cx_attn_many.hip), without
a GPU: what its launch refuses before any kernel runs."""
import ctypes as C
import re
import subprocess

import pytest


@pytest.fixture(scope="module")
def L():
    from cosxamix_amd import _lib
    _lib.load()
    return _lib


def internal(L, name):
    """The library's C++ function `name` (internal: not in the C ABI's header)."""
    out = subprocess.run(["nm", "-D", "--defined-only", L.LIB_PATH], capture_output=True, text=True,
                         check=True).stdout
    found = re.findall(rf"\sT\s(_Z{len(name)}{name}\w*)", out)
    assert len(found) == 1, found
    return getattr(L.load(), found[0])


class Args(C.Structure):  # cx_attn_many_args
    _fields_ = ([(n, C.c_void_p) for n in "qkv"] +
                [(n, C.c_uint32) for n in ("tokens", "pos", "heads", "kvh", "hd")] +
                [(n, C.c_void_p) for n in ("sc", "cm", "inv", "out")])


@pytest.mark.parametrize("which", ["q", "k", "v", "out"])
def test_a_misaligned_tensor_is_refused_before_any_launch(L, which):
    # 16-byte loads of q, k and v and stores of out
    launch = internal(L, "cx_launch_attn_many")
    launch.restype = C.c_int
    a = Args(q=1 << 20, k=2 << 20, v=3 << 20, tokens=64, pos=0, heads=4, kvh=2, hd=64, sc=4 << 20,
             cm=5 << 20, inv=6 << 20, out=7 << 20)
    setattr(a, which, getattr(a, which) + 4)
    assert launch(C.byref(a), None) == L.CX_EINVAL
    assert b"aligned" in L.load().cx_last_error()
