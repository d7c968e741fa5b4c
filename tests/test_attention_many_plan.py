"""The host side of the attention of many query tokens (cx_attn_many.hip), without
a GPU: what its launch refuses before any kernel runs, and how many tokens
cx_attention and a cache's prefill take at a time for the memory they state."""
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


class Floats(C.Structure):  # cx_attn_many_floats
    _fields_ = [(n, C.c_size_t) for n in ("sc", "cm", "inv")]


def test_a_slabs_scores_fit_the_memory_that_the_header_states(L):
    slab, scratch = internal(L, "cx_attn_many_slab"), internal(L, "cx_attn_many_scratch")
    slab.restype, slab.argtypes = C.c_size_t, [C.c_size_t] * 4
    scratch.restype, scratch.argtypes = Floats, [C.c_size_t] * 4

    def need(tokens, total, heads, kv):
        f = scratch(tokens, total, heads, kv)
        return (f.sc + f.cm + f.inv) * 4

    for heads, kv in ((1, 1), (7, 1), (14, 2), (16, 2), (32, 8), (64, 64), (128, 1), (128, 8),
                      (96, 32), (128, 128)):
        for total in (64, 1000, 1024, 2048, 4097, 8192, 12000, 16000):
            for tokens in (1, 2, 33, 63, 64, 65, 300, 512, 1999, total):
                if tokens > total:
                    continue
                n = slab(tokens, total, heads, kv)
                got = need(n, total, heads, kv)
                assert 1 <= n <= tokens
                assert got <= max(256 << 20, 260 * kv * total + 512 * kv), (tokens, total, heads, kv)
                # no smaller than it has to be: all the tokens where they fit, else
                # more than half of what would
                if need(tokens, total, heads, kv) <= 256 << 20:
                    assert n == tokens
                elif need(2 * n, total, heads, kv) <= 256 << 20:
                    assert 2 * n > tokens, (tokens, total, heads, kv, n)


class PrefillSize(C.Structure):  # cx_prefill_size
    _fields_ = [(n, C.c_size_t) for n in ("T", "sc", "cm", "inv")]


def test_a_prefills_scratch_fits_its_bound(L):
    plan, scratch, suits = (internal(L, n) for n in
                            ("cx_prefill_plan", "cx_attn_many_scratch", "cx_attn_many_suits_prefill"))
    plan.restype, plan.argtypes = PrefillSize, [C.c_size_t] * 6
    scratch.restype, scratch.argtypes = Floats, [C.c_size_t] * 4
    suits.restype, suits.argtypes = C.c_bool, [C.c_size_t] * 4
    for heads, kv, hd in ((4, 2, 64), (14, 2, 64), (16, 2, 128), (32, 8, 128), (32, 32, 128),
                          (64, 8, 128), (28, 4, 128), (40, 40, 64), (96, 96, 128)):
        for cap in (1, 7, 64, 600, 1023, 1024, 4096, 8704, 10001, 32768, 131072, 1 << 20):
            few = heads * ((cap + 3) // 4 * 4 + (cap + 63) // 64) * 4  # a token's bytes
            for max_t, bound in ((512, 640 << 20), (256, 256 << 20)):
                z = plan(heads, kv, hd, cap, max_t, bound)
                assert 1 <= z.T <= min(max_t, cap)
                assert (z.sc + z.cm) * 4 <= max(bound, 16 * few), (heads, kv, hd, cap, max_t)
                # no fewer tokens than their scores alone allow, but for whole tiles
                free = min(cap, max(16, min(max_t, bound // few // 16 * 16)))
                assert z.T == free or (z.inv and z.T >= max(64, free - 63)), (heads, kv, hd, cap)
                # the scratch of every chunk that takes the many-token kernels
                for nt in {1, 16, z.T // 2, z.T - 1, z.T} - {0}:
                    for total in {nt, min(cap, 1023), min(cap, 1024), cap}:
                        if total >= nt and z.inv and suits(nt, total, heads, hd):
                            f = scratch(nt, total, heads, kv)
                            assert z.inv >= f.inv and z.sc >= f.sc and z.cm >= f.cm
                if not suits(z.T, cap, heads, hd):  # no padding that nothing uses
                    assert z.inv == 0
                if not z.inv or z.T % 64 == 0:
                    assert (z.sc + z.cm) * 4 == z.T * few
                # given up only where no chunk that suits fits in whole tiles
                for t in range(64, z.T + 1, 16):
                    if not z.inv and suits(t, cap, heads, hd):
                        f = scratch(t, cap, heads, kv)
                        assert (f.sc + f.cm) * 4 > bound
