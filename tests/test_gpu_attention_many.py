"""Attention of many query tokens (cx_attn_many.hip) through ops.atencion, bit
for bit against the oracle's ops::atencion (src/ops.rs:1258-1325), at the edges of
its tiles: rows (tokens x heads per group) around 64 and 128, positions around 32,
64 and 128, one to sixteen heads per group, both head dims, every score tile and
every row count a lane takes, and calls of several slabs. Values that a row does
not see may be anything; a captured call and misaligned tensors take the general
kernel; the scores' buffer is no captured graph's."""
import ctypes as C

import numpy as np
import pytest
import torch

from oracle import oracle as O
from test_attention_many_plan import internal

pytestmark = pytest.mark.gpu


def inputs(seed, tokens, total, heads, kv, hd):
    r = np.random.default_rng(seed)
    return (r.normal(0, 1, (tokens, heads * hd)).astype(np.float32),
            r.normal(0, 1, (total, kv * hd)).astype(np.float32),
            r.normal(0, 1, (total, kv * hd)).astype(np.float32))


def run(dev, q, k, v, heads, kv, hd):
    from cosxamix_amd import ops
    out = torch.full(q.shape, 7.0, dtype=torch.float32, device=dev)
    ops.atencion(torch.from_numpy(q).to(dev), torch.from_numpy(k).to(dev),
                 torch.from_numpy(v).to(dev), (len(q), len(k), heads, kv, hd), out)
    return out.cpu().numpy()


def same(got, want):  # equal bits; a NaN equals a NaN
    got, want = got.reshape(-1), np.asarray(want, np.float32).reshape(-1)
    return np.all((got.view(np.uint32) == want.view(np.uint32)) |
                  (np.isnan(got) & np.isnan(want)))


def oracle(q, k, v, heads, kv, hd):
    return O.attention(q.reshape(-1), k.reshape(-1), v.reshape(-1), len(q), len(k), heads, kv, hd)


@pytest.mark.parametrize("tokens,total,heads,kv,hd", [
    (1, 1024, 4, 4, 64), (2, 1025, 3, 1, 128), (63, 1151, 2, 2, 64), (64, 1024, 1, 1, 128),
    (65, 1153, 7, 1, 64), (8, 1087, 16, 2, 128), (9, 1089, 32, 2, 64), (300, 300, 14, 2, 64),
    (257, 511, 16, 2, 128), (129, 1500, 8, 8, 128), (1100, 1100, 4, 1, 64)])
def test_many_tokens_bit_exact(dev, tokens, total, heads, kv, hd):
    q, k, v = inputs(tokens * 7 + total, tokens, total, heads, kv, hd)
    assert same(run(dev, q, k, v, heads, kv, hd), oracle(q, k, v, heads, kv, hd))


def tile_and_rows(tokens, total, heads, kv, hd):
    """The launch's choice (cx_attn_many.hip): score tile, P.V rows a lane"""
    rows = tokens * (heads // kv)
    tile = 128 if -(-rows // 128) * -(-total // 128) * kv >= 1024 else 64
    one = -(-rows // (1024 // hd)) * kv  # workgroups of one row a lane
    return tile, 4 if one // 4 >= 512 else 2 if one // 2 >= 256 else 1


# every score tile and P.V row count of both head dims that the sizes above (64 x
# 64 tiles, one row a lane at head_dim 64) leave out: the first and last tokens
# against the oracle (each is the last token of its own prefix), and those beside
# the edges of tiles
@pytest.mark.parametrize("tokens,total,heads,kv,hd,tile,rows", [
    (512, 1030, 32, 8, 128, 128, 4), (512, 600, 32, 8, 128, 64, 4), (300, 1100, 16, 2, 128, 64, 2),
    (300, 4200, 16, 2, 128, 128, 2), (130, 8300, 8, 8, 128, 128, 1),
    (1200, 1200, 14, 2, 64, 128, 2), (2600, 2600, 14, 2, 64, 128, 4),
    (700, 1100, 14, 2, 64, 64, 2), (512, 5000, 14, 2, 64, 128, 1)])
def test_large_tiles_bit_exact(dev, tokens, total, heads, kv, hd, tile, rows):
    assert tile_and_rows(tokens, total, heads, kv, hd) == (tile, rows)
    q, k, v = inputs(5, tokens, total, heads, kv, hd)
    got = run(dev, q, k, v, heads, kv, hd)
    for t in (0, 1, 31, 32, tokens // 2 + 7, tokens - 2, tokens - 1):
        n = total - tokens + t + 1
        assert same(got[t], oracle(q[t:t + 1], k[:n], v[:n], heads, kv, hd)), t


# Calls whose scores are more than the buffer holds (256 MB): tokens a slab, by
# cx_attn_many_slab. The first and last tokens of every slab against the oracle.
@pytest.mark.parametrize("tokens,total,heads,kv,hd,slab", [
    (512, 8192, 32, 8, 128, 192),  # three slabs, the last of 128
    (700, 12000, 14, 2, 64, 384),  # two
    (70, 16000, 128, 8, 64, 32),   # below 64 tokens a slab; the last of 6
    (3, 9000, 128, 128, 64, 3)])   # one tile of each group alone is more: all at once
def test_slabs_bit_exact(dev, tokens, total, heads, kv, hd, slab):
    from cosxamix_amd import _lib as L
    plan = internal(L, "cx_attn_many_slab")
    plan.restype, plan.argtypes = C.c_size_t, [C.c_size_t] * 4
    assert plan(tokens, total, heads, kv) == slab
    q, k, v = inputs(tokens + total, tokens, total, heads, kv, hd)
    got = run(dev, q, k, v, heads, kv, hd)
    edges = {t + d for t in range(0, tokens + 1, slab) for d in (-1, 0)} | {tokens - 1}
    for t in sorted(e for e in edges if 0 <= e < tokens):
        n = total - tokens + t + 1
        assert same(got[t], oracle(q[t:t + 1], k[:n], v[:n], heads, kv, hd)), t


@pytest.mark.parametrize("tokens", [40, 300])
def test_special_values(dev, tokens):
    # inf and NaN where rows do not see them, a NaN key, an infinite query
    # (its maximum is not finite), equal keys, scores down to exp's underflow
    total, heads, kv, hd = 1100, 4, 2, 64
    q, k, v = inputs(11, tokens, total, heads, kv, hd)
    v[total - 1, 3] = np.inf
    v[total - 2, 5] = np.nan
    v[total - 5, 7] = -np.inf
    k[total - 3] = np.nan
    q[1] = np.inf
    q[2] *= 60.0
    k[100:164] = k[100]
    assert same(run(dev, q, k, v, heads, kv, hd), oracle(q, k, v, heads, kv, hd))


def test_capture_and_misaligned_rows_take_the_general_kernel(dev):
    from cosxamix_amd import ops
    tokens, total, heads, kv, hd = 70, 1040, 4, 2, 64
    q, k, v = inputs(3, tokens, total, heads, kv, hd)
    want = oracle(q, k, v, heads, kv, hd)
    qd, kd, vd = (torch.from_numpy(t).to(dev) for t in (q, k, v))
    out = torch.zeros_like(qd)
    forma = (tokens, total, heads, kv, hd)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        ops.atencion(qd, kd, vd, forma, out)
    for _ in range(3):
        out.fill_(7.0)
        g.replay()
        assert same(out.cpu().numpy(), want)
    flat = torch.empty(q.size + 1, device=dev)
    flat[1:] = qd.reshape(-1)
    out.fill_(7.0)
    ops.atencion(flat[1:].reshape(q.shape), kd, vd, forma, out)  # 4-byte aligned
    assert same(out.cpu().numpy(), want)


@pytest.mark.parametrize("which", ["k", "v", "out"])
def test_a_misaligned_tensor_takes_the_general_kernel(dev, which):
    # the kernels of many tokens read q, k and v and write out 16 bytes at a
    # time; a view at any float is an operand like any other
    from cosxamix_amd import ops
    tokens, total, heads, kv, hd = 70, 1040, 4, 2, 64
    q, k, v = inputs(3, tokens, total, heads, kv, hd)
    t = dict(q=torch.from_numpy(q).to(dev), k=torch.from_numpy(k).to(dev),
             v=torch.from_numpy(v).to(dev), out=torch.full(q.shape, 7.0, device=dev))
    flat = torch.full((t[which].numel() + 8,), 7.0, device=dev)
    flat[1:1 + t[which].numel()] = t[which].reshape(-1)
    t[which] = flat[1:1 + t[which].numel()].reshape(t[which].shape)
    assert t[which].data_ptr() % 16 == 4
    ops.atencion(t["q"], t["k"], t["v"], (tokens, total, heads, kv, hd), t["out"])
    assert same(t["out"].cpu().numpy(), oracle(q, k, v, heads, kv, hd))
    if which == "out":  # nothing beside it written
        assert torch.all(flat[:1] == 7.0) and torch.all(flat[1 + q.size:] == 7.0)


def test_attention_leaves_a_captured_graphs_scratch_alone(dev):
    # a graph holds the address of the scratch it was captured with: attention
    # between its replays neither grows that scratch nor writes to it
    from cosxamix_amd import ops
    m, n, k = 8, 64, 256
    w = torch.from_numpy(O.daiss_matrix(3, "w", n, k, 0.02, O.Q4_K)).to(dev)
    x = torch.randn(m, k, generator=torch.Generator().manual_seed(1)).to(dev)
    y = torch.zeros(m, n, device=dev)
    ops.matmul_auto((m, k, n), x, w, O.Q4_K, y)  # the scratch has its size
    want = y.clone()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        ops.matmul_auto((m, k, n), x, w, O.Q4_K, y)
    q, kk, v = inputs(4, 300, 2000, 16, 2, 128)  # ~37 MB of scores
    qd, kd, vd = (torch.from_numpy(t).to(dev) for t in (q, kk, v))
    first, again = torch.zeros_like(qd), torch.zeros_like(qd)
    side = torch.cuda.Stream()
    ops.atencion(qd, kd, vd, (300, 2000, 16, 2, 128), first)
    for _ in range(4):
        y.zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(side):  # beside the graph
            ops.atencion(qd, kd, vd, (300, 2000, 16, 2, 128), again)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y.view(torch.int32), want.view(torch.int32))
        assert torch.equal(again.view(torch.int32), first.view(torch.int32))


@pytest.mark.skipif(torch.cuda.device_count() < 2, reason="needs a second GPU")
def test_another_devices_stream_takes_the_general_kernel(dev):
    # the thread's context is on device 0; the call's tensors and stream on 1
    from cosxamix_amd import ops
    tokens, total, heads, kv, hd = 70, 1040, 4, 2, 64
    q, k, v = inputs(3, tokens, total, heads, kv, hd)
    with torch.cuda.device(1):
        out = torch.full(q.shape, 7.0, dtype=torch.float32, device="cuda:1")
        ops.atencion(*(torch.from_numpy(t).to("cuda:1") for t in (q, k, v)),
                     (tokens, total, heads, kv, hd), out)
        assert torch.cuda.current_device() == 1
        assert same(out.cpu().numpy(), oracle(q, k, v, heads, kv, hd))
