"""The contraction with weights in registers (ops.matmul_auto, many rows) bit for
bit against the oracle's per-row matmul at the edges of its tiles: rows of the
weights and of the activations at and beside multiples of 16, 32 and 64, one to
three super-blocks (first stage, both halves of the buffer), every tile height; and
blocks whose scale is infinite or NaN beside finite ones."""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu

D = {O.Q4_K: (0, 2), O.Q5_K: (0, 2)}  # f16 scales: their byte offsets in a block
BPB = {O.Q4_K: 144, O.Q5_K: 176}


def blocks(t, n, k, seed, wild=False):
    """n rows of random block bytes with small scales; wild: some infinite or NaN"""
    r = np.random.default_rng(seed)
    b = r.integers(0, 256, (n, k // 256, BPB[t]), dtype=np.uint8)
    for off in D[t]:
        d = (r.normal(0, 1, b.shape[:2]) * 0.01).astype(np.float16)
        if wild:
            d[r.random(d.shape) < 0.02] = np.inf
            d[r.random(d.shape) < 0.02] = -np.inf
            d[r.random(d.shape) < 0.02] = np.nan
        b[..., off:off + 2] = d[..., None].view(np.uint8)
    return b.reshape(n, -1)


def check(dev, t, n, k, m, wild=False):
    from cosxamix_amd import ops
    w = blocks(t, n, k, n + m, wild)
    x = np.random.default_rng(m).normal(0, 1, (m, k)).astype(np.float32)
    x[0, :32] = 0.0
    out = torch.full((m, n), 7.0, dtype=torch.float32, device=dev)
    ops.matmul_auto((m, k, n), torch.from_numpy(x).to(dev), torch.from_numpy(w).to(dev), t, out)
    got, want = out.cpu().numpy(), O.matmul_fused(t, x, w, n, threads=16)
    ok = (got.view(np.uint32) == want.view(np.uint32)) | (np.isnan(got) & np.isnan(want))
    assert ok.all(), np.argwhere(~ok)[:5]


@pytest.mark.parametrize("t", D, ids=[O.NAMES[t] for t in D])
@pytest.mark.parametrize("n,k,m", [
    (4096, 256, 17), (4097, 512, 33), (4159, 768, 129),   # 64 x 16
    (4096, 256, 131), (4161, 512, 161), (4223, 768, 255),  # 64 x 32
    (4096, 256, 433), (4097, 768, 449), (10001, 512, 193),  # 64 x 64
    (2048, 256, 511), (2111, 512, 500), (3073, 256, 963)])  # few weight rows
def test_tiles_bit_exact(dev, t, n, k, m):
    check(dev, t, n, k, m)


@pytest.mark.parametrize("t", D, ids=[O.NAMES[t] for t in D])
@pytest.mark.parametrize("n,k,m", [(4100, 512, 40), (4100, 512, 150), (4100, 512, 450)])
def test_scales_that_are_not_finite(dev, t, n, k, m):
    check(dev, t, n, k, m, wild=True)
