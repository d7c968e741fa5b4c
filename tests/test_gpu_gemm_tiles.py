"""The contraction with weights in registers (ops.matmul_auto, many rows) bit for
bit against the oracle's per-row matmul at the edges of its tiles: rows of the
weights and of the activations at and beside multiples of 16, 32 and 64, one to
three super-blocks (first stage, both halves of the buffer) and widths that end
inside one for the 32-value blocks, every tile height; blocks whose scale is infinite
or NaN beside finite ones; and rows at an address that is only even."""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu

# f16 scales: their byte offsets in a block
D = {O.Q4_K: (0, 2), O.Q5_K: (0, 2), O.Q2_K: (80, 82), O.Q3_K: (108,), O.Q6_K: (208,),
     O.Q8_0: (0,), O.Q5_0: (0,)}
BPB = {O.Q4_K: 144, O.Q5_K: 176, O.Q2_K: 84, O.Q3_K: 110, O.Q6_K: 210, O.Q8_0: 34, O.Q5_0: 22}
REG = [O.Q4_K, O.Q5_K]
B32 = [O.Q8_0, O.Q5_0]
ANY = [O.Q2_K, O.Q3_K, O.Q6_K] + B32


def blocks(t, n, k, seed, wild=False):
    """n rows of random block bytes with small scales; wild: some infinite or NaN"""
    r = np.random.default_rng(seed)
    b = r.integers(0, 256, (n, k // (32 if t in B32 else 256), BPB[t]), dtype=np.uint8)
    for off in D[t]:
        d = (r.normal(0, 1, b.shape[:2]) * 0.01).astype(np.float16)
        if wild:
            d[r.random(d.shape) < 0.02] = np.inf
            d[r.random(d.shape) < 0.02] = -np.inf
            d[r.random(d.shape) < 0.02] = np.nan
        b[..., off:off + 2] = d[..., None].view(np.uint8)
    return b.reshape(n, -1)


def check(dev, t, n, k, m, wild=False, shift=0):
    from cosxamix_amd import ops
    w = blocks(t, n, k, n + m, wild)
    room = torch.empty(w.size + shift, dtype=torch.uint8, device=dev)
    wd = room[shift:]  # at `shift` bytes past an aligned address
    wd.copy_(torch.from_numpy(w.reshape(-1)))
    x = np.random.default_rng(m).normal(0, 1, (m, k)).astype(np.float32)
    x[0, :32] = 0.0
    out = torch.full((m, n), 7.0, dtype=torch.float32, device=dev)
    ops.matmul_auto((m, k, n), torch.from_numpy(x).to(dev), wd, t, out)
    got = out.cpu().numpy()
    want = (O.matmul_direct if t in B32 else O.matmul_fused)(t, x, w, n, threads=16)
    ok = (got.view(np.uint32) == want.view(np.uint32)) | (np.isnan(got) & np.isnan(want))
    assert ok.all(), np.argwhere(~ok)[:5]


@pytest.mark.parametrize("t", REG, ids=str)
@pytest.mark.parametrize("n,k,m", [
    (4096, 256, 17), (4097, 512, 33), (4159, 768, 129),   # 64 x 16
    (8449, 256, 29), (9001, 512, 32),  # up to 32 rows past one round of those: k_gemm's 64 x 32
    (8449, 512, 61), (16400, 256, 19), (28225, 256, 32),  # past two, or 64 rows half empty: 64 x 32
    (4096, 256, 131), (4161, 512, 161), (4223, 768, 255),  # 64 x 32
    (4096, 256, 433), (4097, 768, 449), (10001, 512, 193),  # 64 x 64
    (2048, 256, 511), (2111, 512, 500), (3073, 256, 963)])  # few weight rows
def test_tiles_bit_exact(dev, t, n, k, m):
    check(dev, t, n, k, m)


@pytest.mark.parametrize("t", REG, ids=str)
@pytest.mark.parametrize("n,k,m", [(4100, 512, 40), (4100, 512, 150), (4100, 512, 450)])
def test_scales_that_are_not_finite(dev, t, n, k, m):
    check(dev, t, n, k, m, wild=True)


@pytest.mark.parametrize("t", ANY, ids=str)
@pytest.mark.parametrize("n,k,m", [
    (63, 256, 2), (64, 512, 16), (65, 768, 17), (2047, 256, 65),  # 64 x 16
    (5121, 256, 33), (2048, 768, 159), (2049, 512, 161),           # 64 x 32
    (4097, 768, 449), (2048, 256, 513), (10001, 512, 193)])         # 64 x 64
def test_any_offset_tiles_bit_exact(dev, t, n, k, m):
    check(dev, t, n, k, m, shift=2)


@pytest.mark.parametrize("t", B32, ids=str)
@pytest.mark.parametrize("k", [32, 64, 224, 288, 480, 736])
@pytest.mark.parametrize("n,m", [(65, 18), (2049, 161), (2048, 515)])
def test_widths_that_end_inside_a_stage(dev, t, k, n, m):
    check(dev, t, n, k, m, shift=2)


@pytest.mark.parametrize("t", ANY, ids=str)
@pytest.mark.parametrize("n,m", [(100, 9), (2049, 161), (4100, 450)])
def test_any_offset_scales_that_are_not_finite(dev, t, n, m):
    check(dev, t, n, 512, m, wild=True)


@pytest.mark.parametrize("base,down,out", [(O.Q8_0, O.Q8_0, O.Q8_0), (O.Q3_K, O.Q2_K, O.Q5_K),
                                           (O.Q2_K, O.Q3_K, O.Q4_K)])
def test_prefill_in_one_launch_equals_token_by_token(dev, base, down, out):
    # q/k/v and gate/up of one type in one launch, the adds in the epilogue
    from cosxamix_amd import forward as F
    c = F.Config(capas=2, dim=512, cabezas=8, cabezas_kv=2, ffn=1024, vocab=700, contexto=256,
                 eps=1e-5, rope=10_000.0)
    m = F.Modelo(c, tipo=base, semilla=3, tipo_down=down, tipo_salida=out)
    toks = np.random.default_rng(1).integers(0, 700, 67).astype(np.uint32)
    many, _ = m.forward(toks, m.nueva_cache(80))
    cache = m.nueva_cache(80)
    for t in toks:
        one, _ = m.forward(np.array([t], np.uint32), cache)
    assert np.array_equal(np.asarray(many).view(np.uint32), np.asarray(one).view(np.uint32))
    m.close()
