"""The in-order f64 sum of squares as a workgroup forms it
(cx_rms_seq_sum_wg, cosxamix_amd/csrc/cx_act.h), modelled on the CPU step by
step and compared with the plain loop bit for bit: runs of values as a pair of
additions (one for each last bit of the incoming sum), composed over the
threads, restarted where the sum leaves its binade."""
import numpy as np
import pytest

from rms_fixtures import seq_sum

HEAD = 128


def _bits(v):
    return np.asarray(v, np.float64).view(np.uint64)


def _wg_sum(x):
    n = x.size
    t = x.astype(np.float64) ** 2
    s = np.float64(seq_sum(x[:HEAD]))
    b, rounds = min(n, HEAD), 0
    while b < n:
        per = 4 * min(4, (n - b + 1023) // 1024)
        v = np.zeros(256 * per)
        v[:min(n - b, 256 * per)] = t[b:b + 256 * per]
        v = v.reshape(256, per)
        frm = 0
        while frm < 256:
            rounds += 1
            e = _bits(s) & np.uint64(0x7FF0000000000000)
            lo = e.view(np.float64)
            lo1 = (e | np.uint64(1)).view(np.float64) if s > 0 else np.float64(0)
            a = np.stack([np.full(256, lo), np.full(256, lo1)])
            for j in range(per):
                a = a + v[:, j]
            d = a - np.array([[lo], [lo1]])
            q = (_bits(a) & np.uint64(1)).astype(int)
            d[:, :frm], q[0, :frm], q[1, :frm] = 0.0, 0, 1
            run_d, run_p, p0 = np.float64(0), int(_bits(s) & np.uint64(1)), None
            at = 256
            for k in range(256):
                before = s + run_d
                run_d, run_p = run_d + d[run_p, k], q[run_p, k]
                after = s + run_d
                if (after >= lo + lo) if s > 0 else after > 0:
                    at = k
                    break
            if at < 256:
                for w in v[at]:
                    before = before + w
                s = before
            else:
                s = after
            frm = at + 1
        b += 256 * per
    return s, rounds


def _vectors(n):
    r = np.random.default_rng(n)
    yield r.normal(0, 1, n)
    yield np.exp(r.normal(0, 6, n)) * r.choice([-1, 1], n)  # a few terms carry the sum
    yield r.integers(1, 1 << 24, n) * 2.0 ** -12  # 48-bit squares
    yield (1 + r.integers(0, 2, n) * 2.0 ** -23) * 2.0 ** r.integers(-3, 4, n)
    x = r.choice([1.0, 2.0 ** -26, 3 * 2.0 ** -27, 2.0 ** -27], n)  # halfway cases
    x[0] = 1.0
    yield x
    yield np.concatenate([np.zeros(n // 2), r.normal(0, 1, n - n // 2)])  # the sum starts late
    yield np.zeros(n)
    x = np.zeros(n)
    x[-1] = 1e-30
    yield x
    yield np.sort(np.exp(r.normal(0, 10, n)))  # the binade changes all along
    yield np.full(n, 1e19)


@pytest.mark.parametrize("n", [4, 124, 128, 132, 896, 1152, 1156, 2048, 4096, 4224, 4228, 11008])
def test_the_workgroup_sum_is_the_sum_in_order(n):
    for i, x in enumerate(_vectors(n)):
        x = x.astype(np.float32)
        got, _ = _wg_sum(x)
        assert float(got) == seq_sum(x), (n, i)
