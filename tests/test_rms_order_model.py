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


def _then(f, g):
    """Two runs one after the other (cx_rms_then): (d0, d1, q) arrays"""
    (f0, f1, fq), (g0, g1, gq) = f, g
    p0, p1 = fq & 1, (fq >> 1) & 1
    return (f0 + np.where(p0, g1, g0), f1 + np.where(p1, g1, g0),
            ((gq >> p0) & 1) | (((gq >> p1) & 1) << 1))


def _from(r, src, has):
    """The run of lane `src` where `has`, else the one that adds nothing"""
    return tuple(np.where(has, v[src], none) for v, none in zip(r, (0.0, 0.0, 2)))


def _wave_scan(r):
    """The 64 lanes' inclusive scan: row shifts by 1, 2, 4, 8, then each odd row of
    16 after the row before it, then rows 2 and 3 after lane 31"""
    lane = np.arange(64)
    for n in (1, 2, 4, 8):
        r = _then(_from(r, np.maximum(lane - n, 0), lane % 16 >= n), r)
    r = _then(_from(r, np.maximum(lane // 16 * 16 - 1, 0), lane // 16 % 2 == 1), r)
    return _then(_from(r, np.full(64, 31), lane >= 32), r)


def _wg_sum_scanned(x):
    """_wg_sum with the runs composed as the lanes and waves compose them"""
    n = x.size
    t = x.astype(np.float64) ** 2
    s = np.float64(seq_sum(x[:HEAD]))
    b = min(n, HEAD)
    while b < n:
        per = 4 * min(4, (n - b + 1023) // 1024)
        v = np.zeros(256 * per)
        v[:min(n - b, 256 * per)] = t[b:b + 256 * per]
        v = v.reshape(256, per)
        frm = 0
        while frm < 256:
            e = _bits(s) & np.uint64(0x7FF0000000000000)
            lo = e.view(np.float64)
            lo1 = (e | np.uint64(1)).view(np.float64) if s > 0 else np.float64(0)
            a0, a1 = np.full(256, lo), np.full(256, lo1)
            for j in range(per):
                a0, a1 = a0 + v[:, j], a1 + v[:, j]
            d0, d1 = a0 - lo, a1 - lo1
            q = (_bits(a0) & np.uint64(1)).astype(int) | (_bits(a1) & np.uint64(1)).astype(int) << 1
            d0[:frm], d1[:frm], q[:frm] = 0.0, 0.0, 2
            waves = [_wave_scan((d0[w:w + 64], d1[w:w + 64], q[w:w + 64])) for w in range(0, 256, 64)]
            p = int(_bits(s) & np.uint64(1))
            ends = []  # each wave's sum after its first thread that leaves, and that thread
            for w in range(4):
                f = (np.zeros(1), np.zeros(1), np.full(1, 2))
                for u in range(w):
                    f = _then(f, tuple(c[63:] for c in waves[u]))
                r = _then(tuple(np.repeat(c, 64) for c in f), waves[w])
                after = s + r[p]
                before = np.concatenate([s + f[p], after[:-1]])
                out = np.flatnonzero(after >= lo + lo if s > 0 else after > 0)
                if out.size:
                    a = before[out[0]]
                    for y in v[64 * w + out[0]]:
                        a = a + y
                    ends.append((a, 64 * w + out[0]))
                else:
                    ends.append((after[63], 256))
            s, frm = next((e for e in ends if e[1] < 256), ends[3])
            frm += 1
        b += 256 * per
    return s


@pytest.mark.parametrize("n", [1028, 1152, 2048, 4096, 4228, 11008])
def test_the_scans_composition_is_the_sum_in_order(n):
    for i, x in enumerate(_vectors(n)):
        x = x.astype(np.float32)
        assert float(_wg_sum_scanned(x)) == seq_sum(x), (n, i)
