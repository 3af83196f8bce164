"""CPU check of the direct schedule's plans (direct.hip.h, compiled by g++): run over Fr scalars,
every plan computes the transform it stands for, with all positions in range and every product
reached by a wave.
"""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import oracle as O

R = O.R_MOD
W512 = pow(5, (R - 1) // 512, R)
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
IFFT_HALF, FFT_HALF, FFT, IFFT = range(4)
NONE = 0xFFFFFFFF


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("direct") / "libdirect_host.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-o", out,
                    os.path.join(ROOT, "tests", "native", "direct_host.cpp")], check=True)
    L = ctypes.CDLL(out)
    n = L.direct_host_build()
    L.direct_host_words.restype = ctypes.POINTER(ctypes.c_uint32)
    words = [int(x) for x in np.ctypeslib.as_array(L.direct_host_words(), shape=(n,))]
    return L, words


def rev(i, bits):
    return int(format(i, "0%db" % bits)[::-1], 2)


def step(words, at, logn, D):
    """One step over Fr as the three kernels run it, in place on the list D."""
    n = 1 << logn
    loga, logb, logblocks, in_map, log_lanes, sum_words, nprod, prod, nout, sums = words[at:at + 10]
    nwaves, waves = words[at + 10:at + 17], words[at + 17:at + 24]
    a, b, lanes = 1 << loga, 1 << logb, 1 << log_lanes
    assert loga + logb + logblocks == logn and 4 <= a <= n
    for g in range(n // a):  # the passes of a radix above 32 together
        idx = [((g >> logb) << (loga + logb)) + (g & (b - 1)) + (t << logb) for t in range(a)]
        pos = [rev(i, logn) if in_map & 1 else i for i in idx]
        x = [0 if in_map & 2 and i >= n // 2 else D[p] for i, p in zip(idx, pos)]
        h = a // 2
        while h:
            x = [x[t] + x[t + h] if t < h else x[t - h] - x[t] if t < 2 * h else x[t] for t in range(a)]
            h //= 2
        for p, v in zip(pos, x):
            D[p] = v % R
    P = []
    last = None
    seen = set()
    for k in range(nprod):
        w = words[prod + k]
        p, e = w & 0xFFFF, w >> 16
        assert p < n and e < 256
        if e != last:
            assert e not in seen  # products of one exponent are next to each other
            seen.add(e)
            last = e
        P.append(D[p] * pow(W512, e, R) % R)
    for lk in range(7):
        covered = []
        for w in words[waves[lk]:waves[lk] + nwaves[lk]]:
            first, count = w & 0xFFFF, w >> 16
            assert 1 <= count <= 1 << lk
            assert len({words[prod + s] >> 16 for s in range(first, first + count)}) == 1
            covered += range(first, first + count)
        assert covered == list(range(nprod))
    out = {}
    for k in range(nout):
        o = words[sums + sum_words * k:sums + sum_words * (k + 1)]
        assert (len(o) - 4) % lanes == 0
        acc, ended = 0, False
        for t in o[4:]:
            if t == NONE:
                ended = True
                continue
            assert not ended and (t & 0x7FFFFFFF) < nprod
            acc += -P[t & 0x7FFFFFFF] if t >> 31 else P[t & 0x7FFFFFFF]
        assert o[0] < n and o[0] not in out
        out[o[0]] = acc % R
    for p, v in out.items():
        D[p] = v


def run(plans, logn, kind, levels, D):
    L, words = plans
    for s in range(levels):
        step(words, L.direct_host_record(logn, kind, levels, s), logn, D)


def dft(x, sign):
    n = len(x)
    w = pow(W512, sign * (512 // n), R)
    pw = [pow(w, i, R) for i in range(n)]
    return [sum(v * pw[i * k % n] for i, v in enumerate(x)) % R for k in range(n)]


@pytest.mark.parametrize("levels", [1, 2, 3])
@pytest.mark.parametrize("logn", [7, 8, 9])
def test_plans_compute_the_transforms(plans, logn, levels):
    n = 1 << logn
    rng = np.random.default_rng(logn * 10 + levels)
    x = [int.from_bytes(rng.bytes(32), "little") % R for _ in range(n)]
    junk = [int.from_bytes(rng.bytes(32), "little") % R for _ in range(n)]
    fwd, inv = dft(x, 1), dft(x, -1)
    D = list(x)
    run(plans, logn, FFT, levels, D)
    assert [D[rev(k, logn)] for k in range(n)] == fwd
    D = [x[rev(p, logn)] for p in range(n)]
    run(plans, logn, IFFT, levels, D)
    assert D == inv
    # hext_fft -> h -> h_fft: the half inverse, then the forward transform of its n/2 outputs
    D = [x[rev(p, logn)] for p in range(n)]
    run(plans, logn, IFFT_HALF, levels, D)
    assert D[:n // 2] == inv[:n // 2]
    D[n // 2:] = junk[n // 2:]  # the upper half is not read
    run(plans, logn, FFT_HALF, levels, D)
    want = dft(inv[:n // 2] + [0] * (n // 2), 1)
    assert [D[rev(k, logn)] for k in range(n)] == want


def test_row_lanes(plans):
    L, _ = plans
    for rows in range(1, 200):
        lr = L.direct_host_row_lanes(rows)
        assert lr == min(6, (rows - 1).bit_length())


@pytest.mark.parametrize("max_lr", [5, 6])  # two lanes per ladder, one
def test_waves_cover_rows_and_products(plans, max_lr):
    """Every (product, row) once or more, every wave's lanes on one exponent, nothing else."""
    L, words = plans
    buf = (ctypes.c_uint32 * 128)()
    for logn, levels in ((7, 2), (8, 3), (9, 2)):
        rec = L.direct_host_record(logn, FFT, levels, levels - 1)
        nprod, prod = words[rec + 6], words[rec + 7]
        for rows in (1, 2, 3, 7, 13, 31, 32, 33, 37, 48, 63, 64, 65, 100, 127, 128, 200, 256):
            seen = set()
            n = L.direct_host_waves(rec, rows, max_lr)
            for local in range(n):
                L.direct_host_wave(rec, rows, max_lr, local, buf)
                lanes = {(buf[2 * p], buf[2 * p + 1]) for p in range(1 << max_lr)}
                assert len({words[prod + s] >> 16 for _, s in lanes}) == 1
                seen |= lanes
            assert seen == {(r, s) for r in range(rows) for s in range(nprod)}
