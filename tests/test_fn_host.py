"""CPU check of the transforms' Fr form (fr.hip.h fn_*), compiled by g++ from the source the kernels
inline, against Python integers, with digits at their extremes."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import oracle as O

R = O.R_MOD
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def L(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("fn") / "libfn_host.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-fsanitize=signed-integer-overflow",
                    "-fsanitize-undefined-trap-on-error", "-o", out,
                    os.path.join(ROOT, "tests", "native", "fn_host.cpp")], check=True)
    return ctypes.CDLL(out)


def call(f, n, dtype, *args):
    z = np.zeros(n, dtype=dtype)
    a = [np.asarray(x, dtype=t) for x, t in args]
    f(z.ctypes.data_as(ctypes.c_void_p), *[x.ctypes.data_as(ctypes.c_void_p) for x in a])
    return z


def val(d):
    return sum(int(x) << (29 * i) for i, x in enumerate(d))


def words(v):
    return [(v >> (32 * i)) & 0xFFFFFFFF for i in range(8)]


def test_products_norm_and_canonical_form(L):
    rng = np.random.default_rng(201)
    big, top = (1 << 31) - 1, (16 * R) >> (29 * 8)
    ops = [[s * big] * 8 + [t * top] for s in (1, -1) for t in (1, -1)]
    ops += [[int(x) for x in rng.choice([-big, big], 8)] + [int(rng.choice([-top, top]))] for _ in range(80)]
    ops += [[int(x) for x in rng.integers(-big, big, 8)] + [int(rng.integers(-top, top))] for _ in range(80)]
    edge = [0, 1, R - 1, R - 2, (R - 1) // 2, 2**254]
    ws = edge + [int.from_bytes(rng.bytes(32), "little") % R for _ in range(60)]
    for n, a in enumerate(ops):
        w = ws[n % len(ws)]
        wd = call(L.fn_host_from_words, 9, np.int32, (words(w), np.uint32))
        assert val(wd) == w and all(abs(int(x)) <= 1 << 28 for x in wd[:8])
        z = call(L.fn_host_mul, 9, np.int32, (a, np.int32), (wd, np.int32))
        v = val(z)
        assert v % R == val(a) * w * pow(2, -261, R) % R
        assert abs(v) <= abs(val(a) * w) // 2**261 + R + 1 and all(0 <= int(x) < 1 << 29 for x in z[:8])
        if -1.2 * R < v < 0.2 * R:
            got = call(L.fn_host_canon, 8, np.uint32, (z, np.int32))
            assert sum(int(x) << (32 * i) for i, x in enumerate(got)) == v % R
        y = call(L.fn_host_norm, 9, np.int32, (a, np.int32))
        assert val(y) == val(a) and all(abs(int(x)) <= (1 << 28) + 4 for x in y[:8])
    # canonical form of products at the ends of its range
    for v in (0, 1, -1, R // 8, -R, -R + 1, -R - 1, -R - R // 8, R // 6, -(R // 2)):
        d = [(v >> (29 * i)) & 0x1FFFFFFF for i in range(8)] + [v >> 232]
        got = call(L.fn_host_canon, 8, np.uint32, (d, np.int32))
        assert sum(int(x) << (32 * i) for i, x in enumerate(got)) == v % R
    for v in edge + [R, R + 1, 2**256 - 1] + ws:
        assert val(call(L.fn_host_unpack, 9, np.int32, (words(v), np.uint32))) == v
