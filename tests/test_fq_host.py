"""CPU check of the signed Fp form (fq.hip.h) and its points (g1q.hip.h), compiled by g++ from
the source the HIP kernels inline, against Python integers and the oracle: exact values, digit
and value bounds, with digits at their extremes.
"""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import oracle as O
from fk20_amd import synthetic as S

P = O.P_MOD
RINV = pow(2, -390, P)
BAL = 554_000_000  # bound of balanced digits (fq.hip.h)
TOP = 1 << 27
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def L(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("fq") / "libfq_host.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-fsanitize=signed-integer-overflow",
                    "-fsanitize-undefined-trap-on-error", "-o", out,
                    os.path.join(ROOT, "tests", "native", "fq_host.cpp")], check=True)
    return ctypes.CDLL(out)


def ptr(a):
    return a.ctypes.data_as(ctypes.c_void_p)


def val(d):
    return sum(int(x) << (30 * i) for i, x in enumerate(d))


def digits(v):
    """Balanced digits of an integer."""
    d = []
    for _ in range(12):
        x = v & ((1 << 30) - 1)
        if x >> 29:
            x -= 1 << 30
        d.append(x)
        v = (v - x) >> 30
    return d + [v]


def raw(L, op, *ops):
    z = np.zeros(13, dtype=np.int32)
    a = [np.array(x, dtype=np.int32) for x in ops] + [np.zeros(13, dtype=np.int32)] * (4 - len(ops))
    L.fq_host_raw(op, ptr(z), *[ptr(x) for x in a])
    return z


def words(v, n=12):
    return np.array([(v >> (32 * i)) & 0xFFFFFFFF for i in range(n)], dtype=np.uint32)


def unwords(w):
    return sum(int(x) << (32 * i) for i, x in enumerate(w))


def extremes(rng, count):
    """Balanced operands: every digit at +-BAL with each sign pattern of a few, and random."""
    out = [[s * BAL] * 12 + [t * TOP] for s in (1, -1) for t in (1, -1)]
    out += [[BAL * (1 if i % 2 else -1) for i in range(12)] + [TOP]]
    for _ in range(count):
        out.append([int(x) for x in rng.choice([-BAL, BAL], 12)] + [int(rng.choice([-TOP, TOP]))])
        out.append([int(x) for x in rng.integers(-BAL, BAL + 1, 12)] + [int(rng.integers(-TOP, TOP + 1))])
    return out


def check_product(z, exact):
    v = val(z)
    assert v % P == exact * RINV % P
    # |V| < |exact| / R + (1/2 + 2^-10) p, and the digit offsets' p / 32
    assert abs(v) < abs(exact) / 2**390 + 0.54 * P
    assert all(abs(int(x)) <= BAL for x in z[:12])


def test_products_at_digit_extremes(L):
    rng = np.random.default_rng(101)
    ops = extremes(rng, 60)
    for n, a in enumerate(ops):
        b, c, d = (ops[int(k)] for k in rng.integers(0, len(ops), 3))
        wide = [2 * x for x in b]
        check_product(raw(L, 0, a, b), val(a) * val(b))
        check_product(raw(L, 0, a, wide), val(a) * val(wide))
        check_product(raw(L, 0, wide, a), val(a) * val(wide))
        check_product(raw(L, 1, a), val(a) ** 2)
        check_product(raw(L, 2, a, b, c, d), val(a) * val(b) + val(c) * val(d))
        check_product(raw(L, 3, a, b, c), val(a) * val(b) - val(c) ** 2)
    a = ops[0]
    check_product(raw(L, 2, a, a, a, a), 2 * val(a) ** 2)
    check_product(raw(L, 2, a, a, ops[2], ops[3]), val(a) ** 2 + val(ops[2]) * val(ops[3]))


def test_linear_operations(L):
    rng = np.random.default_rng(102)
    ops = extremes(rng, 40)
    for a in ops:
        b, c = (ops[int(k)] for k in rng.integers(0, len(ops), 2))
        for op, args, want in ((4, [[2 * x for x in a]], 2 * val(a)), (5, [a, b], val(a) + val(b)),
                               (6, [a, b], val(a) - val(b)), (7, [a, b, c], val(a) - val(b) - val(c)),
                               (8, [a, b], 9 * val(a) - 2 * val(b)),
                               (10, [a, b, c], val(a) - 4 * val(b) - 8 * val(c))):
            z = raw(L, op, *args)
            assert val(z) == want
            assert all(abs(int(x)) <= (1 << 29) + 64 for x in z[:12])
    z = raw(L, 9, [BAL] * 12 + [1 << 24])
    assert val(z) == 12 * val([BAL] * 12 + [1 << 24])


def test_forms_round_trip(L):
    rng = np.random.default_rng(103)
    edge = [0, 1, 2, P - 1, P, P + 1, 2 * P, 2**381, 9 * P, 2**384 - 1, (P - 1) // 2, (P + 1) // 2]
    for v in edge + [int.from_bytes(rng.bytes(48), "little") for _ in range(300)]:
        m = np.zeros(13, dtype=np.int32)
        L.fq_host_from_std(ptr(m), ptr(words(v)))
        assert val(m) % P == v * 2**390 % P and abs(val(m)) < 0.6 * P
        w = np.zeros(12, dtype=np.uint32)
        L.fq_host_to_std(ptr(w), ptr(m))
        assert unwords(w) == v % P
        L.fq_host_canon(ptr(w), ptr(m))
        assert unwords(w) == v * 2**390 % P
        assert L.fq_host_is_zero(ptr(m)) == int(v % P == 0)
        # any representative within the stored range survives pack / unpack exactly
        for k in (-3, -1, 0, 1, 3):
            d = np.array(digits(val(m) + k * P), dtype=np.int32)
            L.fq_host_pack(ptr(w), ptr(d))
            assert unwords(w) == val(d) + 4 * P
            u = np.zeros(13, dtype=np.int32)
            L.fq_host_unpack(ptr(u), ptr(w))
            assert val(u) == val(d) and all(abs(int(x)) <= (1 << 29) + 1 for x in u[:12])
            L.fq_host_to_std(ptr(w), ptr(d))
            assert unwords(w) == v % P


def test_inverse(L):
    """Zero, units, values with long runs of equal bits (long and short division chains), and
    random ones, as any representative a product can leave."""
    rng = np.random.default_rng(104)
    vals = [0, 1, 2, 3, P - 1, P - 2, (P + 1) // 2, 2**380, 2**380 - 1, 2**190, P >> 1, 0x30003]
    vals += [pow(2, k, P) for k in range(1, 781, 30)] + [int.from_bytes(rng.bytes(48), "little") % P for _ in range(400)]
    for n, v in enumerate(vals):
        z = raw(L, 11, digits(v * 2**390 % P + (n % 5 - 2) * P))
        assert val(z) % P == pow(v, P - 2, P) * 2**390 % P
        assert abs(val(z)) < 0.6 * P and all(abs(int(x)) <= BAL for x in z[:12])


def test_points_against_oracle(L):
    G = O.g1p_gen()
    pts = [O.g1p_op("mul", G, O.fr(k)) for k in (1, 2, 3, 12345, O.R_MOD - 1)]
    pts += [O.g1p_op("mul", G, k) for k in S.random_fr(4, 5)] + list(S.curve_points(3, 6)) + [O.g1p_inf()]
    pts = [np.ascontiguousarray(p, dtype=np.uint64) for p in pts]

    def run(op, p, q):
        r = np.zeros(18, dtype=np.uint64)
        L.g1q_host_op(op, ptr(r), ptr(p), ptr(np.ascontiguousarray(q, dtype=np.uint64)))
        return r
    for p in pts:
        assert O.g1p_eq(run(2, p, p), O.g1p_op("dbl", p))
        assert O.g1p_eq(run(3, p, p), O.g1p_op("neg", p))
        for q in pts:
            assert O.g1p_eq(run(0, p, q), O.g1p_op("add", p, q))
            if not O.g1p_is_inf(q):
                qa = np.zeros(18, dtype=np.uint64)
                qa[:12] = O.to_affine(q)
                assert O.g1p_eq(run(1, p, qa), O.g1p_op("add", p, q))
        w = np.zeros(12, dtype=np.uint32)
        L.g1q_host_compress(ptr(w), ptr(p))
        assert w.tobytes() == bytes(O.g1_compress(p))
