"""The transforms' Fr form at the ends of the range that any 256-bit inputs reach: products of sums of
eight of them, and the canonical form on both sides of what a product can be."""
import numpy as np

import oracle as O
from test_fn_host import L, call, val, words  # noqa: F401  (L: the host build)

R = O.R_MOD


def digits(v):
    return [(v >> (29 * i)) & 0x1FFFFFFF for i in range(8)] + [v >> 232]


def test_products_of_eight_inputs(L):  # noqa: F811
    rng = np.random.default_rng(301)
    top = 2**256 - 1
    assert 8 * top < 18 * R
    ws = [R - 1, R - 2, (R - 1) // 2, 1] + [int.from_bytes(rng.bytes(32), "little") % R for _ in range(20)]
    # four inputs a sum as dft8 adds them, digit by digit, then the balanced halves of eight
    four = [sum(x) for x in zip(*[digits(top)] * 4)]
    half = call(L.fn_host_norm, 9, np.int32, (four, np.int32))
    eight = [2 * int(x) for x in half]
    assert val(eight) == 8 * top
    for a in (four, [-x for x in four], eight, [-x for x in eight], digits(18 * R - 1), digits(1 - 18 * R)):
        for w in ws:
            wd = call(L.fn_host_from_words, 9, np.int32, (words(w), np.uint32))
            z = call(L.fn_host_mul, 9, np.int32, (a, np.int32), (wd, np.int32))
            v = val(z)
            assert v % R == val(a) * w * pow(2, -261, R) % R and -126 * R < 100 * v < 26 * R
            got = call(L.fn_host_canon, 8, np.uint32, (z, np.int32))
            assert sum(int(x) << (32 * i) for i, x in enumerate(got)) == v % R


def test_canonical_form_over_its_whole_range(L):  # noqa: F811
    for v in (-2 * R, -2 * R + 1, -2 * R + R // 2, -R - 1, -R, -R + 1, -1, 0, 1, R // 2, R - 2, R - 1):
        got = call(L.fn_host_canon, 8, np.uint32, (digits(v), np.int32))
        assert sum(int(x) << (32 * i) for i, x in enumerate(got)) == v % R, v
