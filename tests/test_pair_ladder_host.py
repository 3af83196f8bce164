"""CPU check of the two-lane ladder (ladder_pair.hip.h, both lanes emulated): every twiddle program
and the short w^128 form on random points given as non-normalised projective inputs."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import oracle as O
from fk20_amd import prover, synthetic as S

P, R = O.P_MOD, O.R_MOD
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def L(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("pair") / "libpair_host.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-fsanitize=signed-integer-overflow",
                    "-fsanitize-undefined-trap-on-error", "-o", out,
                    os.path.join(ROOT, "tests", "native", "pair_host.cpp")], check=True)
    return ctypes.CDLL(out)


def ptr(a):
    return a.ctypes.data_as(ctypes.c_void_p)


def test_programs_and_short_form(L):
    rng = np.random.default_rng(301)
    w = pow(5, (R - 1) // 512, R)
    exps = [e for e in range(1, 256) if e != 128] + [128]
    s = S.random_fr(len(exps), 302)
    zs = np.array([O.fp(int.from_bytes(rng.bytes(48), "little") % (P - 1) + 1) for _ in exps])
    pts = np.ascontiguousarray(O.gen_mul_projective(s, zs))
    want = O.gen_mul_affine(np.array([O.fr(pow(w, e, R) * O.limbs_to_int(k) % R) for e, k in zip(exps, s)]))
    r = np.zeros((2, len(exps), 18), dtype=np.uint64)
    for n, e in enumerate(exps):
        if e == 128:
            L.pair_host_z3(ptr(r[0, n]), ptr(r[1, n]), ptr(pts[n]))
        else:
            L.pair_host_tw_mul(ptr(r[0, n]), ptr(r[1, n]), ptr(pts[n]), ptr(prover.twiddle_program(0, e)))
    assert np.array_equal(r[0], r[1])
    bad, first = O.match_affine(r[0], want)
    assert bad == 0, exps[first]


def test_doublings(L):
    """[2^n] of projective points in G1 and of curve points outside it."""
    s = S.random_fr(4, 303)
    zs = np.array([O.fp(7 + k) for k in range(4)])
    pts = np.concatenate([O.gen_mul_projective(s, zs), S.curve_points(4, 304)])
    r = np.zeros((2, 18), dtype=np.uint64)
    for p in pts:
        for n in (0, 1, 6, 40):
            L.pair_host_dbl_n(ptr(r[0]), ptr(r[1]), ptr(p), n)
            want = p
            for _ in range(n):
                want = O.g1p_op("dbl", want)
            assert np.array_equal(r[0], r[1])
            assert np.array_equal(O.to_affine(r[:1]), O.to_affine(np.asarray(want).reshape(1, 18))), n


def test_membership(L):
    """The pair's comparison against the definition [r]P = 0: points of G1, infinity, curve points,
    points of small order and their sums with G1 points."""
    from test_device_arith_host import H_COF, _mul_big
    G = O.g1p_gen()
    curve = list(S.curve_points(3, 305))
    pts = [G, O.g1p_inf(), O.g1p_op("mul", G, O.fr(R - 1))] + curve + [_mul_big(curve[0], H_COF)]
    small = []
    for q in curve:
        rq = O.g1p_op("mul", q, O.fr(R))
        small += [t for t in (_mul_big(rq, H_COF // m) for m in (3, 11, 121)) if not O.g1p_is_inf(t)]
    assert small
    pts += small + [O.g1p_op("add", G, t) for t in small[:2]]
    for p in pts:
        want = O.g1p_is_inf(O.g1p_op("mul", p, O.fr(R)))
        assert L.pair_host_in_subgroup(ptr(np.ascontiguousarray(p))) == int(want)
