"""Batches beyond the direct schedule's (more than 256 rows of one item): the radix-2^2 launches of
every schedule variant, and the halves on two streams, against each other and the closed form."""
import ctypes

import numpy as np
import pytest

import oracle as O
from fk20_amd import synthetic as S
from fk20_amd.lib import DeviceBuffer, Stream, synchronize
from fk20_amd.prover import Prover

pytestmark = pytest.mark.gpu


def batch(prover, shape):
    """[(setup, polynomials)] and the secrets, of (N, rows) items."""
    groups, taus = [], []
    for N, rows in shape:
        taus.append(S.random_secret(N + rows))
        groups.append((prover.load_setup(O.xext_fft_from_tau(taus[-1], N), N, 8), S.random_polys(rows, N, N + 5)))
    return groups, taus


def pin(groups, taus, outs):
    for (_, poly), tau, got in zip(groups, taus, outs):
        ends = [0, poly.shape[0] - 1]
        assert O.match_affine(got[ends], O.fk20_closed_form_affine(poly[ends], tau)) == (0, -1)


def test_every_schedule_variant():
    with Prover() as p:
        # one row past a group of 64, few rows, a group and a row
        groups, taus = batch(p, [(1024, 257), (4096, 3), (2048, 65)])
        want = p.prove_batch(groups)
        pin(groups, taus, want)
        for (sid, poly), w in zip(groups, want):  # the same rows alone, in the direct schedule
            assert np.array_equal(p.prove(sid, poly[-3:]), w[-3:])
        for wnaf in (3, 4, 5):
            for radix in (2, 4):
                for waves in (2, 3):
                    p.set_schedule(wnaf, radix, waves)
                    for got, w in zip(p.prove_batch(groups), want):
                        assert np.array_equal(got, w), (wnaf, radix, waves)
            p.set_schedule(wnaf, 4, 2)
            p.set_chain(True)
            for got, w in zip(p.prove_batch(groups), want):
                assert np.array_equal(got, w), (wnaf, "chain")
            p.set_chain(False)


# 16 groups of 64 rows and more of several sizes run in halves: ragged ones, items that only the
# first half has, and a second half of one item
@pytest.mark.parametrize("shape", [[(1024, 641), (2048, 300), (4096, 40)], [(2048, 20), (1024, 963), (4096, 64)]])
def test_halves_on_two_streams(shape):
    with Prover() as p:
        groups, taus = batch(p, shape)
        p.set_streams(1)
        want = p.prove_batch(groups)
        pin(groups, taus, want)
        p.set_streams(2)
        for _ in range(2):
            for got, w in zip(p.prove_batch(groups), want):
                assert np.array_equal(got, w)
        p.set_chain(True)
        for got, w in zip(p.prove_batch(groups), want):
            assert np.array_equal(got, w)
        p.set_chain(False)
        # captured once, with the fork and the join, and replayed between eager work
        polys = [DeviceBuffer.from_array(poly) for _, poly in groups]
        outs = [DeviceBuffer(w.nbytes) for w in want]
        items = [(sid, poly.shape[0], pb, hb) for (sid, poly), pb, hb in zip(groups, polys, outs)]
        st = Stream()
        p.set_graph(True)
        for _ in range(3):
            for hb in outs:
                hb.fill(0x3C)
            synchronize()
            p.prove_batch_device(items, ctypes.c_void_p(st.handle))
            st.synchronize()
            for hb, w in zip(outs, want):
                assert np.array_equal(hb.download(w.shape), w)
        p.set_graph(False)
        st.destroy()
