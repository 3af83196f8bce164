"""The direct schedule of small batches (direct.hip.h) against the radix-2^2 launches a large batch
takes: same rows, same words (proofs have z = 1), at the row counts where its packing of rows and
products into waves changes, for every size, entry point and workspace it runs in.
"""
import ctypes

import numpy as np
import pytest

import oracle as O
from fk20_amd import ops, synthetic as S
from fk20_amd.lib import DeviceBuffer, call, lib, synchronize
from fk20_amd.prover import BatchItem, Prover

pytestmark = pytest.mark.gpu

LARGE = 300  # rows beyond the direct schedule's largest batch


@pytest.fixture(scope="module")
def prover():
    p = Prover()
    yield p
    p.close()


@pytest.mark.parametrize("N", [1024, 2048, 4096])
def test_small_batches_equal_rows_of_a_large_one(prover, N):
    sid = prover.load_setup(O.xext_fft_from_tau(S.random_secret(N + 1), N), N, 8)
    poly = S.random_polys(LARGE, N, N + 2)
    poly[3] = 0  # a zero row: every proof is infinity
    poly[4, 1:] = 0
    want = prover.prove(sid, poly)
    for rows in (1, 2, 3, 5, 8, 9, 16, 17, 21, 32, 33, 64, 65, 130):
        got = prover.prove(sid, poly[:rows])
        assert np.array_equal(got, want[:rows]), rows
    # a workspace of exactly the documented size has no room for two levels' products
    for rows in (1, 7, 40):
        ws = DeviceBuffer(int(lib().fk20_rows_workspace_bytes(rows, N)))
        pb, hb = DeviceBuffer.from_array(poly[:rows]), DeviceBuffer(rows * (N // 8) * 144)
        item = (BatchItem * 1)(BatchItem(sid, rows, pb.ptr, hb.ptr))
        call("fk20_prove_batch_ws", prover.ctx, item, 1, ws.ptr, ctypes.c_size_t(ws.nbytes), None)
        synchronize()
        assert np.array_equal(hb.download((rows, N // 8, 18)), want[:rows]), rows
    prover.unload_setup(sid)


def test_small_uneven_batch(prover):
    groups, want = [], []
    for N, rows in ((4096, 3), (1024, 18), (2048, 1)):
        sid = prover.load_setup(O.xext_fft_from_tau(S.random_secret(N + 3), N), N, 8)
        poly = S.random_polys(LARGE, N, N + 4)
        want.append(prover.prove(sid, poly)[:rows])
        groups.append((sid, poly[:rows]))
    for got, exp in zip(prover.prove_batch(groups), want):
        assert np.array_equal(got, exp)


@pytest.mark.parametrize("n", [128, 256, 512])
def test_drop_in_transforms(n):
    G = O.g1p_gen()
    k = S.random_fr(LARGE * n, n + 5)
    x = ops.g1p_op("mul", np.tile(G, (LARGE * n, 1)), k=k).reshape(LARGE, n, 18)
    x[2, 5] = O.g1p_inf()
    for inverse in (False, True):
        want = ops.g1p_fft(x, inverse=inverse)
        for count in (1, 4, 6, 33, 65):
            assert np.array_equal(ops.g1p_fft(x[:count], inverse=inverse), want[:count]), (inverse, count)
    want = ops.hext_fft2h_fft(x)
    for count in (1, 11, 64):
        assert np.array_equal(ops.hext_fft2h_fft(x[:count]), want[:count]), count


def test_drop_in_rows():
    N = 2048
    xext = O.xext_fft_from_tau(S.random_secret(9), N)
    poly = S.random_polys(LARGE, N, 10)
    want = ops.poly2h_fft(poly, xext)
    for rows in (1, 12, 50):
        assert np.array_equal(ops.poly2h_fft(poly[:rows], xext), want[:rows]), rows
