"""Commitments at the row counts where the kernel's lanes per row and coefficients per lane change:
each row equals the same row committed in a large batch, whose first rows are pinned by the oracle."""
import numpy as np
import pytest

import oracle as O
from fk20_amd import ops, synthetic as S
from fk20_amd.prover import Prover

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,window", [(1024, 13), (2048, 8), (4096, 9)])
def test_small_batches_equal_rows_of_a_large_one(N, window):
    rows = 130
    srs = S.device_srs(N, S.random_secret(N)).download((N, 18))
    poly = S.random_polys(rows, N, N + 1)
    poly[1] = 0
    with Prover() as p:
        sid = p.load_commit_setup(srs, N, window)
        want = ops.to_affine(p.commit(sid, poly))
        assert np.array_equal(want[:3], np.stack([O.to_affine(c) for c in O.commit(poly[:3], srs)]))
        for r in (1, 2, 3, 4, 5, 16, 17, 32, 33, 63, 64, 65, 128):
            assert np.array_equal(ops.to_affine(p.commit(sid, poly[:r])), want[:r]), r
