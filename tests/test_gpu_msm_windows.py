"""fk20_msm where its kernel, window and lanes per row change (LDS kernel, 16, 4 and 1 lanes per row,
windows of 7 to 10 bits): the rows of a small call equal the same rows of a large one, whose ends
are pinned by the oracle, with scalars at the digit recoding's extremes and exceptional sums."""
import numpy as np
import pytest

import oracle as O
from fk20_amd import ops, synthetic as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [128, 512])
def test_rows_do_not_depend_on_the_call(n):
    rows = 260
    x = ops.g1p_op("mul", np.tile(O.g1p_gen(), (16 * n, 1)), k=S.random_fr(16 * n, n)).reshape(16, n, 18)
    x[3, 5] = O.g1p_inf()
    x[7, 9] = x[6, 9]                         # equal bases: additions of equal points
    x[8, 9] = O.g1p_op("neg", x[6, 9])        # and of opposite ones
    x[9, 11] = S.curve_points(1, n)[0]        # a base outside G1
    tc = S.random_fr(rows * 16 * n, n + 1).reshape(rows, 16, n, 4)
    tc[0, :, :8] = 0xFFFFFFFFFFFFFFFF         # any 256-bit scalar
    tc[1, :, :8] = 0
    tc[2] = 0
    tc[2, :, :, 3] = 1 << 63
    tc[3, 6:9, 9] = tc[3, 6, 9]               # k X + k X - k X
    want = ops.to_affine(ops.msm(tc, x))
    for r in (0, 1, 2, 3):
        for j in (0, 5, 9, 11):
            acc = O.g1p_inf()
            for i in range(16):
                acc = O.g1p_op("add", acc, O.g1p_op("mul", x[i, j], tc[r, i, j]))
            assert np.array_equal(O.to_affine(acc), want[r, j]), (r, j)
    for r in (4, 16, 17, 33, 64, 65, 100, 129):
        assert np.array_equal(ops.to_affine(ops.msm(tc[:r], x)), want[:r]), r


@pytest.mark.parametrize("n", [128, 256, 512])
def test_few_rows(n):
    """Two lanes per ladder and one (up to 8, 4, 2 rows and beyond), rows after infinities, equal,
    opposite and small-multiple sums, and a base outside G1."""
    x = ops.g1p_op("mul", np.tile(O.g1p_gen(), (16 * n, 1)), k=S.random_fr(16 * n, n + 7)).reshape(16, n, 18)
    x[3, 5] = O.g1p_inf()
    x[7, 9] = x[6, 9]
    x[8, 9] = O.g1p_op("neg", x[6, 9])
    x[9, 11] = S.curve_points(1, n + 8)[0]
    rows = 17
    tc = S.random_fr(rows * 16 * n, n + 9).reshape(rows, 16, n, 4)
    tc[0, :, :8] = 0xFFFFFFFFFFFFFFFF
    tc[1, :, 8:16] = 0
    tc[1, :, 9, 1] = 64                       # a leading zero digit, then infinity + d P
    tc[1, 6:9, 9] = tc[0, 6, 9]
    want = ops.to_affine(ops.msm(tc, x))
    for r in (0, 1):
        for j in (0, 5, 8, 9, 11, 100):
            acc = O.g1p_inf()
            for i in range(16):
                acc = O.g1p_op("add", acc, O.g1p_op("mul", x[i, j], tc[r, i, j]))
            assert np.array_equal(O.to_affine(acc), want[r, j]), (r, j)
    for r in (1, 2, 3, 4, 5, 8, 9, 16):
        assert np.array_equal(ops.to_affine(ops.msm(tc[:r], x)), want[:r]), r
    for r in range(2, 9):
        assert np.array_equal(ops.to_affine(ops.msm(tc[r:r + 1], x)), want[r:r + 1]), r
