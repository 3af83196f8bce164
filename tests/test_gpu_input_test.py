"""The membership test that the drop-in transforms run beside the load of their inputs: one flag per
transform, whichever schedule follows.  The transforms of one curve point outside G1 in the first,
a middle and the last row equal the same rows transformed alone (which the oracle pins), the rows
between them those of an all-G1 batch.
"""
import numpy as np
import pytest

import oracle as O
from fk20_amd import ops, synthetic as S

pytestmark = pytest.mark.gpu


def aff(pts):
    return O.to_affine(np.ascontiguousarray(pts, dtype=np.uint64).reshape(-1, 18))


@pytest.mark.parametrize("rows", [1, 2, 65, 257])  # direct (pairs of lanes, single lanes), radix 2^2
@pytest.mark.parametrize("kind", ["fft", "ifft", "fused"])
def test_flags_are_per_row(rows, kind):
    n = 128
    run = {"fft": ops.g1p_fft, "ifft": lambda x: ops.g1p_fft(x, inverse=True), "fused": ops.hext_fft2h_fft}[kind]
    x = ops.g1p_op("mul", np.tile(O.g1p_gen(), (rows * n, 1)), k=S.random_fr(rows * n, 61)).reshape(rows, n, 18)
    clean = run(x)
    bad = sorted({0, rows // 2, rows - 1})
    for r in bad:
        x[r, n - 1 if r else 0] = S.curve_points(1, 62 + r)[0]
    got = run(x)
    keep = [r for r in range(rows) if r not in bad]
    assert np.array_equal(got[keep], clean[keep])
    for r in bad:
        assert np.array_equal(aff(got[r]), aff(run(x[r:r + 1])))
        assert not np.array_equal(aff(got[r]), aff(clean[r]))
