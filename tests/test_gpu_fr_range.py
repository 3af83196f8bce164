"""fr_fft and fr_ift over the largest inputs, any 256-bit values, in both forms of the kernel: many
transforms (8 points per lane) against few (one product per thread), and the oracle."""
import numpy as np
import pytest

import oracle as O
from fk20_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,count", [(128, 4101), (256, 2051), (512, 1025)])
def test_extremes_in_both_forms(n, count):
    rng = np.random.default_rng(n)
    x = np.zeros((count, n, 4), dtype=np.uint64)
    x[rng.integers(0, 2, (count, n)) == 1] = 0xFFFFFFFFFFFFFFFF
    x[0] = 0xFFFFFFFFFFFFFFFF
    x[1, ::2] = 0xFFFFFFFFFFFFFFFF
    x[1, 1::2] = 0
    x[2] = 0
    x[2, : n // 2] = 0xFFFFFFFFFFFFFFFF
    ends = [0, 1, 2, 3, count - 2, count - 1]
    for inverse in (False, True):
        got = ops.fr_fft(x, inverse=inverse)
        assert np.array_equal(got[ends], ops.fr_fft(x[ends], inverse=inverse))
        assert np.array_equal(got[:100], ops.fr_fft(x[:100], inverse=inverse))
        for k in ends:
            assert np.array_equal(got[k], O.fr_fft(x[k], inverse=inverse)), (k, inverse)
