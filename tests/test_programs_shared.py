"""What lets one set of programs serve both directions and every user: w^-i runs w^(512 - i)'s, and a
program depends on its scalar and width alone."""
import numpy as np
import pytest

from fk20_amd import prover


@pytest.mark.parametrize("wnaf", [3, 4, 5])
def test_inverse_programs_are_the_forward_ones(wnaf):
    fwd = [prover.twiddle_program(0, i, wnaf) for i in range(512)]
    for i in range(512):
        assert np.array_equal(prover.twiddle_program(1, i, wnaf), fwd[(512 - i) % 512]), i
    if wnaf == 5:
        status, total, width = prover.twiddle_selfcheck()
        assert (status, width) == (0, 5) and total == 2 * sum(len(p) for p in fwd)
