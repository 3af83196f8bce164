"""What a context's workspace holds after calls of one size, for calls of another."""
import numpy as np
import pytest

import oracle as O
from fk20_amd import synthetic as S
from fk20_amd.lib import DeviceBuffer, synchronize
from fk20_amd.prover import Prover

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("before", [None, (4, 4096), (5, 4096), (10, 1024)])
def test_a_single_row_runs_in_one_step(before):
    """A row of 4096 takes the direct schedule in one step (4 launches per transform, 12 of two
    steps' both) whatever was reserved first."""
    N, n = 4096, 512
    tau = S.random_secret(81)
    poly = S.random_polys(1, N, 82)
    with Prover() as p:
        sid = p.load_setup(O.xext_fft_from_tau(tau, N), N, 8)
        if before:
            p.reserve(*before)
        pb, hb = DeviceBuffer.from_array(poly), DeviceBuffer(n * 144)
        p.set_launch_timing(True)
        p.prove_device(sid, hb, pb, 1)
        synchronize()
        assert len(p.launch_times()) == 3 + 2 * 4
        got = hb.download((1, n, 18))
    assert O.match_affine(got, O.fk20_closed_form_affine(poly, tau)) == (0, -1)
