"""fk20_commit_workspace_bytes: what a call cannot do without, linear in its rows, so that no call
after a larger one needs more."""
import pytest

from fk20_amd import lib as L


@pytest.mark.parametrize("N", [1024, 2048, 4096])
def test_linear_in_the_rows(N):
    f = L.lib().fk20_commit_workspace_bytes
    per_row = (N // 16 + N // 256) * 144
    for rows in list(range(0, 70)) + [128, 129, 191, 192, 193, 256, 320, 511, 512, 513, 4096]:
        assert f(rows, N) == rows * per_row, rows
