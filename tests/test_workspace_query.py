"""lekf_solve_workspace_bytes covers jobs with and without trans and pao (CPU): for
32 < k <= 64 a record with trans holds the recorded rotations, 2 k^2 + 8 k pairs."""
import pytest

from letkf_amd import _lib


@pytest.mark.parametrize("k", [33, 40, 50, 64])
def test_query_covers_the_trans_records(k):
    rec = _lib.lib().lekf_solve_workspace_bytes(1, k)
    # the Gram, Q and the rotation stream with its columns
    assert rec >= 8 * (2 * k * k + 2 * (2 * k * k + 8 * k)) + 2 * (2 * k * k + 8 * k)


@pytest.mark.parametrize("k", [65, 95])
def test_query_covers_the_plain_records(k):
    rec = _lib.lib().lekf_solve_workspace_bytes(1, k)
    assert rec >= 8 * (2 * k * k + 17 * k)  # the Gram, the reflectors, 17 rows
