"""What the adjoint asks of memory."""

import pytest

from galax_amd import _lib


@pytest.mark.parametrize("K", [1, 8, 64, 500])
def test_a_workspace_serves_every_smaller_batch(K):
    """A program sizes its workspace once, for its largest batch and longest
    span: no smaller one may need more."""
    if not _lib.LIB_PATH.exists():
        pytest.skip("libgalaxhip.so not built")
    size = _lib.lib().gx_adjoint_workspace_bytes
    ns = [0, 1, 127, 1000, 24_028, 25_001, 76_000, 132_701, 160_037, 200_000, 5_000_000]
    steps = [0, 1, 49, 490, 1000, 3000, 10_000, 400_000]
    table = [[int(size(n, m, K)) for m in steps] for n in ns]
    for i, row in enumerate(table):
        assert row == sorted(row)
        if i:
            assert all(a <= b for a, b in zip(table[i - 1], row))
