"""A workspace sized for the most intersects a program sorts does for fewer."""
import pytest

EDGES = [1 << 12, 1 << 21, 1 << 22, 1 << 23, 1 << 24]


@pytest.mark.parametrize("edge", EDGES)
def test_sort_intersects_workspace_does_not_shrink(edge):
    from gstex_cuda_amd import _lib

    size = _lib.lib().gstex_sort_intersects_workspace_size
    counts = sorted({edge + d for d in (-200_000, -4096, -2048, -1, 0, 1, 2048, 4096, 200_000)
                     if edge + d > 0})
    sizes = [size(n) for n in counts]
    assert sizes == sorted(sizes), dict(zip(counts, sizes))
