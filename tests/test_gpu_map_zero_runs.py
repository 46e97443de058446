"""The intersect keys of scenes with long runs of Gaussians that count nothing, and
of wrapped rectangles wider than a 32-bit integer holds."""
import numpy as np
import pytest
import torch

from gpu_helpers import log, np_, to_dev

pytestmark = pytest.mark.gpu


def _inputs(n, visible):
    c = np.full((n, 2), 100, np.float32)
    e = np.zeros((n, 2), np.float32)
    e[visible] = 12.0  # tiles 5..7 in both directions: nine
    cum = np.cumsum(np.where(e[:, 0] > 0, 9, 0)).astype(np.int32)
    return [to_dev(x) for x in (c, e, np.linspace(1, 2, n).astype(np.float32), cum)], int(cum[-1])


def _map(n, m, dev):
    from gstex_cuda_amd import cuda as _C

    return _C.map_gaussian_to_intersects(n, m, *dev, (20, 20, 1), 16)


@pytest.mark.parametrize("n,first,last,more", [
    (1_000_100, 50, 50, 0), (1_000_100, 1, 99, 7), (300_000, 3, 0, 5000), (70_000, 0, 300, 1),
    (5000, 299, 299, 3)])
def test_zero_run(n, first, last, more):
    visible = np.r_[0:first, n - last:n]
    dev, m = _inputs(n, visible)
    keys, ids = _map(n, m + more, dev)
    tiles = np.array([y * 20 + x for y in (5, 6, 7) for x in (5, 6, 7)])
    depth = np_(dev[2]).view(np.int32).astype(np.int64)[visible]
    want = ((tiles[None].astype(np.int64) << 32) | depth[:, None]).reshape(-1)
    assert np.array_equal(np_(keys), np.r_[want, np.zeros(more, np.int64)])
    assert np.array_equal(np_(ids), np.r_[np.repeat(visible, 9), np.zeros(more)])


def test_zero_run_time():
    # a run of a million against the same Gaussians spread evenly
    n, k = 1_000_200, 200
    times = []
    for visible in (np.arange(k) * (n // k), np.r_[0:k // 2, n - k // 2:n]):
        dev, m = _inputs(n, visible)
        _map(n, m + 5, dev)
        e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        e[0].record()
        for _ in range(3):
            _map(n, m + 5, dev)
        e[1].record()
        torch.cuda.synchronize()
        times.append(e[0].elapsed_time(e[1]) / 3)
    log("map ms, spread and in one run", times)
    assert times[1] < 4 * times[0] + 1.0


@pytest.mark.parametrize("axis", [0, 1, None])
def test_wrapped_huge_extent(axis):
    # tile corners saturate at the ends of the 32-bit range; each Gaussian writes
    # the first tiles of its row-major rectangle, as many as it counts
    from gstex_cuda_amd import cuda as _C

    lo, nx, ny = -2**31, 20, 13
    e = np.full((3, 2), 1e12, np.float32)
    if axis is not None:
        e[:, 1 - axis] = 12.0  # tiles 5..7
    c = np.full((3, 2), 100, np.float32)
    d = np.array([1, 2, 3], np.float32)
    counts = np.array([5, 40, 3000])
    cum = np.cumsum(counts).astype(np.int32)
    keys, ids = _C.map_gaussian_to_intersects(3, int(cum[-1]), to_dev(c), to_dev(e), to_dev(d),
                                              to_dev(cum), (nx, ny, 1), 16, wrapped=True)
    x0, x1 = (5, 8) if axis == 1 else (lo, 2**31 - 1)
    y0, y1 = (5, 8) if axis == 0 else (lo, 2**31 - 1)
    want_k, want_i = [], []
    for g in range(3):
        k = np.arange(counts[g])
        r, q = k // (x1 - x0), k % (x1 - x0)
        tile = ((y0 + r) % ny) * nx + (x0 + q) % nx
        key = (tile.astype(np.int64) << 32) | int(d[g:g + 1].view(np.int32)[0])
        written = r < y1 - y0
        want_k.append(np.where(written, key, 0))
        want_i.append(np.where(written, g, 0))
    assert np.array_equal(np_(keys), np.concatenate(want_k))
    assert np.array_equal(np_(ids), np.concatenate(want_i))
