"""The offset scan over depth-ordered Gaussians at the edges of its tiles (4
positions a thread up to 200,000 Gaussians, 8 beyond) through the binning."""
import numpy as np
import pytest
import torch

from gpu_helpers import DEV, np_, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 1023, 1024, 1025, 200_000, 200_001, 204_800, 204_805])
def test_binning_at_scan_tile_edges(n):
    from gstex_cuda_amd import cuda as _C
    from gstex_cuda_amd.utils import bin_and_sort_gaussians, compute_cumulative_intersects

    rng = np.random.default_rng(n)
    h, w, bw = 240, 320, 16
    c = to_dev((rng.uniform(-0.1, 1.1, (n, 2)) * [w, h]).astype(np.float32))
    e = rng.uniform(0.5, 12, (n, 2)).astype(np.float32)
    e[rng.random(n) < 0.1] = 0
    e = to_dev(e)
    d = to_dev(rng.uniform(0.1, 9, n).astype(np.float32))
    nt = _C.num_tiles_hit(c, e, h, w, bw)
    m, cum = compute_cumulative_intersects(nt)
    if m == 0:
        return
    tb = ((w + bw - 1) // bw, (h + bw - 1) // bw, 1)
    _, _, _, ids, bins = bin_and_sort_gaussians(n, m, c, e, d, cum, tb, bw)
    got = _C.bin_gaussians(n, m, c, e, d, nt, tb, bw)
    assert np.array_equal(np_(got[0]), np_(ids))
    assert np.array_equal(np_(got[1]), np_(bins))
