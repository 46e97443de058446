"""The intersect keys, written by position: runs of 8 positions a thread and
2,048 a workgroup, against the oracle, at counts that are the rectangles', that
are larger (slots left zero), or smaller (rows cut), with Gaussians that count
nothing in between.  And the stable 64-bit sort on both sides of its tile rule."""
import numpy as np
import pytest
import torch

from gpu_helpers import np_, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wrapped", [False, True])
@pytest.mark.parametrize("counts", ["own", "more", "less"])
@pytest.mark.parametrize("n", [1, 7, 300, 5000])
def test_map_by_position(oracle, n, counts, wrapped):
    if counts == "less" and not wrapped:
        pytest.skip("the oracle bounds writes by the counts in wrapped mode only")
    from gstex_cuda_amd import cuda as _C

    rng = np.random.default_rng(n)
    bw, w, h = 16, 200, 136
    tb = ((w + bw - 1) // bw, (h + bw - 1) // bw, 1)
    c = (rng.uniform(-0.3, 1.3, (n, 2)) * [w, h]).astype(np.float32)
    e = np.exp(rng.uniform(0, 4.5, (n, 2))).astype(np.float32)
    e[rng.random(n) < 0.2] = 0
    d = rng.uniform(0.1, 9, n).astype(np.float32)
    nt = oracle.num_tiles_hit(c, e, h, w, bw, wrapped=wrapped).astype(np.int64)
    if counts == "more":
        nt = nt + rng.integers(0, 12, n) * (rng.random(n) < 0.5)
    elif counts == "less":
        nt = nt // rng.integers(1, 4, n)
    cum = np.cumsum(nt).astype(np.int32)
    for m in (int(cum[-1]), int(cum[-1]) + 5):  # five positions past the last count
        if m == 0:
            continue
        keys, ids = _C.map_gaussian_to_intersects(n, m, to_dev(c), to_dev(e), to_dev(d),
                                                  to_dev(cum), tb, bw, wrapped=wrapped)
        o_keys, o_ids = oracle.map_gaussian_to_intersects(c, e, d, cum, tb, bw, num_intersects=m,
                                                          wrapped=wrapped)
        assert np.array_equal(np_(keys), o_keys)
        assert np.array_equal(np_(ids), o_ids)


@pytest.mark.parametrize("n", [(1 << 22) + 1, (1 << 23) - 1, 1 << 23])
def test_sort_tiles_of_64_bit_pairs(n):
    from gstex_cuda_amd import cuda as _C

    rng = np.random.default_rng(n)
    k = (rng.integers(0, 300, n) << 32) | rng.integers(0, 1 << 12, n)
    ks, vs = _C.sort_intersects(to_dev(k), torch.arange(n, dtype=torch.int32, device="cuda"), 41)
    order = np.argsort(k, kind="stable")
    assert np.array_equal(np_(vs), order)
    assert np.array_equal(np_(ks), k[order])
