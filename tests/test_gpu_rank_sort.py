"""The one-launch sort of few 32-bit pairs at the edges of its workgroups (64
items), quarters and range (8,192), with ties, extreme keys and an in-place call."""
import numpy as np
import pytest
import torch

from gpu_helpers import np_, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 63, 64, 65, 255, 257, 1000, 4095, 8191, 8192, 8193])
@pytest.mark.parametrize("spread", [3, 1 << 32])
def test_sort_few_pairs(n, spread):
    from gstex_cuda_amd import cuda as _C

    rng = np.random.default_rng(n)
    k = rng.integers(0, spread, n).astype(np.uint32)
    k[rng.random(n) < 0.1] = 0xFFFFFFFF
    k[rng.random(n) < 0.05] = 0
    order = np.argsort(k, kind="stable")
    vals = torch.arange(n, dtype=torch.int32, device="cuda")
    ks, vs = _C.sort_pairs_u32(to_dev(k.view(np.int32)), vals, 32)
    assert np.array_equal(np_(vs), order)
    assert np.array_equal(np_(ks).view(np.uint32), k[order])
