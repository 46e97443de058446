"""texture_sample at every compiled channel count and at the ends of a
thread's and a workgroup's share of the adjoint (16 and 4,096 queries), with
charts whose sides do not fit the packed records."""
import numpy as np
import pytest

from gpu_helpers import np_, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("channels,q", [(1, 1), (1, 17), (2, 4096), (2, 4099), (3, 15), (3, 8193),
                                        (4, 4095), (4, 70), (5, 4097), (7, 3)])
def test_sample_channel_counts(oracle, channels, q):
    from gstex_cuda_amd import cuda as _C

    rng = np.random.default_rng(channels * 10000 + q)
    h = np.array([1, 2, 5, 16, 70000, 1, 1])
    w = np.array([1, 3, 4, 16, 1, 66000, 1])
    start = np.concatenate([[0], np.cumsum(h * w)[:-1]])
    dims = np.stack([h, w, start], 1).astype(np.int32)
    X = int((h * w).sum())
    tex = rng.uniform(0, 1, (X, channels)).astype(np.float32)
    qd = dims[rng.integers(0, len(h), q)]
    uvs = rng.uniform(0, 1, (q, 2)).astype(np.float32)
    v = rng.standard_normal((q, channels)).astype(np.float32)
    info = (len(h), 1, channels)
    # against float64: the fraction of h u comes from one fused multiply-add,
    # so it is exact to a rounding of the fraction also on the long charts
    # (the float32 oracle rounds the product first, half an ulp of 70,000)
    got = np_(_C.texture_sample_forward(info, to_dev(qd), to_dev(uvs), to_dev(tex)))
    np.testing.assert_allclose(got, oracle.texture_sample(qd, uvs, tex, "f64"), atol=1e-6)
    back = np_(_C.texture_sample_backward(info, to_dev(qd), to_dev(uvs), to_dev(tex), to_dev(v)))
    want = oracle.texture_sample_vjp(qd, uvs, v, X, "f64")
    # float32 sums of up to q terms of size 1 on a one-texel chart
    np.testing.assert_allclose(back, want, atol=2e-6 * max(float(np.abs(want).max()), 1.0) *
                               max(q, 1) ** 0.5 + 1e-6)
