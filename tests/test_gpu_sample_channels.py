"""texture_sample at every compiled channel count, against the kernels for a
runtime count (the same channels among more), at the ends of a thread's and a
workgroup's share of the adjoint (16 and 4,096 queries), with charts whose
sides do not fit the packed records."""
import numpy as np
import pytest

from gpu_helpers import np_, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("channels,q", [(1, 1), (1, 17), (2, 4096), (2, 4099), (3, 15), (3, 8193),
                                        (4, 4095), (4, 70), (5, 4097), (7, 3)])
def test_sample_channel_counts(channels, q):
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

    def run(t, g):
        info, c = (len(h), 1, t.shape[1]), channels
        a = (info, to_dev(qd), to_dev(uvs), to_dev(t))
        return (np_(_C.texture_sample_forward(*a))[:, :c],
                np_(_C.texture_sample_backward(*a, to_dev(g)))[:, :c])

    got, back = run(tex, v)
    # five channels more, whose values are others: the runtime-count kernels
    want, want_back = run(np.concatenate([tex, rng.uniform(0, 1, (X, 5)).astype(np.float32)], 1),
                          np.concatenate([v, rng.standard_normal((q, 5)).astype(np.float32)], 1))
    np.testing.assert_allclose(got, want, atol=1e-6)
    # float32 sums of up to q terms of size 1 on a one-texel chart, in atomic order
    np.testing.assert_allclose(back, want_back, atol=2e-6 * max(float(np.abs(want_back).max()), 1.0)
                               * max(q, 1) ** 0.5 + 1e-6)
