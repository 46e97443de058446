"""Launch shapes at their ends: the projection with its total (at most 1,024
workgroups, each over several strides) against the projection without it, and
the SH forward's staged bfloat16 rows against float32 rows of the same values."""
import numpy as np
import pytest
import torch

from gpu_helpers import DEV, np_, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 255, 262_144, 262_145, 600_001])
def test_projection_total(n):
    from gstex_cuda_amd import cuda as _C
    from gstex_cuda_amd._lib import call

    rng = np.random.default_rng(n)
    means = rng.uniform(-1, 1, (n, 3)).astype(np.float32) + np.array([0, 0, 4], np.float32)
    scales = np.exp(rng.uniform(-4, -2, (n, 3))).astype(np.float32)
    q = rng.standard_normal((n, 4)).astype(np.float32)
    q /= np.linalg.norm(q, axis=1, keepdims=True)
    t = [to_dev(a) for a in (means, scales, q, np.eye(4, dtype=np.float32))]
    want = _C.project_gaussians(t[0], t[1], 1.0, t[2], t[3], 300.0, 300.0, 160.0, 120.0, 240, 320,
                                16)
    got = [torch.empty_like(w) for w in want]
    total = torch.zeros(1, dtype=torch.int32, device=DEV)
    call("gstex_project_gaussians_total", n, t[0].data_ptr(), t[1].data_ptr(), 1.0,
         t[2].data_ptr(), t[3].data_ptr(), 300.0, 300.0, 160.0, 120.0, 240, 320, 16,
         *[g.data_ptr() for g in got], total.data_ptr(), torch.cuda.current_stream().cuda_stream)
    for g, w in zip(got, want):
        assert np.array_equal(np_(g), np_(w), equal_nan=True)
    assert int(total.item()) == int(want[3].sum().item())


# rows of 3, 12, 27, 48 and 75 values (whole words for 12 and 48 only)
@pytest.mark.parametrize("degree", [0, 1, 2, 3, 4])
@pytest.mark.parametrize("n", [1, 256, 1021])
def test_sh_forward_bf16_rows(degree, n):
    from gstex_cuda_amd import cuda as _C

    g = torch.Generator(device="cuda").manual_seed(degree * 7 + n)
    dirs = torch.randn((n, 3), device=DEV, generator=g)
    c = torch.randn((n, (degree + 1) ** 2, 3), device=DEV, generator=g).bfloat16()
    got = _C.compute_sh_forward(n, degree, degree, dirs, c)
    want = _C.compute_sh_forward(n, degree, degree, dirs, c.float())
    assert np.array_equal(np_(got), np_(want))
    # an offset that breaks the 16-byte alignment takes the direct reads
    flat = torch.cat([c.new_zeros(1), c.reshape(-1)])[1:].reshape(c.shape)
    assert np.array_equal(np_(_C.compute_sh_forward(n, degree, degree, dirs, flat)), np_(want))
