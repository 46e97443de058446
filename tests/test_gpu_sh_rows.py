"""SH colours from coefficient rows of every kind: through LDS (16-byte aligned) and
through registers (other addresses, rows of a broken word, degree 4) they are the
same bits, and those of the float64 formula up to float32 rounding."""
import numpy as np
import pytest
import torch

from gpu_helpers import DEV, np_

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("degree", range(5))
@pytest.mark.parametrize("n", [1, 255, 257, 1000])
def test_rows(oracle, n, degree, dtype):
    from gstex_cuda_amd import cuda as _C

    rng = np.random.default_rng(degree)
    d = (degree + 1) ** 2
    dirs = torch.from_numpy(rng.standard_normal((n, 3)).astype(np.float32)).to(DEV)
    co = torch.from_numpy(rng.standard_normal((n, d, 3)).astype(np.float32)).to(DEV).to(dtype)
    for use in range(degree + 1):
        ref = np_(_C.compute_sh_forward(n, degree, use, dirs, co))
        want = oracle.sh_forward(degree, use, np_(dirs), np_(co.float()), "f64")
        assert np.abs(ref - want).max() < 1e-5 * max(1.0, np.abs(want).max())
        for shift in (1, 2, 3):
            buf = torch.full((n * d * 3 + 8,), float("nan"), device=DEV, dtype=dtype)
            row = buf[shift:shift + n * d * 3].view(n, d, 3)
            row.copy_(co)
            got = np_(_C.compute_sh_forward(n, degree, use, dirs, row))
            assert np.array_equal(got, ref), (use, shift)
