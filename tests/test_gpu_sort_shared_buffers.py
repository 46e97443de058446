"""sort_pairs_u32 on outputs that share memory with the inputs: in place, crossed
and partly overlapping, at sizes of the one-launch sort and past it."""
import numpy as np
import pytest
import torch

from gpu_helpers import DEV, np_

pytestmark = pytest.mark.gpu

# offsets of (keys, values, sorted keys, sorted values) in one buffer, in units
# of n words and of single words
LAYOUTS = {
    "apart": ((0, 0), (1, 0), (2, 0), (3, 0)),
    "in_place": ((0, 0), (1, 0), (0, 0), (1, 0)),
    "keys_in_place": ((0, 0), (1, 0), (0, 0), (2, 0)),
    "values_in_place": ((0, 0), (1, 0), (2, 0), (1, 0)),
    "crossed": ((0, 0), (1, 0), (1, 0), (0, 0)),
    "keys_shifted": ((0, 0), (2, 0), (0, 16), (3, 16)),
    "values_shifted": ((0, 0), (1, 16), (3, 0), (1, 1)),
    "crossed_in_part": ((0, 0), (1, 0), (1, 40), (3, 0)),
    "one_word": ((0, 0), (2, 0), (1, -1), (4, 0)),
}


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("n", [65, 1000, 8192, 8193])
def test_sort_shared_buffers(n, layout):
    from gstex_cuda_amd import _lib

    rng = np.random.default_rng(n)
    k = rng.integers(0, 1 << 32, n).astype(np.uint32)
    k[rng.random(n) < 0.3] = 7
    v = rng.integers(0, 1 << 31, n).astype(np.uint32)
    at = [a * n + b for a, b in LAYOUTS[layout]]
    buf = torch.zeros(5 * n + 64, dtype=torch.int32, device=DEV)
    for data, o in zip((k, v), at):
        buf[o:o + n] = torch.from_numpy(data.view(np.int32)).to(DEV)
    size = _lib.lib().gstex_sort_pairs_u32_workspace_size(n)
    ws = torch.empty(size, dtype=torch.uint8, device=DEV)
    p = [buf.data_ptr() + 4 * o for o in at]
    _lib.call("gstex_sort_pairs_u32", n, 32, *p, ws.data_ptr(), size,
              torch.cuda.current_stream().cuda_stream)
    order = np.argsort(k, kind="stable")
    got = np_(buf).view(np.uint32)
    assert np.array_equal(got[at[2]:at[2] + n], k[order])
    assert np.array_equal(got[at[3]:at[3] + n], v[order])
