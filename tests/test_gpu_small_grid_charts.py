"""The small-grid backward on charts larger than its window and pool: the same
gradients as the 8x8 kernels', and no slower where the rule selects it."""
import dataclasses

import numpy as np
import pytest
import torch

from gpu_helpers import DEV, log, project_and_bin, random_grads, raster_inputs, to_dev
from test_gpu_small_grids import PAD, _compare, _sized

pytestmark = pytest.mark.gpu


# few charts past the 4x4 window, the pool (3,072 values) and its four 16x16 charts
# a batch, among charts of one to four texels, so that the lists name few values
@pytest.mark.parametrize("n,w,h,channels,large", [(900, 96, 64, 3, (16, 40)),
                                                  (3000, 200, 150, 4, (9, 16, 31)),
                                                  (400, 64, 48, 1, (60, 5)),
                                                  (1500, 160, 90, 3, (16,))])
@pytest.mark.parametrize("settings", [1 << 8, (1 << 8) | (1 << 9)])
def test_few_large_charts(n, w, h, channels, large, settings):
    s = _sized(n, n, w, h, 1, channels)
    rng = np.random.default_rng(n)
    side = rng.integers(1, 3, n)
    big = rng.random(n) < 0.04
    side[big] = rng.choice(large, int(big.sum()))
    t = side * side
    dims = np.stack([side, side, np.cumsum(t) - t], 1).astype(np.int32)
    s = dataclasses.replace(s, texture_dims=dims,
                            texture=rng.random((int(t.sum()), channels)).astype(np.float32))
    _compare(s, settings)


def _backward_us(s):
    """Microseconds of the backward as the rule selects it, and of the 8x8 kernel."""
    from gstex_cuda_amd import cuda as _C

    pb = project_and_bin(s)
    r = raster_inputs(s)
    rec = _C.build_splat_records(r["means"], r["scales"], 1.0, r["quats"], r["colors"],
                                 r["opacities"], r["uv0"], r["umap"], r["vmap"],
                                 r["texture_dims"], r["viewmat"], r["c2w"], s.fx, s.fy, s.cx, s.cy)
    cot = [to_dev(v) for v in random_grads(np.random.default_rng(3), s.img_h, s.img_w, 3).values()]
    us = []
    for ids in (pb["ids"], torch.cat([pb["ids"], torch.zeros(PAD, dtype=torch.int32, device=DEV)])):
        a = (rec, len(s.texture_dims), s.img_w, s.img_h, 16, 3, 1 << 8, ids, pb["bins"], r["texture"],
             r["viewmat"], r["c2w"], s.fx, s.fy, s.cx, s.cy, r["background"])
        out, m = _C.raster_forward(*a, wave_masks=True)
        times = []
        for _ in range(6):
            e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
            e[0].record()
            for _ in range(10):  # back to back, so that the host is not what is timed
                _C.raster_backward(*a, out[5], out[6], out[7], out[8], *cot, wave_masks=m)
            e[1].record()
            torch.cuda.synchronize()
            times.append(e[0].elapsed_time(e[1]) * 1e2)
        us.append(sorted(times)[2])
    log("backward us, as selected and with the 8x8 kernels", us, pb["num_intersects"])
    return us


@pytest.mark.parametrize("n,side", [(20000, 16), (20000, 8), (60000, 16)])
def test_large_charts_are_not_slower(n, side):
    us = _backward_us(_sized(3, n, 637, 359, side, 3))
    assert us[0] < 1.15 * us[1] + 20


# small charts of one size gain at any count up to the rule's (150K entries here,
# 7.2M values: 422 against 209 us)
def test_small_charts_of_one_size_are_faster():
    us = _backward_us(_sized(3, 28000, 500, 300, 4, 3))
    assert us[0] < 0.8 * us[1]
