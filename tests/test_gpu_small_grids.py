"""The raster kernels for small tile grids (4x4 pixels a wave, four entries at
a time) against the 8x8 kernels, on the same lists: padding the id buffer past
the size rule, with bins that never reach the padding, selects the latter.
Forward outputs are equal bit for bit, gradients up to the order of float
sums."""
import dataclasses

import numpy as np
import pytest
import torch

from gpu_helpers import DEV, log, np_, project_and_bin, random_grads, raster_inputs, to_dev
from test_gpu_culling import _grads_match, _scene

pytestmark = pytest.mark.gpu

PAD = 700_000  # ids past which the 8x8 kernels run


def _render(s, pb, ids, settings, cot, masks=True, bf16=False):
    from gstex_cuda_amd import cuda as _C

    r = raster_inputs(s)
    C = s.texture.shape[1]
    tex = r["texture"].bfloat16() if bf16 else r["texture"]
    rec = _C.build_splat_records(r["means"], r["scales"], 1.0, r["quats"], r["colors"],
                                 r["opacities"], r["uv0"], r["umap"], r["vmap"],
                                 r["texture_dims"], r["viewmat"], r["c2w"], s.fx, s.fy, s.cx, s.cy)
    a = (rec, s.num_points, s.img_w, s.img_h, 16, C, settings, ids, pb["bins"], tex, r["viewmat"],
         r["c2w"], s.fx, s.fy, s.cx, s.cy, r["background"])
    out, m = _C.raster_forward(*a, wave_masks=masks)
    grads = _C.raster_backward(*a, out[5], out[6], out[7], out[8], *cot, wave_masks=m)
    return [np_(o) for o in out], [np_(g) for g in grads]


def _compare(s, settings=1 << 8, masks=True, bf16=False, rel=1e-5):
    pb = project_and_bin(s)
    cot = [to_dev(v) for v in random_grads(np.random.default_rng(3), s.img_h, s.img_w,
                                           s.texture.shape[1]).values()]
    pad = torch.zeros(PAD, dtype=torch.int32, device=DEV)
    log(f"{s.img_w}x{s.img_h} intersects {pb['num_intersects']}")
    f0, g0 = _render(s, pb, pb["ids"], settings, cot, masks, bf16)
    f1, g1 = _render(s, pb, torch.cat([pb["ids"], pad]), settings, cot, masks, bf16)
    for k, (x, y) in enumerate(zip(f0, f1)):
        assert np.array_equal(x, y, equal_nan=True), k
    for k, (x, y) in enumerate(zip(g0, g1)):
        ok, info = _grads_match(x, y, rel)
        assert ok, (k, info)


def _sized(seed, n, w, h, side=0, channels=3):
    from gstex_cuda_amd.synthetic import SceneSpec, make_scene

    return make_scene(seed=seed, spec=SceneSpec(
        num_points=n, img_w=w, img_h=h, focal=float(h), z_range=(2.0, 12.0),
        texel_side=max(side, 1), texel_budget=0 if side else 4 * n, channels=channels,
        background=(0.3, 0.1, 0.7)))


# image edges inside a 4x4, an 8x8 and a tile; one pixel; lists around the
# 64-entry batches and 256-entry steps; charts that fit the 4x4 window, its
# neighbourhood, the pool, and none of them
@pytest.mark.parametrize("n,w,h,side,channels", [
    (1, 1, 1, 1, 3), (40, 33, 18, 1, 1), (300, 130, 71, 2, 2), (900, 96, 64, 0, 3),
    (4000, 61, 77, 3, 4), (4000, 200, 150, 16, 3), (500, 120, 100, 40, 3), (20000, 64, 64, 0, 3)])
@pytest.mark.parametrize("settings", [1 << 8, (1 << 8) | (1 << 9) | (1 << 15)])
def test_small_grid_equals_8x8(n, w, h, side, channels, settings):
    _compare(_sized(n + w, n, w, h, side, channels), settings)


@pytest.mark.parametrize("masks,bf16,settings", [(False, False, 1 << 8), (True, True, 1 << 8),
                                                 (False, True, 0)])
def test_small_grid_variants(masks, bf16, settings):
    _compare(_sized(5, 1500, 150, 90), settings, masks, bf16)


@pytest.mark.parametrize("kind", ["opacity_extremes", "saturated", "thin_rotated", "tiny",
                                  "near_camera"])
def test_small_grid_hard_scenes(kind):
    _compare(_scene(kind))


@pytest.mark.parametrize("opacity", [0.0, 0.6])
def test_small_grid_copy_runs(opacity):
    # 3,000 copies of Gaussian 0 at the front of tile 0 (clipped Gaussians that
    # were counted), and 9,000 for the strides of 2,048
    for copies in (3000, 9000):
        s = _sized(9, 600, 64, 48)
        s.opacities[0, 0] = opacity
        pb = project_and_bin(s)
        ids, bins = np_(pb["ids"]), np_(pb["bins"]).copy()
        ids = np.concatenate([np.zeros(copies, np.int32), ids])
        bins[bins[:, 1] > bins[:, 0]] += copies
        bins[0] = [0, max(bins[0, 1], copies)]
        cot = [to_dev(v) for v in random_grads(np.random.default_rng(1), s.img_h, s.img_w,
                                               3).values()]
        pb = dict(pb, bins=to_dev(bins))
        f0, g0 = _render(s, pb, to_dev(ids), 1 << 8, cot)
        f1, g1 = _render(s, pb, to_dev(np.concatenate([ids, np.zeros(PAD, np.int32)])), 1 << 8,
                         cot)
        for k, (x, y) in enumerate(zip(f0, f1)):
            assert np.array_equal(x, y, equal_nan=True), k
        for k, (x, y) in enumerate(zip(g0, g1)):
            ok, info = _grads_match(x, y, 1e-5)
            assert ok, (k, info)


def test_small_grid_charts_outside_the_texture():
    s = _sized(11, 800, 100, 80)
    d = s.texture_dims.copy()
    d[::7, 2] = s.texture.shape[0]          # starts past the end
    d[1::7, 2] = -5
    d[2::7, 0] = 1 << 20                    # h w past 2^31
    d[2::7, 1] = 1 << 20
    d[3::7, 1] = 0
    _compare(dataclasses.replace(s, texture_dims=d))
