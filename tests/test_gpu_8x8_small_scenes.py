"""The 8x8 raster kernels on small scenes, which by themselves select the kernels
for small tile grids: id buffers padded past the size rule (bins never reach the
padding).  Culling on against off, with masks against without, on the scenes
built to break the bounds; and parity with the oracle."""
import numpy as np
import pytest
import torch

from gpu_helpers import (DEV, grad_close, gpu_backward, gpu_forward, log, np_, oracle_with,
                         project_and_bin, random_grads, to_dev)
from test_gpu_culling import KINDS, _grads_match, _scene
from test_gpu_small_grids import PAD, _render, _sized

pytestmark = pytest.mark.gpu

UV, BLUR = 1 << 8, 1 << 9


def _padded(ids):
    return torch.cat([ids, torch.zeros(PAD, dtype=torch.int32, device=DEV)])


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("settings", [UV, UV | BLUR])
def test_culling_changes_nothing(kind, settings):
    from gstex_cuda_amd import cuda as _C

    s = _scene(kind, settings)
    log(f"case {kind} settings={settings}")
    pb = project_and_bin(s)
    ids = _padded(pb["ids"])
    cot = [to_dev(v) for v in random_grads(np.random.default_rng(3), s.img_h, s.img_w,
                                           s.texture.shape[1]).values()]
    f_on, g_on = _render(s, pb, ids, settings, cot)
    _, g_no_masks = _render(s, pb, ids, settings, cot, masks=False)
    prev = _C.set_raster_culling(False)
    try:
        f_off, g_off = _render(s, pb, ids, settings, cot)
    finally:
        _C.set_raster_culling(prev)
    f_small, g_small = _render(s, pb, pb["ids"], settings, cot)
    for k, x in enumerate(f_on):
        assert np.array_equal(x, f_off[k], equal_nan=True), k
        assert np.array_equal(x, f_small[k], equal_nan=True), k
    for k, x in enumerate(g_on):
        for other in (g_off, g_no_masks, g_small):
            ok, info = _grads_match(x, other[k], 1e-5)
            assert ok, (k, info)


@pytest.mark.parametrize("n,w,h,side,channels", [(300, 130, 71, 2, 2), (900, 96, 64, 0, 3),
                                                 (4000, 61, 77, 3, 4), (500, 120, 100, 16, 3),
                                                 (400, 117, 90, 1, 1)])
@pytest.mark.parametrize("settings", [UV, UV | BLUR])
def test_parity(oracle, n, w, h, side, channels, settings):
    s = _sized(n, n, w, h, side, channels)
    pb = project_and_bin(s)
    ids = _padded(pb["ids"])
    f, _ = gpu_forward(s, ids, pb["bins"], settings=settings)
    sc = oracle_with(oracle, s, pb["ids"], pb["bins"], settings=settings)
    o = oracle.texture_forward(sc, "f64")
    for k in ("out_img", "out_texture", "out_normal", "final_Ts"):
        assert np.mean(np.abs(np_(f[k]) - o[k]) < 1e-4) > 0.999, k
    grads = random_grads(np.random.default_rng(side), s.img_h, s.img_w, channels, 1e-3)
    g = gpu_backward(s, ids, pb["bins"], f, grads, settings=settings)
    og = oracle.texture_backward(sc, o, grads["img"], grads["depth"], grads["reg"],
                                 grads["alpha"], grads["tex"], grads["normal"], "f64")
    # (the mean's and the scale's gradients also carry the float32 plane hit of
    # edge-on splats, whichever kernel forms it)
    for k in ("v_texture", "v_uv0", "v_umap", "v_vmap", "v_colors", "v_opacity"):
        ok, l2, frac = grad_close(np_(g[k]), og[k])
        log("8x8", n, channels, settings, k, "relL2 %.2e" % l2, "frac %.4f" % frac)
        assert ok, (k, l2, frac)
