"""GPU parity of the raster for more than four texture channels: the texel
gradients' routes (one texel, shared quad, 3x3 / 2x3 / 3x2 windows, LDS
accumulator, direct atomics) over groups of four channels, with counts at and
off a group's end."""
import numpy as np
import pytest

from gpu_helpers import (grad_close, gpu_backward, gpu_forward, log, np_, oracle_with,
                         project_and_bin, random_grads)

pytestmark = pytest.mark.gpu


# side 0: charts of 1..16 texels a side by projected area.  16 x 16 charts of
# 5 channels overflow the LDS accumulator (1,024 values), as 8 x 8 of 64 do.
@pytest.mark.parametrize("side,channels,settings,bw", [
    (1, 5, 0, 16), (1, 8, 0, 16), (1, 64, 0, 16), (2, 6, 0, 16), (2, 9, 0, 8), (3, 12, 0, 16),
    (4, 7, 1 << 2, 16), (0, 8, 1 << 9, 16), (0, 33, 0, 16), (16, 5, 0, 16), (8, 64, 0, 5)])
def test_backward_wide_channels(oracle, side, channels, settings, bw):
    from gstex_cuda_amd.synthetic import SceneSpec, make_scene

    spec = SceneSpec(num_points=500, img_w=117, img_h=90, focal=90.0, z_range=(2.0, 8.0),
                     texel_side=max(side, 1), texel_budget=20_000 if side == 0 else 0,
                     channels=channels)
    s = make_scene(seed=side * 100 + channels, spec=spec)
    settings |= 1 << 8
    pb = project_and_bin(s, bw)
    g, _ = gpu_forward(s, pb["ids"], pb["bins"], settings=settings, bw=bw)
    sc = oracle_with(oracle, s, pb["ids"], pb["bins"], settings=settings, bw=bw)
    o = oracle.texture_forward(sc, "f64")
    assert np.mean(np.abs(np_(g["out_texture"]) - o["out_texture"]) < 1e-4) > 0.999
    grads = random_grads(np.random.default_rng(side), s.img_h, s.img_w, channels, 1e-3)
    gg = gpu_backward(s, pb["ids"], pb["bins"], g, grads, settings=settings, bw=bw)
    og = oracle.texture_backward(sc, o, grads["img"], grads["depth"], grads["reg"],
                                 grads["alpha"], grads["tex"], grads["normal"], "f64")
    # the gradients that pass through the texels (the mean's also carries the
    # float32 plane hit of edge-on splats, whatever the channel count)
    for k in ("v_texture", "v_uv0", "v_umap", "v_vmap"):
        ok, l2, frac = grad_close(np_(gg[k]), og[k])
        log("wide", side, channels, settings, bw, k, "relL2 %.2e" % l2, "frac %.4f" % frac)
        assert ok, (k, l2, frac)
