"""Texel sums on the matrix instructions: charts whose quads and windows end at
the chart's edge (1xN, Nx1, 2xN, ...), for the edit (four channels and the
weight) and the gradients of more than four channels, against the oracle; and a
canvas with values that are not finite."""
import numpy as np
import pytest

from gpu_helpers import (grad_close, gpu_backward, gpu_forward, log, np_, oracle_with,
                         project_and_bin, random_grads, to_dev)
from helpers import oracle_scene, tile_bounds

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1), (1, 2), (2, 1), (1, 7), (7, 1), (2, 2), (2, 5), (3, 2), (3, 3), (4, 4), (5, 3),
          (15, 13), (16, 16)]


def _scene(seed, channels, bw):
    from gstex_cuda_amd.synthetic import SceneSpec, make_scene

    s = make_scene(seed=seed, spec=SceneSpec(num_points=400, img_w=117, img_h=90, focal=90.0,
                                             z_range=(2.0, 8.0), texel_side=2,
                                             channels=channels))
    s.block_width = bw
    rng = np.random.default_rng(seed)
    hw = np.array(SHAPES)[rng.integers(0, len(SHAPES), s.num_points)]
    n = hw[:, 0] * hw[:, 1]
    s.texture_dims = np.stack([hw[:, 0], hw[:, 1], np.cumsum(n) - n], 1).astype(np.int32)
    s.texture = rng.random((int(n.sum()), channels)).astype(np.float32)
    return s


def _edit(s, b, st, img, al, lo, hi):
    from gstex_cuda_amd import cuda as _C

    X, C = s.texture.shape
    tb = tile_bounds(s.img_w, s.img_h, s.block_width)
    return np_(_C.texture_edit(
        tb, (s.block_width, s.block_width, 1), (s.img_w, s.img_h, 1), (s.num_points, 1, C), X,
        to_dev(s.texture_dims), to_dev(img), to_dev(al), to_dev(lo), to_dev(hi), b["ids"],
        b["bins"], to_dev(s.opacities), to_dev(s.means), to_dev(s.scales), 1.0, to_dev(s.quats),
        to_dev(s.uv0), to_dev(s.umap), to_dev(s.vmap), to_dev(s.viewmat), to_dev(s.c2w), s.fx,
        s.fy, s.cx, s.cy, st, to_dev(s.background)))


@pytest.mark.parametrize("channels,bw,blur,window", [(5, 16, 0, False), (5, 8, 0, True),
                                                     (7, 5, 0, False), (5, 16, 1, True)])
def test_edit_at_chart_edges(oracle, channels, bw, blur, window):
    s = _scene(channels + bw, channels, bw)
    rng = np.random.default_rng(bw)
    shape = (s.img_h, s.img_w)
    img = rng.random(shape + (3,)).astype(np.float32)
    al = rng.random(shape).astype(np.float32)
    lo = (rng.uniform(0, 4, shape) if window else np.zeros(shape)).astype(np.float32)
    hi = (lo + 3 if window else np.full(shape, 1e3)).astype(np.float32)
    b = project_and_bin(s, bw)
    got = _edit(s, b, blur, img, al, lo, hi)
    sc = oracle_scene(oracle, s, ids_sorted=np_(b["ids"]), tile_bins=np_(b["bins"]), settings=blur)
    ref = oracle.texture_edit(sc, img, al, lo, hi, "f64")
    # as the edit's own test: float atomics in any order, float32 pair math
    for k in range(5):
        err = np.abs(got[:, k] - ref[:, k]) / np.abs(ref[:, k]).max()
        assert np.mean(err < 1e-4) >= 0.999 and err.max() < 5e-2, (k, float(err.max()))
    assert not got[:, 5:].any()


@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_edit_canvas_not_finite(oracle, bad):
    s = _scene(3, 5, 16)
    shape = (s.img_h, s.img_w)
    img = np.random.default_rng(0).random(shape + (3,)).astype(np.float32)
    al = np.ones(shape, np.float32)
    lo, hi = np.zeros(shape, np.float32), np.full(shape, 1e3, np.float32)
    img[40, 50, 1] = bad
    b = project_and_bin(s, 16)
    got = _edit(s, b, 0, img, al, lo, hi)
    sc = oracle_scene(oracle, s, ids_sorted=np_(b["ids"]), tile_bins=np_(b["bins"]), settings=0)
    ref = oracle.texture_edit(sc, img, al, lo, hi, "f64")
    hit = ~np.isfinite(got)
    assert hit[:, 1].any() and not hit[:, [0, 2, 3, 4]].any()
    assert not (hit & np.isfinite(ref)).any()  # only texels which that pixel samples
    ok = np.isfinite(ref)
    for k in range(5):
        g, r = got[ok[:, k], k], ref[ok[:, k], k]
        err = np.abs(g - r) / np.abs(r).max()
        assert np.mean(err < 1e-4) >= 0.999 and err.max() < 5e-2, (k, float(err.max()))


@pytest.mark.parametrize("channels,settings,bw", [(5, 0, 16), (8, 1 << 2, 16), (10, 0, 8),
                                                  (8, 1 << 9, 5)])
def test_wide_gradients_at_chart_edges(oracle, channels, settings, bw):
    s = _scene(channels, channels, bw)
    settings |= 1 << 8
    b = project_and_bin(s, bw)
    g, _ = gpu_forward(s, b["ids"], b["bins"], settings=settings, bw=bw)
    sc = oracle_with(oracle, s, b["ids"], b["bins"], settings=settings, bw=bw)
    o = oracle.texture_forward(sc, "f64")
    grads = random_grads(np.random.default_rng(1), s.img_h, s.img_w, channels, 1e-3)
    gg = gpu_backward(s, b["ids"], b["bins"], g, grads, settings=settings, bw=bw)
    og = oracle.texture_backward(sc, o, grads["img"], grads["depth"], grads["reg"],
                                 grads["alpha"], grads["tex"], grads["normal"], "f64")
    ok, l2, frac = grad_close(np_(gg["v_texture"]), og["v_texture"])
    log("wide edges", channels, settings, bw, "relL2 %.2e" % l2, "frac %.4f" % frac)
    assert ok, (l2, frac)


# 8x8 tiles: up to four channels on 16x16 tiles take the small-grid kernels here
@pytest.mark.parametrize("channels,settings", [(1, 0), (2, 0), (3, 0), (4, 0), (3, 1 << 2),
                                               (4, 1 << 2), (3, 1 << 9), (3, 1 << 10)])
def test_gradients_at_chart_edges(oracle, channels, settings):
    s = _scene(20 + channels, channels, 8)
    settings |= 1 << 8
    b = project_and_bin(s, 8)
    g, _ = gpu_forward(s, b["ids"], b["bins"], settings=settings, bw=8)
    sc = oracle_with(oracle, s, b["ids"], b["bins"], settings=settings, bw=8)
    o = oracle.texture_forward(sc, "f64")
    grads = random_grads(np.random.default_rng(2), s.img_h, s.img_w, channels, 1e-3)
    gg = gpu_backward(s, b["ids"], b["bins"], g, grads, settings=settings, bw=8)
    og = oracle.texture_backward(sc, o, grads["img"], grads["depth"], grads["reg"],
                                 grads["alpha"], grads["tex"], grads["normal"], "f64")
    for k in ("v_texture", "v_uv0", "v_umap", "v_vmap", "v_colors"):
        ok, l2, frac = grad_close(np_(gg[k]), og[k])
        log("edges", channels, settings, k, "relL2 %.2e" % l2, "frac %.4f" % frac)
        assert ok, (k, l2, frac)
    flat = s.texture_dims[:, 0] * s.texture_dims[:, 1] == 1
    for k in ("v_uv0", "v_umap", "v_vmap"):  # one texel: no uv gradient at all
        assert not np_(gg[k])[flat].any(), k
