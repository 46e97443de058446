"""A pixel with a cotangent that is not finite gives such texel gradients only to
the texels it samples: on images whose sides are not multiples of the tile, at
pixel (0, 0) and inside, on the routes of four and more channels and in the
kernels for small tile grids."""
import numpy as np
import pytest

from gpu_helpers import (gpu_backward, gpu_forward, log, np_, oracle_with, project_and_bin,
                         random_grads)
from test_gpu_texel_windows import _scene

pytestmark = pytest.mark.gpu


def _check(oracle, channels, bw, settings, bad, pixels, seed):
    s = _scene(seed, channels, bw)
    settings |= 1 << 8
    b = project_and_bin(s, bw)
    g, _ = gpu_forward(s, b["ids"], b["bins"], settings=settings, bw=bw)
    grads = random_grads(np.random.default_rng(1), s.img_h, s.img_w, channels, 1e-3)
    for i, j in pixels:
        grads["tex"][i, j, channels // 2] = bad
    got = np_(gpu_backward(s, b["ids"], b["bins"], g, grads, settings=settings, bw=bw)["v_texture"])
    sc = oracle_with(oracle, s, b["ids"], b["bins"], settings=settings, bw=bw)
    o = oracle.texture_forward(sc, "f64")
    ref = oracle.texture_backward(sc, o, grads["img"], grads["depth"], grads["reg"],
                                  grads["alpha"], grads["tex"], grads["normal"],
                                  "f64")["v_texture"]
    hit, ok = ~np.isfinite(got), np.isfinite(ref)
    log("nonfinite", channels, bw, settings, bad, "texels", int(hit.any(1).sum()), "of",
        int((~ok).any(1).sum()))
    assert hit.any() or ok.all()
    assert not (hit & ok).any()
    # the other texels are what they would be without it
    both = ok & ~hit
    err = np.abs(got - ref)[both] / np.abs(ref[ok]).max()
    assert np.mean(err < 1e-4) >= 0.999 and err.max() < 5e-2, float(err.max())


@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("channels,bw,settings", [(5, 16, 0), (8, 16, 0), (5, 5, 0), (8, 5, 0),
                                                  (4, 8, 0), (8, 16, 1 << 2), (4, 8, 1 << 2),
                                                  (6, 16, 1 << 9)])
def test_wide_channels(oracle, channels, bw, settings, bad):
    _check(oracle, channels, bw, settings, bad, [(0, 0)], channels + bw)
    _check(oracle, channels, bw, settings, bad, [(40, 50), (89, 116)], channels + bw)


@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("channels,settings", [(1, 0), (3, 0), (4, 0), (3, 1 << 9)])
def test_small_grids(oracle, channels, settings, bad):
    _check(oracle, channels, 16, settings, bad, [(40, 50), (89, 116)], channels + 40)
