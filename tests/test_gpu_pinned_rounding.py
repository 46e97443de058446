"""The rounding of the raster backward, on a grid of 1,500 tiles (the 8x8 kernels).

Every splat lies inside one 8x8 pixel block, so one wave forms each of its sums
and the bits do not depend on the order of float atomics.  Adam divides a
gradient by its size, so sums that cancel turn another rounding of a product into
another step: the digests hold the bits that the kernels gave before charts of one
texel took a path of their own.  A change of a formula or of the compiler changes
them; then the float64 tests say whether the new values are as good."""
import dataclasses
import hashlib

import numpy as np
import pytest

from gpu_helpers import gpu_backward, gpu_forward, log, np_, project_and_bin, random_grads

pytestmark = pytest.mark.gpu

UV, BLUR, NDC, NEAREST, FLIP = 1 << 8, 1 << 9, 1 << 10, 1 << 2, 1 << 15
MIXED, FLAT = (1, 1, 2, 3, 4, 6), (1,)
# by (kinds of chart, settings, tile side)
DIGESTS = {
    (6, 256, 16): "b3e75d72c1cd6f89",
    (1, 256, 16): "09c629ef4b0757b4",
    (6, 0, 16): "31b8409b93e2bd64",
    (6, 33024, 16): "b0c2ace2aee0b07f",
    (6, 768, 16): "97b074545673e600",
    (1, 768, 16): "0039aa4ca694d485",
    (6, 1280, 16): "f8d9b9e1ff4cd904",
    (6, 1792, 16): "bd1a244a9393f5c9",
    (6, 260, 16): "ad1b8b76d58d2802",
    (6, 256, 8): "556c9e36a074d92f",
}


def one_wave_scene(sides, w=800, h=480, blocks=400, per_block=3, seed=0):
    from gstex_cuda_amd.synthetic import SceneSpec, make_scene, quat_axes_np

    rng = np.random.default_rng(seed)
    n = blocks * per_block
    s = make_scene(seed=seed, spec=SceneSpec(num_points=n, img_w=w, img_h=h, focal=400.0,
                                             texel_side=1))
    b = rng.choice((w // 8) * (h // 8), blocks, replace=False).repeat(per_block)
    px = (b % (w // 8)) * 8 + 4 + rng.uniform(-0.4, 0.4, n)
    py = (b // (w // 8)) * 8 + 4 + rng.uniform(-0.4, 0.4, n)
    z = rng.uniform(3, 9, n)
    means = np.stack([(px - s.cx) / s.fx * z, (py - s.cy) / s.fy * z, z], 1).astype(np.float32)
    # up to 0.8 pixels: alpha reaches 1/255 within 3.1 pixels of the block's centre
    sc = (rng.uniform(0.35, 0.8, (n, 2)) * (z / s.fx)[:, None]).astype(np.float32)
    a1, a2 = quat_axes_np(s.quats)[:2]
    side = np.array(sides)[rng.integers(0, len(sides), n)]
    t = side * side
    return dataclasses.replace(
        s, means=means, scales=np.concatenate([sc, np.full((n, 1), 1e-5, np.float32)], 1),
        umap=(a1 / (6.0 * sc[:, :1])).astype(np.float32).reshape(n, 1, 3),
        vmap=(a2 / (6.0 * sc[:, 1:])).astype(np.float32).reshape(n, 1, 3),
        texture_dims=np.stack([side, side, np.cumsum(t) - t], 1).astype(np.int32),
        texture=rng.random((int(t.sum()), 3)).astype(np.float32),
        opacities=rng.uniform(0.2, 0.95, (n, 1)).astype(np.float32))


def digest(sides, settings, bw):
    s = one_wave_scene(sides)
    b = project_and_bin(s, bw)
    f, _ = gpu_forward(s, b["ids"], b["bins"], settings=settings, bw=bw)
    cot = random_grads(np.random.default_rng(3), s.img_h, s.img_w, 3)
    g = gpu_backward(s, b["ids"], b["bins"], f, cot, settings=settings, bw=bw)
    d = hashlib.sha256()
    for k in sorted(f):
        d.update(np.ascontiguousarray(np_(f[k])).tobytes())
    for k in sorted(g):
        d.update(np.ascontiguousarray(np_(g[k])).tobytes())
    return d.hexdigest()[:16]


CASES = [(MIXED, UV, 16), (FLAT, UV, 16), (MIXED, 0, 16), (MIXED, UV | FLIP, 16),
         (MIXED, UV | BLUR, 16), (FLAT, UV | BLUR, 16), (MIXED, UV | NDC, 16),
         (MIXED, UV | BLUR | NDC, 16), (MIXED, UV | NEAREST, 16), (MIXED, UV, 8)]


@pytest.mark.parametrize("sides,settings,bw", CASES)
def test_bits(sides, settings, bw):
    got = digest(sides, settings, bw)
    log("digest", len(sides), settings, bw, got)
    assert got == DIGESTS[len(sides), settings, bw]
