"""Culling with the blur alone (the plain kernels with the blur): an entry is
kept by its screen ellipse or its blur disc, and the outputs equal those of the
full walk bit for bit, on the scenes built to break the bounds."""
import numpy as np
import pytest

from gpu_helpers import log, random_grads
from test_gpu_culling import FWD_NAMES, GRAD_NAMES, KINDS, _grads_match, _run, _scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", KINDS)
def test_blur_culling_changes_nothing(kind):
    s = _scene(kind, (1 << 8) | (1 << 9))
    log(f"case {kind}")
    cot = random_grads(np.random.default_rng(3), s.img_h, s.img_w, s.texture.shape[1])
    f_on, g_on, _ = _run(s, True, True, cot)
    f_off, g_off, _ = _run(s, False, True, cot)
    _, g_no_masks, _ = _run(s, True, False, cot)
    for k in FWD_NAMES:
        assert np.array_equal(f_on[k], f_off[k], equal_nan=True), k
    for k in GRAD_NAMES:
        for other in (g_off, g_no_masks):
            ok, info = _grads_match(g_on[k], other[k], 1e-5)
            assert ok, (k, info)
