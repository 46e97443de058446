"""Timed cases of the textured-2DGS path, through its public entry points.

A case is a dict of plain values.  ``kind`` says which entry point a program
calls:

  render    one view without gradients: projection, (SH colours), rasterise
  autograd  the same with the backward to every parameter, as a torch program
            that uses ``texture_gaussians`` as a layer runs it
  step      ``RenderStep``: one training view, forward + L2 loss + backward;
            with ``regularised`` also the distortion and normal terms
  views     ``MultiViewStep``: a captured batch of views, gradients summed
  train     ``TrainStep``: preprocessing, render, example loss, backward, Adam
  sh        SH colours of all Gaussians, forward and coefficient gradient
  sample    bilinear queries into the texel charts, forward and texel gradient
  edit      an edit canvas splatted onto the texel charts
  bin       intersect keys, their sort and the tile bin edges

Scenes follow ``gstex_cuda_amd.synthetic``'s distributions (means xy U[-1, 1],
z U[2, 20], or U[2, 6] for scenes of up to 5,000 Gaussians; log-scales
U[-4, -2]; random rotations; opacities sigmoid(N(0, 1)); charts of 1x1 to
16x16 texels by projected area, or of one fixed side), generated on the GPU
from the seed.
"""
import math

import numpy as np
import torch

from gstex_cuda_amd import get_aabb_2d, sh as sh_ops, texture, texture_edit, texture_sample, utils
from gstex_cuda_amd.pipeline import Camera, MultiViewStep, RenderStep
from gstex_cuda_amd.train import TrainStep

UV_GRAD, BLUR = 1 << 8, 1 << 9
LR, EPS = 1e-2, 1e-8


def _view(kind, n, width, height, **more):
    c = dict(kind=kind, n=n, width=width, height=height, channels=3, side=0, texels=4 * n, sh=-1,
             bf16=False, block=16, settings=UV_GRAD)
    c.update(more)
    return c


def listed():
    return [
        # the smallest call: a 256x256 preview of 1,000 Gaussians
        dict(_view("render", 1000, 256, 256, side=4, texels=0), name="preview_256_1k"),
        # a small training view of ragged size through autograd
        dict(_view("autograd", 20011, 637, 359), name="autograd_637x359_20k"),
        # feature textures (more channels than colour) with the blur option
        dict(_view("autograd", 50000, 800, 600, channels=8, texels=150000,
                   settings=UV_GRAD | BLUR), name="features_8ch_blur_50k"),
        # a viewer's frame: full HD, 500k Gaussians, SH degree 3, blur
        dict(_view("render", 500000, 1920, 1080, sh=3, texels=2000000,
                   settings=UV_GRAD | BLUR), name="viewer_1080p_500k"),
        # the benchmark's training view
        dict(_view("step", 500000, 1920, 1080, sh=3, texels=2000000, regularised=False),
             name="step_1080p_500k"),
        # untextured Gaussians (one texel each) with the regularised loss
        dict(_view("step", 1000000, 1600, 1200, side=1, texels=0, regularised=True),
             name="step_1600x1200_1m_untextured"),
        # the trainer of the example: raw parameters, Adam on every tensor
        dict(_view("train", 100000, 960, 540, texels=400000), name="train_960x540_100k"),
        # the largest: a batch of eight full HD views of 3M Gaussians, bfloat16 storage
        dict(_view("views", 3000000, 1920, 1080, sh=3, texels=8000000, bf16=True, views=8,
                   orbit=False), name="batch_8x1080p_3m_bf16"),
        # SH colours alone
        dict(kind="sh", n=500000, sh=3, bf16=False, name="sh3_500k"),
        # texel queries, as a texture bake or a regulariser over texels makes them
        dict(kind="sample", n=500000, queries=4000000, side=0, texels=2000000, channels=3,
             name="sample_4m"),
        # an edit painted on one full HD frame
        dict(_view("edit", 500000, 1920, 1080, texels=2000000, channels=5, window=False),
             name="edit_1080p_500k"),
        # the reference-shaped keys, sort and edges of one frame
        dict(kind="bin", n=300000, width=1920, height=1080, block=16, name="bin_1080p_300k"),
    ]


# relative frequencies of the drawn kinds
_KINDS = ("render", "render", "autograd", "autograd", "autograd", "step", "step", "views", "train",
          "sh", "sample", "edit", "bin")


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(_KINDS)
    if kind == "sh":
        return dict(kind=kind, n=_log_int(rng, 1000, 2000000), sh=rng.randrange(5),
                    bf16=rng.random() < 0.3)
    n = _log_int(rng, 1000, 1000000)
    side = rng.choice((0, 0, 0, 1, 4))
    if kind == "sample":
        return dict(kind=kind, n=n, queries=_log_int(rng, 1000, 16000000), side=side,
                    texels=0 if side else 4 * n, channels=rng.choice((1, 3, 3, 3, 4, 8)))
    width, height = _log_int(rng, 128, 1920), _log_int(rng, 128, 1080)
    block = rng.choice((16, 16, 16, 16, 8))
    if kind == "bin":
        return dict(kind=kind, n=n, width=width, height=height, block=block)
    # up to 8 texels a Gaussian
    c = _view(kind, n, width, height, side=side, texels=0 if side else int(n * rng.uniform(2, 8)),
              block=block, sh=rng.choice((-1, -1, 0, 1, 2, 3, 3)))
    if kind in ("render", "autograd"):
        c["channels"] = rng.choice((1, 3, 3, 3, 4, 8, 16))
        c["settings"] = UV_GRAD | rng.choice((0, 0, BLUR))
    if kind in ("render", "step"):
        c["bf16"] = rng.random() < 0.3
    if kind == "step":
        c["regularised"] = rng.random() < 0.5
    if kind == "train":
        c["sh"] = rng.choice((-1, 3))
    if kind == "views":
        c.update(n=_log_int(rng, 10000, 500000), views=rng.randrange(2, 9), sh=3,
                 orbit=rng.random() < 0.5, bf16=rng.random() < 0.5)
        c["texels"] = 0 if side else 4 * c["n"]
    if kind == "edit":
        c.update(channels=5, window=rng.random() < 0.5, sh=-1)
    return c


# ------------------------------------------------------------------ inputs
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _axes(q):
    w, x, y, z = q.unbind(-1)
    return (torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y + w * z), 2 * (x * z - w * y)], -1),
            torch.stack([2 * (x * y - w * z), 1 - 2 * (x * x + z * z), 2 * (y * z + w * x)], -1),
            torch.stack([2 * (x * z + w * y), 2 * (y * z - w * x), 1 - 2 * (x * x + y * y)], -1))


def _geometry(case, g):
    """Means, scales and rotations (float32) of the scene."""
    n, kw = case["n"], dict(device="cuda", generator=g)
    far = 6.0 if n <= 5000 else 20.0
    means = torch.rand((n, 3), **kw)
    means[:, :2] = 2 * means[:, :2] - 1
    means[:, 2] = 2 + (far - 2) * means[:, 2]
    scales = torch.exp(2 * torch.rand((n, 3), **kw) - 4)
    scales[:, 2] = 1e-5 * scales[:, :2].mean(1)
    quats = torch.randn((n, 4), **kw)
    quats = quats / quats.norm(dim=1, keepdim=True)
    return dict(means=means, scales=scales, quats=quats)


def _area(p):
    """Projected area of the +-3 sigma corners' box, at unit focal length."""
    m, s = p["means"].double(), p["scales"].double()
    a1, a2, _ = _axes(p["quats"].double())
    px = []
    for i in (3, -3):
        for j in (3, -3):
            c = m + i * s[:, :1] * a1 + j * s[:, 1:2] * a2
            px.append(c[:, :2] / c[:, 2:].clamp(min=0.01))
    px = torch.stack(px, 1)
    return (px.amax(1) - px.amin(1)).prod(1)


def _charts(case, p):
    """(n, 3) int32 rows (h, w, start): charts of one fixed side, or square
    ones of 1 to 16 texels a side, their texels in proportion to the projected
    area.  The sides are those of one scene of the case, given to this scene's
    Gaussians by the rank of their areas, so that the texel count is the
    case's and not the seed's."""
    n = case["n"]
    if case["side"]:
        side = torch.full((n,), case["side"], dtype=torch.int64, device="cuda")
    else:
        model = torch.sort(_area(_geometry(case, _generator(0)))).values
        model = torch.sqrt(case["texels"] * model / model.sum()).round().clamp(1, 16).long()
        side = torch.empty_like(model)
        side[torch.argsort(_area(p))] = model
    hw = side * side
    return torch.stack([side, side, torch.cumsum(hw, 0) - hw], 1).to(torch.int32), int(hw.sum())


def _scene(case, seed):
    """Render inputs (reference layouts) of a case, float32."""
    g = _generator(seed)
    kw = dict(device="cuda", generator=g)
    n = case["n"]
    p = _geometry(case, g)
    a1, a2, _ = _axes(p["quats"])
    p["umap"] = (a1 / (6 * p["scales"][:, :1])).reshape(n, 1, 3)
    p["vmap"] = (a2 / (6 * p["scales"][:, 1:2])).reshape(n, 1, 3)
    p["uv0"] = torch.full((n, 1, 2), 0.5, device="cuda")
    p["opacities"] = torch.sigmoid(torch.randn((n, 1), **kw))
    p["texture_dims"], x = _charts(case, p)
    p["texture"] = torch.rand((x, case["channels"]), **kw)
    if case["sh"] >= 0:
        p["sh_coeffs"] = 0.1 * torch.randn((n, (case["sh"] + 1) ** 2, 3), **kw)
    else:
        p["colors"] = torch.rand((n, 3), **kw)
    if case["bf16"]:
        for k in ("texture", "sh_coeffs"):
            if k in p:
                p[k] = p[k].bfloat16()
    return p, g


def _camera(c2w, width, height):
    """A pinhole camera at the row-major 4x4 pose c2w, focal length = height."""
    up = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda()  # noqa: E731
    return Camera(viewmat=up(np.linalg.inv(c2w)), c2w=up(c2w), fx=float(height), fy=float(height),
                  cx=width / 2, cy=height / 2, img_h=height, img_w=width)


def _poses(case, seed):
    """Camera poses of a batch: around the identity (up to 6 degrees and 0.15
    a coordinate), or on a sphere of radius 8 looking at the origin."""
    rng = np.random.default_rng(seed)
    poses = []
    for _ in range(case["views"]):
        c2w = np.eye(4)
        if case["orbit"]:
            eye = rng.standard_normal(3)
            eye *= 8 / np.linalg.norm(eye)
            z = -eye / 8
            x = np.cross(z, [0.0, 1.0, 0.0] if abs(z[1]) < 0.95 else [1.0, 0.0, 0.0])
            x /= np.linalg.norm(x)
            c2w[:3, 0], c2w[:3, 1], c2w[:3, 2], c2w[:3, 3] = x, np.cross(z, x), z, eye
        else:
            a = rng.standard_normal(3)
            a /= np.linalg.norm(a)
            t = math.radians(rng.uniform(-6, 6))
            k = np.array([[0, -a[2], a[1]], [a[2], 0, -a[0]], [-a[1], a[0], 0]])
            c2w[:3, :3] = np.eye(3) + math.sin(t) * k + (1 - math.cos(t)) * (k @ k)
            c2w[:3, 3] = rng.uniform(-0.15, 0.15, 3)
        poses.append(c2w)
    return poses


def _targets(case, g, count=1):
    shape = (case["height"], case["width"], 3)
    return [torch.rand(shape, device="cuda", generator=g) for _ in range(count)]


def _cotangents(case, g):
    """Cotangents of the six outputs, of the size a mean over the pixels gives."""
    h, w = case["height"], case["width"]
    rnd = lambda *s: torch.randn(s, device="cuda", generator=g) / (h * w)  # noqa: E731
    return [rnd(h, w, 3), rnd(h, w), rnd(h, w), rnd(h, w), rnd(h, w, case["channels"]),
            rnd(h, w, 3)]


def _raw(p):
    """The trainer's raw parameters of a scene."""
    s = p["scales"].double()
    n = s.shape[0]
    logit = lambda t: torch.logit(t.double().clamp(1e-4, 1 - 1e-4)).float()  # noqa: E731
    mapping = torch.zeros((n, 1, 4), device="cuda")
    mapping[:, 0, :2] = p["uv0"][:, 0]
    mapping[:, 0, 2] = torch.log(1 / (6 * torch.sqrt(s[:, 0] * s[:, 1]))).float()
    raw = dict(means=p["means"].clone(), log_scales=torch.log(s).float(), quats=p["quats"].clone(),
               mapping=mapping, opacity_logits=logit(p["opacities"]),
               texture_logits=logit(p["texture"]))
    if "sh_coeffs" in p:
        raw["sh_coeffs"] = p["sh_coeffs"].clone()
    else:
        raw["rgb_logits"] = logit(p["colors"])
    return raw


_LEAVES = ("means", "scales", "quats", "opacities", "uv0", "umap", "vmap", "texture", "sh_coeffs",
           "colors")


def _sh_inputs(case, seed):
    g = _generator(seed)
    n, d = case["n"], (case["sh"] + 1) ** 2
    dirs = torch.randn((n, 3), device="cuda", generator=g)
    coeffs = 0.1 * torch.randn((n, d, 3), device="cuda", generator=g)
    v = torch.randn((n, 3), device="cuda", generator=g)
    return dirs, coeffs.bfloat16() if case["bf16"] else coeffs, v


def _sample_inputs(case, seed):
    g = _generator(seed)
    q, c = case["queries"], case["channels"]
    dims, x = _charts(case, _geometry(case, g))
    which = torch.randint(0, case["n"], (q,), device="cuda", generator=g)
    uvs = torch.rand((q, 2), device="cuda", generator=g)
    tex = torch.rand((x, c), device="cuda", generator=g)
    v = torch.randn((q, c), device="cuda", generator=g)
    return dims[which].contiguous(), uvs, tex, v


def _edit_inputs(case, g):
    """The canvas, its alpha and the per-pixel depth window."""
    shape = (case["height"], case["width"])
    img = torch.rand(shape + (3,), device="cuda", generator=g)
    alpha = torch.rand(shape, device="cuda", generator=g)
    lo, hi = torch.zeros(shape, device="cuda"), torch.full(shape, 1000.0, device="cuda")
    if case["window"]:
        lo = 2 + 3 * torch.rand(shape, device="cuda", generator=g)
        hi = lo + 4
    return img, alpha, lo, hi


def prepare(case, seed):
    kind = case["kind"]
    if kind == "sh":
        dirs, coeffs, v = _sh_inputs(case, seed)
        return dict(case=case, dirs=dirs, coeffs=coeffs.requires_grad_(True), v=v)
    if kind == "sample":
        dims, uvs, tex, v = _sample_inputs(case, seed)
        return dict(case=case, dims=dims, uvs=uvs, tex=tex.requires_grad_(True), v=v)
    if kind == "bin":
        # one scene's screen boxes in an order and at depths of the seed's, so
        # that the number of intersects is the case's
        p, g = _geometry(case, _generator(0)), _generator(seed)
        cam = _camera(np.eye(4), case["width"], case["height"])
        cen, ext, _, tiles = get_aabb_2d.project_gaussians(
            p["means"], p["scales"], 1.0, p["quats"], cam.viewmat, (cam.fx, cam.fy, cam.cx, cam.cy),
            cam.img_h, cam.img_w, case["block"])
        at = torch.randperm(case["n"], device="cuda", generator=g)
        dep = 2 + 18 * torch.rand(case["n"], device="cuda", generator=g)
        return dict(case=case, cam=cam, centers=cen[at], extents=ext[at], depths=dep,
                    tiles=tiles[at])
    p, g = _scene(case, seed)
    if kind == "views":
        cams = [_camera(c, case["width"], case["height"]) for c in _poses(case, seed)]
        mv = MultiViewStep(p, cams, _targets(case, g, case["views"]), block_width=case["block"],
                           settings=case["settings"], sh_degree=case["sh"])
        mv.capture()
        return dict(case=case, mv=mv)
    cam = _camera(np.eye(4), case["width"], case["height"])
    state = dict(case=case, cam=cam)
    if kind == "step":
        state["target"] = _targets(case, g)[0]
        state["step"] = RenderStep(p, cam, block_width=case["block"], settings=case["settings"],
                                   sh_degree=case["sh"])
    elif kind == "train":
        state["step"] = TrainStep(_raw(p), p["texture_dims"], cam, _targets(case, g)[0], lr=LR,
                                  eps=EPS, train_mapping=True, block_width=case["block"],
                                  settings=case["settings"], sh_degree=case["sh"])
    else:
        if kind == "edit":
            state["edit"] = _edit_inputs(case, g)
        elif kind == "autograd":
            state["cots"] = _cotangents(case, g)
            for k in _LEAVES:
                if k in p:
                    p[k].requires_grad_(True)
        state["p"] = p
        state["background"] = torch.zeros(3, device="cuda")
    return state


# ------------------------------------------------------------------ passes
def _project(s):
    c, p, cam = s["case"], s["p"], s["cam"]
    return get_aabb_2d.project_gaussians(
        p["means"].detach(), p["scales"].detach(), 1.0, p["quats"].detach(), cam.viewmat,
        (cam.fx, cam.fy, cam.cx, cam.cy), cam.img_h, cam.img_w, c["block"])


def _rasterise(s):
    c, p, cam = s["case"], s["p"], s["cam"]
    cen, ext, dep, tiles = _project(s)
    if "sh_coeffs" in p:
        dirs = p["means"].detach() - cam.c2w[:3, 3]
        colors = sh_ops.spherical_harmonics(c["sh"], dirs, p["sh_coeffs"])
    else:
        colors = p["colors"]
    return texture.texture_gaussians(
        (c["n"], 1, c["channels"]), p["texture_dims"], cen, ext, dep, tiles, colors,
        p["opacities"], p["means"], p["scales"], 1.0, p["quats"], p["uv0"], p["umap"], p["vmap"],
        p["texture"], cam.viewmat, cam.c2w, cam.fx, cam.fy, cam.cx, cam.cy, cam.img_h, cam.img_w,
        c["block"], c["settings"], background=s["background"])


_OUT = ("img", "depth", "reg", "alpha", "texture", "normal")


def run(state):
    s, c = state, state["case"]
    kind = c["kind"]
    if kind == "render":
        with torch.no_grad():
            return dict(zip(_OUT, _rasterise(s)))
    if kind == "autograd":
        out = _rasterise(s)
        names = [k for k in _LEAVES if k in s["p"]]
        grads = torch.autograd.grad(out, [s["p"][k] for k in names], s["cots"])
        return dict(zip(_OUT, out), **{"v_" + k: v for k, v in zip(names, grads)})
    if kind == "step":
        r = s["step"]
        (r.regularised_step if c["regularised"] else r.step)(s["target"])
        return dict(r.grads, img=r.out_img, depth=r.out_depth, reg=r.out_reg,
                    texture=r.out_texture, normal=r.out_normal, final_Ts=r.final_Ts)
    if kind == "views":
        mv = s["mv"]
        mv.replay()
        return dict(mv.grads, imgs=[v.out_img for v in mv.views],
                    textures=[v.out_texture for v in mv.views])
    if kind == "train":
        t = s["step"]
        t.step()
        r = t.render
        return dict({"raw_" + k: v for k, v in t.raw.items()}, texture=r.out_texture,
                    normal=r.out_normal, reg=r.out_reg)
    if kind == "sh":
        colors = sh_ops.spherical_harmonics(c["sh"], s["dirs"], s["coeffs"])
        return dict(colors=colors, v_coeffs=torch.autograd.grad(colors, s["coeffs"], s["v"])[0])
    if kind == "sample":
        out = texture_sample.texture_sample((c["n"], 1, c["channels"]), s["dims"], s["tex"],
                                            s["uvs"])
        return dict(out=out, v_texture=torch.autograd.grad(out, s["tex"], s["v"])[0])
    if kind == "bin":
        cam = s["cam"]
        bw = c["block"]
        bounds = ((cam.img_w + bw - 1) // bw, (cam.img_h + bw - 1) // bw, 1)
        m, cum = utils.compute_cumulative_intersects(s["tiles"])
        return list(utils.bin_and_sort_gaussians(c["n"], m, s["centers"], s["extents"],
                                                 s["depths"], cum, bounds, bw))
    p, cam = s["p"], s["cam"]
    cen, ext, dep, tiles = _project(s)
    img, alpha, lo, hi = s["edit"]
    return texture_edit.texture_edit(
        (c["n"], 1, c["channels"]), p["texture_dims"], img, alpha, lo, hi, cen, ext, dep, tiles,
        p["opacities"], p["means"], p["scales"], 1.0, p["quats"], p["uv0"], p["umap"], p["vmap"],
        cam.viewmat, cam.c2w, cam.fx, cam.fy, cam.cx, cam.cy, cam.img_h, cam.img_w, c["block"],
        c["settings"] & BLUR and 1, background=s["background"])


# ------------------------------------------------------------------ unavoidable work
def work(case):
    """Bytes of one pass with each input read once and each output written
    once.  The arithmetic per (pixel, Gaussian) pair depends on the data and
    is left out."""
    kind, n = case["kind"], case["n"]
    if kind == "sh":
        d = 3 * (case["sh"] + 1) ** 2 * (2 if case["bf16"] else 4)
        return dict(bytes=n * (12 + d + 12 + 12 + d), flops=n * 12 * (case["sh"] + 1) ** 2)
    texels = case.get("texels") or n * case.get("side", 0) ** 2
    if kind == "sample":
        q, c = case["queries"], case["channels"]
        return dict(bytes=2 * q * (12 + 8) + 8 * q * c + 8 * texels * c, flops=16.0 * q * c)
    if kind == "bin":
        # about one intersect per 0.5 (tile side / splat size)^2: at least one per Gaussian
        return dict(bytes=n * 28 + n * 24.0, flops=0)
    pixels, c = case["width"] * case["height"], case["channels"]
    e = 2 if case["bf16"] else 4
    colour = 12 * (case["sh"] + 1) ** 2 * e / 4 if case["sh"] >= 0 else 12
    shape = 12 + 12 + 16 + 4 + 32 + 12  # means, scales, quats, opacity, uv maps, texture_dims
    inputs = n * (shape + colour) + texels * c * e
    grads = n * (76 + colour * 4 / e) + texels * c * 4
    out = pixels * 4 * (9 + c)
    if kind == "render":
        return dict(bytes=inputs + out, flops=0)
    if kind == "autograd":
        return dict(bytes=inputs + 2 * out + grads, flops=0)
    if kind == "step":
        return dict(bytes=inputs + out + pixels * 12 + grads, flops=0)
    if kind == "views":
        return dict(bytes=inputs + case["views"] * (out + pixels * 12) + grads, flops=0)
    if kind == "train":
        # parameters and both moments, read and written
        return dict(bytes=6 * (n * (60 + colour) + texels * c * 4) + out + pixels * 12, flops=0)
    return dict(bytes=n * shape + pixels * 24 + texels * c * 4, flops=0)


# ------------------------------------------------------------------ 64-bit values
# A dense float64 restatement of the path.  Per chunk of tiles every (list
# entry, pixel) pair is tested without gradients; the pairs that composite are
# packed per pixel, and only those run through the differentiable formulas.
T_NEAR, T_FAR, MOST_PAIRS = 0.01, 1000.0, 8.0e9


class _Lists:
    """Tile lists of one view: Gaussians by depth in every tile of their rectangle."""

    def __init__(self, p, cam, bw):
        vm = cam.viewmat.double()
        m, s = p["means"], p["scales"]
        pv = m @ vm[:3, :3].T + vm[:3, 3]
        a1, a2, _ = _axes(p["quats"])
        pix = []
        for i in (3, -3):
            for j in (3, -3):
                c = (m + i * s[:, :1] * a1 + j * s[:, 1:2] * a2) @ vm[:3, :3].T + vm[:3, 3]
                w = c[:, 2].clamp(min=T_NEAR) + 1e-6
                pix.append(torch.stack([c[:, 0] / w * cam.fx + cam.cx,
                                        c[:, 1] / w * cam.fy + cam.cy], 1))
        pix = torch.stack(pix, 1)
        lim = torch.tensor([-(-cam.img_w // bw), -(-cam.img_h // bw)], device="cuda")
        zero = torch.zeros_like(lim)
        cen, ext = (pix.amax(1) + pix.amin(1)) / 2, (pix.amax(1) - pix.amin(1)) / 2
        lo = torch.minimum(torch.maximum(torch.trunc((cen - ext) / bw).long(), zero), lim)
        hi = torch.minimum(torch.maximum(torch.trunc((cen + ext) / bw + 1).long(), zero), lim)
        wh = (hi - lo).clamp(min=0) * (pv[:, 2:] > T_NEAR)
        cnt = wh[:, 0] * wh[:, 1]
        order = torch.argsort(pv[:, 2].float(), stable=True)
        gs = torch.repeat_interleave(order, cnt[order])
        first = torch.cumsum(cnt[order], 0) - cnt[order]
        k = torch.arange(gs.numel(), device="cuda") - torch.repeat_interleave(first, cnt[order])
        tile = (lo[gs, 1] + k // wh[gs, 0]) * lim[0] + lo[gs, 0] + k % wh[gs, 0]
        tile, at = torch.sort(tile, stable=True)
        self.ids = gs[at]
        self.tx, self.tiles = int(lim[0]), int(lim[0] * lim[1])
        edges = torch.searchsorted(tile, torch.arange(self.tiles + 1, device="cuda"))
        self.start, self.count = edges[:-1], edges[1:] - edges[:-1]


def _pick(p, gid, names):
    """Rows gid of the named parameters: the backward is an index add."""
    flat = gid.reshape(-1)
    return [p[k].reshape(p[k].shape[0], -1).index_select(0, flat).reshape(*gid.shape, -1)
            for k in names]


def _ray(cam, px, py):
    c2w = cam.c2w.double()
    d = torch.stack([(px + 0.5 - cam.cx) / cam.fx, (py + 0.5 - cam.cy) / cam.fy,
                     torch.ones_like(px)], -1) @ c2w[:3, :3].T
    d = d / d.norm(dim=-1, keepdim=True)
    return d, d @ cam.viewmat.double()[2, :3]


def _alpha(p, cam, gid, px, py, ray, blur):
    """t, hit offset and alpha of pairs; gid (..., K) against pixels (..., 1)."""
    m, s, q, o = _pick(p, gid, ("means", "scales", "quats", "opacities"))
    a1, a2, a3 = _axes(q)
    mo = m - cam.c2w.double()[:3, 3]
    r = ray.unsqueeze(-2)
    den = (a3 * r).sum(-1)
    den = torch.where(den.abs() < 1e-6, torch.where(den < 0, -1e-6, 1e-6).to(den), den)
    t = (a3 * mo).sum(-1) / den
    d = t.unsqueeze(-1) * r - mo
    sig = 0.5 * (((d * a1).sum(-1) / s[..., 0]) ** 2 + ((d * a2).sum(-1) / s[..., 1]) ** 2)
    e = torch.exp(-sig)
    if blur:
        vm = cam.viewmat.double()
        pv = m @ vm[:3, :3].T + vm[:3, 3]
        w = pv[..., 2] + 1e-6
        sb = ((pv[..., 0] / w * cam.fx + cam.cx - px - 0.5) ** 2 +
              (pv[..., 1] / w * cam.fy + cam.cy - py - 0.5) ** 2)
        e = torch.where(sb < sig, torch.exp(-sb), e)
    alpha = (o[..., 0] * e).clamp(max=0.99)
    return t, d, a3, alpha, (t < T_NEAR) | (t > T_FAR) | (alpha < 1 / 255)


def _taps(p, gid, d):
    """Texel rows of pairs (near, far in v, far in u, far in both) and the
    fractions along u and v."""
    uv0, um, vm = _pick(p, gid, ("uv0", "umap", "vmap"))
    dims = p["texture_dims"].long()[gid]
    ft, lo, hi = [], [], []
    for k, mp in enumerate((um, vm)):
        u = uv0[..., k] + (d * mp).sum(-1)
        # the gradient passes the clamp unchanged
        x = dims[..., k] * (u + (u.detach().clamp(0, 1) - u.detach()))
        i = torch.trunc(x.detach())
        ft.append(x - i)
        lo.append(torch.minimum(i.long(), dims[..., k] - 1))
        hi.append(torch.minimum(i.long() + 1, dims[..., k] - 1))
    (fu, fv), w, st = ft, dims[..., 1], dims[..., 2]
    return [st + lo[0] * w + lo[1], st + lo[0] * w + hi[1], st + hi[0] * w + lo[1],
            st + hi[0] * w + hi[1]], fu, fv


def _composited(p, cam, lists, bw, blur):
    """Per chunk of tiles: pixel coordinates (M,), the composited Gaussians of
    each (M, K) in depth order, and which of the K are there (M, K)."""
    dev = dict(device="cuda")
    pl = torch.arange(bw * bw, **dev)
    order = torch.argsort(lists.count)
    counts = lists.count[order].tolist()
    i = 0
    while i < len(counts):
        j = i
        while j < len(counts) and (j == i or (j - i + 1) * max(counts[j], 1) * bw * bw < 16e6):
            j += 1
        tiles, length = order[i:j], max(counts[j - 1], 1)
        px, py = (tiles % lists.tx * bw)[:, None] + pl % bw, (tiles // lists.tx * bw)[:, None] + pl // bw
        ok = (px < cam.img_w) & (py < cam.img_h)
        k = torch.arange(length, **dev)
        there = k < lists.count[tiles][:, None]
        at = (lists.start[tiles][:, None] + k).clamp(max=max(lists.ids.numel() - 1, 0))
        gid = lists.ids[at] if lists.ids.numel() else torch.zeros_like(at)
        # (tile, pixel, entry)
        fx, fy = px.double(), py.double()
        ray, _ = _ray(cam, fx, fy)
        _, _, _, alpha, skip = _alpha_tiles(p, cam, gid, fx, fy, ray, blur)
        live = there[:, None, :] & ok[:, :, None]
        f = torch.where(skip | ~live, 1.0, 1 - alpha)
        t = torch.cat([torch.ones_like(f[..., :1]), torch.cumprod(f, -1)[..., :-1]], -1)
        stop = torch.cumsum(((t * (1 - alpha) <= 1e-4) & live).int(), -1) > 0
        take = live & ~skip & ~stop
        b, q, e = take.nonzero(as_tuple=True)
        num = take.sum(-1)
        keep = ok.reshape(-1)
        most = max(int(num.max()), 1)
        slot = torch.cumsum(take.int(), -1)[b, q, e] - 1
        ids = torch.zeros((*num.shape, most), dtype=torch.int64, **dev)
        ids[b, q, slot] = gid[b, e]
        have = torch.arange(most, **dev) < num[..., None]
        ids, have = ids.reshape(-1, most)[keep], have.reshape(-1, most)[keep]
        px, py = px.reshape(-1)[keep], py.reshape(-1)[keep]
        per = max(1, int(2e6) // most)
        for a in range(0, px.numel(), per):
            yield px[a:a + per], py[a:a + per], ids[a:a + per], have[a:a + per]
        i = j


def _alpha_tiles(p, cam, gid, px, py, ray, blur):
    """_alpha for all pixels of tiles against the tiles' entries, without the
    intermediate vectors of every pair."""
    m, s, q, o = _pick(p, gid, ("means", "scales", "quats", "opacities"))
    a1, a2, a3 = _axes(q)
    mo = m - cam.c2w.double()[:3, 3]
    dot = lambda a: sum(ray[:, :, None, k] * a[:, None, :, k] for k in range(3))  # noqa: E731
    den = dot(a3)
    den = torch.where(den.abs() < 1e-6, torch.where(den < 0, -1e-6, 1e-6).to(den), den)
    t = (a3 * mo).sum(-1)[:, None] / den
    l1 = (t * dot(a1) - (mo * a1).sum(-1)[:, None]) / s[:, None, :, 0]
    l2 = (t * dot(a2) - (mo * a2).sum(-1)[:, None]) / s[:, None, :, 1]
    sig = 0.5 * (l1 * l1 + l2 * l2)
    e = torch.exp(-sig)
    if blur:
        vm = cam.viewmat.double()
        pv = m @ vm[:3, :3].T + vm[:3, 3]
        w = pv[..., 2] + 1e-6
        sb = (((pv[..., 0] / w * cam.fx + cam.cx)[:, None] - px[..., None] - 0.5) ** 2 +
              ((pv[..., 1] / w * cam.fy + cam.cy)[:, None] - py[..., None] - 0.5) ** 2)
        e = torch.where(sb < sig, torch.exp(-sb), e)
    alpha = (o[..., 0][:, None] * e).clamp(max=0.99)
    return t, None, None, alpha, (t < T_NEAR) | (t > T_FAR) | (alpha < 1 / 255)


def _dense(p, cam, bw, settings, loss):
    """The six outputs as float64 images; with ``loss`` (a function of a
    chunk's outputs and its pixels), gradients accumulate in the leaves."""
    h, w, c = cam.img_h, cam.img_w, p["texture"].shape[1]
    with torch.no_grad():
        lists = _Lists(p, cam, bw)
        if lists.ids.numel() * bw * bw > MOST_PAIRS:
            return None
    z = dict(dtype=torch.float64, device="cuda")
    out = [torch.zeros(s, **z) for s in ((h, w, 3), (h, w), (h, w), (h, w), (h, w, c), (h, w, 3))]
    chunks = _composited({k: v.detach() for k, v in p.items()}, cam, lists, bw, settings & BLUR)
    while True:
        with torch.no_grad():
            try:
                px, py, ids, have = next(chunks)
            except StopIteration:
                return out
        with torch.set_grad_enabled(loss is not None):
            fx, fy = px.double(), py.double()
            ray, vd = _ray(cam, fx, fy)
            t, d, a3, alpha, _ = _alpha(p, cam, ids, fx[:, None], fy[:, None], ray,
                                        settings & BLUR)
            alpha = torch.where(have, alpha, 0.0)
            trans = torch.cumprod(1 - alpha, 1)
            before = torch.cat([torch.ones_like(trans[:, :1]), trans[:, :-1]], 1)
            vis = alpha * before
            color, = _pick(p, ids, ("colors",))
            img = (vis[..., None] * color).sum(1)
            rows, fu, fv = _taps(p, ids, d)
            fu, fv = fu[..., None], fv[..., None]
            t0, t1, t2, t3 = (p["texture"].index_select(0, r.reshape(-1)).reshape(*r.shape, c)
                              for r in rows)
            # by differences: no gradient at all where the taps are one texel
            val = t0 + fv * (t1 - t0) + fu * ((t2 - t0) + fv * ((t3 - t1) - (t2 - t0)))
            tex = (vis[..., None] * val).sum(1)
            normal = (vis[..., None] * a3).sum(1)
            tv = t * vd[:, None]
            med = (have & (before > 0.5)).sum(1)
            depth = torch.where(med > 0, tv.gather(1, (med - 1).clamp(min=0)[:, None])[:, 0], 0.0)
            dv = torch.where(have, t, 0.0)
            w1, w2 = vis * dv, vis * dv * dv
            cum = lambda x: torch.cumsum(x, 1) - x  # noqa: E731
            reg = (vis * (dv * dv * cum(vis) + cum(w2) - 2 * dv * cum(w1))).sum(1)
            got = (img, depth, reg, 1 - trans[:, -1], tex, normal)
            if loss is not None:
                loss(got, px, py).backward()
        for o, g in zip(out, got):
            o[py, px] = g.detach()


def _sh_basis(dirs, degree):
    x, y, z = (dirs / dirs.norm(dim=1, keepdim=True)).unbind(1)
    xx, yy, zz = x * x, y * y, z * z
    pi = math.pi
    b = [torch.full_like(x, math.sqrt(1 / (4 * pi)))]
    if degree >= 1:
        k = math.sqrt(3 / (4 * pi))
        b += [-k * y, k * z, -k * x]
    if degree >= 2:
        k = math.sqrt(15 / (4 * pi))
        b += [k * x * y, -k * y * z, math.sqrt(5 / (16 * pi)) * (2 * zz - xx - yy), -k * x * z,
              k / 2 * (xx - yy)]
    if degree >= 3:
        k, m, n = math.sqrt(35 / (32 * pi)), math.sqrt(105 / (4 * pi)), math.sqrt(21 / (32 * pi))
        b += [-k * y * (3 * xx - yy), m * x * y * z, -n * y * (4 * zz - xx - yy),
              math.sqrt(7 / (16 * pi)) * z * (2 * zz - 3 * xx - 3 * yy),
              -n * x * (4 * zz - xx - yy), m / 2 * z * (xx - yy), -k * x * (xx - 3 * yy)]
    if degree >= 4:
        k, m = math.sqrt(315 / (16 * pi)), math.sqrt(315 / (32 * pi))
        n, o = math.sqrt(45 / (16 * pi)), math.sqrt(45 / (32 * pi))
        b += [k * x * y * (xx - yy), -m * y * z * (3 * xx - yy), n * x * y * (7 * zz - 1),
              -o * y * z * (7 * zz - 3), math.sqrt(9 / (256 * pi)) * (zz * (35 * zz - 30) + 3),
              -o * x * z * (7 * zz - 3), n / 2 * (xx - yy) * (7 * zz - 1),
              -m * x * z * (xx - 3 * yy),
              k / 4 * (xx * (xx - 3 * yy) - yy * (3 * xx - yy))]
    return torch.stack(b, 1)


def _exact_params(p, grad):
    """The float64 leaves of a scene and the same with its colours."""
    leaves = {k: v.detach().double().requires_grad_(grad) for k, v in p.items() if k in _LEAVES}
    full = dict(leaves, texture_dims=p["texture_dims"])
    return leaves, full


def _colours(leaves, full, cam, case):
    """A leaf for the SH colours, so that chunks share no graph; returns what
    carries its gradient to the coefficients."""
    if "sh_coeffs" not in leaves:
        return lambda: None
    dirs = leaves["means"].detach() - cam.c2w.double()[:3, 3]
    col = (_sh_basis(dirs, case["sh"])[:, :, None] * leaves["sh_coeffs"]).sum(1)
    leaf = col.detach().requires_grad_(col.requires_grad)
    full["colors"] = leaf

    def carry():
        if leaf.grad is not None:
            col.backward(leaf.grad)
    return carry


def _l2(case, target, reg=0.0, normal=0.0, image=True):
    """The summed loss of a chunk: L2 of image + texture (or texture alone),
    distortion and normal terms, each a mean over the frame."""
    hw = case["height"] * case["width"]

    def loss(got, px, py):
        img, _, r, _, tex, n = got
        d = (img + tex if image else tex) - target[py, px]
        total = (d * d).sum() / (3 * hw)
        if reg:
            total = total + reg * r.sum() / hw
        if normal:
            total = total + normal * (n[:, 0] ** 2 + n[:, 1] ** 2 + (1 - n[:, 2]) ** 2).sum() / hw
        return total
    return loss


def _grad(v):
    return torch.zeros_like(v) if v.grad is None else v.grad


def _exact_view(case, seed, kind):
    p, g = _scene(case, seed)
    cam = _camera(np.eye(4), case["width"], case["height"])
    leaves, full = _exact_params(p, kind != "render")
    carry = _colours(leaves, full, cam, case)
    loss = None
    if kind == "step":
        target = _targets(case, g)[0].double()
        loss = _l2(case, target, *((100.0, 0.05) if case["regularised"] else ()))
    elif kind == "autograd":
        cots = [t.double() for t in _cotangents(case, g)]
        loss = lambda got, px, py: sum((a * b[py, px]).sum() for a, b in zip(got, cots))  # noqa: E731
    out = _dense(full, cam, case["block"], case["settings"], loss)
    if out is None:
        return None
    carry()
    if kind == "step":
        names = dict(opacities="opacity")
        r = {"v_" + names.get(k, k): _grad(v) for k, v in leaves.items()}
        r["v_colors"] = _grad(full["colors"])
        return dict(r, img=out[0], depth=out[1], reg=out[2], texture=out[4], normal=out[5],
                    final_Ts=1 - out[3])
    r = dict(zip(_OUT, out))
    if kind == "autograd":
        r.update({"v_" + k: _grad(v) for k, v in leaves.items()})
    return r


def _exact_views(case, seed):
    p, g = _scene(case, seed)
    if case["views"] * case["n"] * case["width"] * case["height"] > 3e11:
        return None
    cams = [_camera(c, case["width"], case["height"]) for c in _poses(case, seed)]
    targets = _targets(case, g, case["views"])
    leaves, full = _exact_params(p, True)
    imgs, texs, v_colors = [], [], 0
    for cam, target in zip(cams, targets):
        carry = _colours(leaves, full, cam, case)
        leaves_color = full["colors"]
        out = _dense(full, cam, case["block"], case["settings"], _l2(case, target.double()))
        if out is None:
            return None
        carry()
        if "sh_coeffs" in leaves:
            v_colors = v_colors + _grad(leaves_color)
        imgs.append(out[0])
        texs.append(out[4])
    r = {"v_" + dict(opacities="opacity").get(k, k): _grad(v) for k, v in leaves.items()}
    if "sh_coeffs" in leaves:
        r["v_colors"] = v_colors
    return dict(r, imgs=imgs, textures=texs)


def _exact_train(case, seed):
    p, g = _scene(case, seed)
    raw = {k: v.double().requires_grad_(True) for k, v in _raw(p).items()}
    target = _targets(case, g)[0].double()
    cam = _camera(np.eye(4), case["width"], case["height"])
    n = case["n"]
    xy = torch.exp(raw["log_scales"][:, :2])
    quats = raw["quats"] / raw["quats"].norm(dim=1, keepdim=True)
    a1, a2, _ = _axes(quats)
    mp = raw["mapping"][:, 0]
    k, cos, sin = torch.exp(mp[:, 2:3]), torch.cos(mp[:, 3:]), torch.sin(mp[:, 3:])
    made = dict(means=raw["means"], scales=torch.cat([xy, 1e-5 * xy.mean(1, True).detach()], 1),
                quats=quats, opacities=torch.sigmoid(raw["opacity_logits"]),
                uv0=mp[:, :2].reshape(n, 1, 2), umap=(k * (a1 * cos + a2 * sin)).reshape(n, 1, 3),
                vmap=(k * (a2 * cos - a1 * sin)).reshape(n, 1, 3),
                texture=torch.sigmoid(raw["texture_logits"]))
    if "sh_coeffs" in raw:
        made["sh_coeffs"] = raw["sh_coeffs"]
    else:
        made["colors"] = torch.sigmoid(raw["rgb_logits"])
    leaves = {k: v.detach().requires_grad_(True) for k, v in made.items()}
    full = dict(leaves, texture_dims=p["texture_dims"])
    carry = _colours(leaves, full, cam, case)
    out = _dense(full, cam, case["block"], case["settings"], _l2(case, target, 1.0, 1.0, False))
    if out is None:
        return None
    carry()
    names = [k for k in made if leaves[k].grad is not None]
    torch.autograd.backward([made[k] for k in names], [leaves[k].grad for k in names])
    # the first Adam step: both moments are the gradient's own
    with torch.no_grad():
        new = {"raw_" + k: v - LR * _grad(v) / (_grad(v).abs() + EPS) for k, v in raw.items()}
    return dict(new, texture=out[4], normal=out[5], reg=out[2])


def _exact_sample(case, seed):
    dims, uvs, tex, v = _sample_inputs(case, seed)
    dims, tex, v = dims.long(), tex.double(), v.double()
    # the tap indices are those of the float32 products
    x = [dims[:, k] * uvs[:, k] for k in (0, 1)]
    i = [torch.trunc(a).long() for a in x]
    fu, fv = (dims[:, k] * uvs[:, k].double() - i[k] for k in (0, 1))
    lo = [torch.minimum(i[k], dims[:, k] - 1) for k in (0, 1)]
    hi = [torch.minimum(i[k] + 1, dims[:, k] - 1) for k in (0, 1)]
    out, back = torch.zeros_like(v), torch.zeros_like(tex)
    for a, wu in ((lo[0], 1 - fu), (hi[0], fu)):
        for b, wv in ((lo[1], 1 - fv), (hi[1], fv)):
            row, wt = dims[:, 2] + a * dims[:, 1] + b, (wu * wv)[:, None]
            out += wt * tex[row]
            back.index_add_(0, row, wt * v)
    return dict(out=out, v_texture=back)


def _exact_edit(case, seed):
    p, g = _scene(case, seed)
    img, alpha, lo, hi = (t.double() for t in _edit_inputs(case, g))
    cam = _camera(np.eye(4), case["width"], case["height"])
    _, full = _exact_params(p, False)
    lists = _Lists(full, cam, case["block"])
    if lists.ids.numel() * case["block"] ** 2 > MOST_PAIRS:
        return None
    out = torch.zeros((p["texture"].shape[0], case["channels"]), dtype=torch.float64,
                      device="cuda")
    blur = case["settings"] & BLUR
    for px, py, ids, have in _composited(full, cam, lists, case["block"], blur):
        fx, fy = px.double(), py.double()
        ray, vd = _ray(cam, fx, fy)
        t, d, _, _, _ = _alpha(full, cam, ids, fx[:, None], fy[:, None], ray, blur)
        tv = t * vd[:, None]
        take = have & (tv >= lo[py, px][:, None]) & (tv <= hi[py, px][:, None])
        a = alpha[py, px][:, None]
        val = torch.cat([img[py, px] * a, a, torch.ones_like(a)], 1)[:, None, :]
        rows, fu, fv = _taps(full, ids, d)
        for wt, row in zip(((1 - fu) * (1 - fv), (1 - fu) * fv, fu * (1 - fv), fu * fv), rows):
            add = torch.where(take, wt, 0.0)[..., None] * val
            out[:, :5].index_add_(0, torch.where(take, row, 0).reshape(-1), add.reshape(-1, 5))
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "bin":
        return None  # whole numbers
    if kind == "sh":
        dirs, coeffs, v = _sh_inputs(case, seed)
        b = _sh_basis(dirs.double(), case["sh"])
        return dict(colors=(b[:, :, None] * coeffs.double()).sum(1),
                    v_coeffs=b[:, :, None] * v.double()[:, None, :])
    if kind == "sample":
        return _exact_sample(case, seed)
    if kind == "edit":
        with torch.no_grad():
            return _exact_edit(case, seed)
    if kind == "views":
        return _exact_views(case, seed)
    if kind == "train":
        return _exact_train(case, seed)
    return _exact_view(case, seed, kind)
