"""The rasterizer's work, as cases to time: what programs that use this package have it do.

A case is one call of a public rasterizer class (``ds_splat.GaussianRasterizer`` or the adaptor
``ds_splat_amd.inria_compat.GaussianRasterizer``) on a synthetic scene: the forward alone (a viewer,
an evaluation run) or the forward and the backward of a training step.

    listed()            the cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) the scene on the GPU, with the camera and the upstream gradient
    run(state)          one pass; returns the image, the radii and the gradients
    work(case)          bytes and operations that a pass cannot do without
    tolerance(case)     how far two correct implementations' outputs are apart
"""
import math

import torch

from ds_splat import GaussianRasterizationSettings, GaussianRasterizer
from ds_splat_amd import inria_compat

ZNEAR, ZFAR, FOVX_DEG = 0.01, 100.0, 60.0

# What a case says where it is silent.  Geometry: means uniform in [-half, half]^2 x [z0, z1], scales
# exp(N(scale_mu, scale_sigma)) per axis, opacities sigmoid(N(opacity_mu, opacity_sigma)).
DEFAULTS = dict(
    sh_degree=3,            # bands in use; the coefficient tensor always holds 16
    half=5.0, z0=2.0, z1=20.0, scale_mu=-3.5, scale_sigma=0.6, opacity_mu=0.0, opacity_sigma=1.0,
    backward=True,
    colors=False,           # colours given per Gaussian instead of SH coefficients
    cov3d=False,            # 3-D covariances given instead of scales and rotations
    api="ds_splat",         # or "inria": channel-first image with the background composited
    new_view=True,          # settings and rasterizer made for every pass (a trainer visits another view each
                            # step) or kept (a viewer, a benchmark loop)
    turn=8.0,               # the camera is turned and moved a little, by up to so many degrees, another way each seed
)


def _case(name, n, width, height, **more):
    c = dict(DEFAULTS, name=name, n=n, width=width, height=height)
    c.update(more)
    return c


def listed():
    return [
        # a thumbnail of a small object: nothing but latency and launches
        _case("thumb_fwd", 2_048, 64, 64, sh_degree=0, half=2.0, z1=10.0, scale_mu=-3.0, scale_sigma=0.5,
              backward=False, new_view=False),
        # the benchmark's smallest configuration: 16 K Gaussians at 256 x 256
        _case("cfg0_fwd", 16_384, 256, 256, sh_degree=0, half=2.0, z1=10.0, scale_mu=-3.0, scale_sigma=0.5,
              backward=False, new_view=False, turn=0.0),
        # one object in training, all SH bands on
        _case("object_train", 50_000, 512, 512, half=1.5, z0=2.0, z1=5.0, scale_mu=-4.0, scale_sigma=0.6,
              opacity_mu=-0.5),
        # the first steps of a training run: the points of the initial cloud, large and faint, one SH band;
        # an image size that no tile divides, through the adaptor that the usual trainers call
        _case("start_train", 100_000, 979, 546, sh_degree=0, scale_mu=-3.0, scale_sigma=0.4, opacity_mu=-2.2,
              opacity_sigma=0.1, api="inria"),
        # colours and covariances computed by the caller's own model
        _case("precomp_train", 300_000, 1237, 822, colors=True, cov3d=True, scale_mu=-3.3, opacity_mu=-0.5),
        # the benchmark's second configuration: 500 K Gaussians at 1080p
        _case("cfg1_train", 500_000, 1920, 1080, scale_mu=-3.0, scale_sigma=0.5, new_view=False, turn=0.0),
        # a viewer on a trained scene
        _case("view_fwd", 1_000_000, 1280, 720, scale_mu=-3.8, opacity_mu=-0.5, opacity_sigma=1.5, backward=False),
        # a scene in the middle of its training, part of the SH bands on, odd sizes
        _case("mid_train", 1_400_003, 1557, 1038, sh_degree=2, scale_mu=-3.6, opacity_mu=-1.5, api="inria"),
        # the headline: 3 M Gaussians at 1080p
        _case("cfg2_train", 3_000_000, 1920, 1080, new_view=False, turn=0.0),
        # a 4K rendering of 6 M Gaussians
        _case("cfg3_fwd", 6_000_000, 3840, 2160, half=8.0, z0=1.0, z1=30.0, scale_mu=-4.0, scale_sigma=0.5,
              backward=False, new_view=False, turn=0.0),
        # large Gaussians that overlap many times: hundreds of millions of (tile, Gaussian) pairs
        _case("cfg4_train", 1_000_000, 1920, 1080, half=3.0, z1=12.0, scale_mu=-1.5, scale_sigma=0.7,
              opacity_mu=-1.0, new_view=False, turn=0.0),
        # faint Gaussians: no pixel saturates, every visible Gaussian receives a gradient
        _case("dense_train", 2_000_000, 1920, 1080, opacity_mu=-3.3, opacity_sigma=0.4, new_view=False, turn=0.0),
    ]


def draw(rng):
    def log(lo, hi):
        return math.exp(rng.uniform(math.log(lo), math.log(hi)))

    backward = rng.random() < 0.65
    n = int(log(2_000, 3_000_000 if backward else 6_000_000))
    pixels = log(4_096, 1920 * 1080 if backward else 3840 * 2160)
    aspect = log(0.6, 2.0)
    width = max(40, int(math.sqrt(pixels * aspect)))
    height = max(40, int(pixels / width))
    half, z1 = log(1.5, 8.0), rng.uniform(5.0, 30.0)
    c = _case("", n, width, height, sh_degree=rng.choice((0, 1, 2, 3, 3)), half=round(half, 2),
              z0=round(rng.uniform(1.0, 2.0), 2), z1=round(z1, 2), scale_mu=round(rng.uniform(-4.2, -2.6), 2),
              scale_sigma=round(rng.uniform(0.3, 0.7), 2), opacity_mu=round(rng.uniform(-3.5, 0.5), 2),
              opacity_sigma=round(rng.uniform(0.1, 1.5), 2), backward=backward, colors=rng.random() < 0.15,
              cov3d=rng.random() < 0.15, api=rng.choice(("ds_splat", "ds_splat", "inria")),
              new_view=rng.random() < 0.7)
    del c["name"]
    # no more work than the largest listed cases: the deep walk's blended pairs, the 4K rendering's overlap
    while _blend(c)[1] * width * height * (1.0 if backward else 0.4) > 4.5e8 or _blend(c)[0] > 3000.0:
        c["n"] = int(c["n"] * 0.8)
        if c["n"] < 2_000:
            c["n"], c["scale_mu"] = 2_000 + rng.randrange(1000), round(c["scale_mu"] - 0.3, 2)
    return c


def _blend(c):
    """(Gaussians over a pixel, Gaussians blended at a pixel until it is opaque): means, from the distributions."""
    tanx = math.tan(math.radians(FOVX_DEG) / 2.0)
    tany = tanx * c["height"] / c["width"]
    focal = c["width"] / (2.0 * tanx)
    s2 = math.exp(2.0 * c["scale_mu"] + c["scale_sigma"] ** 2)
    op = 1.0 / (1.0 + math.exp(-c["opacity_mu"]))
    reach = max(math.log(255.0 * op), 0.1)
    steps, over = 64, 0.0
    for i in range(steps):
        z = c["z0"] + (c["z1"] - c["z0"]) * (i + 0.5) / steps
        seen = min(1.0, z * tanx / c["half"]) * min(1.0, z * tany / c["half"])
        # (the part of the screen that the cloud covers at this depth gets all of them)
        over += seen * 2.0 * math.pi * (focal * focal * s2 / (z * z) + 0.3) * reach
    over *= c["n"] / steps / (c["width"] * c["height"])
    alpha = min(0.9, max(op - 1.0 / 255.0, 1e-3) / reach)
    return over, min(over, math.log(1e4) / -math.log(1.0 - alpha))


def _camera(c, g):
    """(tanfovx, tanfovy, view matrix, projection matrix, camera position), matrices transposed as the API takes them."""
    tanx = math.tan(math.radians(FOVX_DEG) / 2.0)
    tany = tanx * c["height"] / c["width"]
    turn = [(float(x) * 2.0 - 1.0) for x in torch.rand(5, generator=g)]
    yaw, pitch = (math.radians(c["turn"]) * t for t in turn[:2])
    pos = torch.tensor(turn[2:]) * (0.02 * c["turn"])
    cy, sy, cp, sp = math.cos(yaw), math.sin(yaw), math.cos(pitch), math.sin(pitch)
    R = torch.tensor([[cy, 0.0, -sy], [0.0, 1.0, 0.0], [sy, 0.0, cy]]) @ torch.tensor(
        [[1.0, 0.0, 0.0], [0.0, cp, sp], [0.0, -sp, cp]])
    V = torch.eye(4)
    V[:3, :3] = R
    V[:3, 3] = -(R @ pos)
    P = torch.zeros(4, 4)
    P[0, 0], P[1, 1] = 1.0 / tanx, 1.0 / tany
    P[2, 2], P[2, 3], P[3, 2] = ZFAR / (ZFAR - ZNEAR), -ZFAR * ZNEAR / (ZFAR - ZNEAR), 1.0
    return tanx, tany, V.t().contiguous().cuda(), (P @ V).t().contiguous().cuda(), pos.cuda()


def prepare(case, seed):
    c = dict(DEFAULTS, **case)
    n, dev = c["n"], torch.device("cuda")
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    rand = lambda *s: torch.rand(*s, generator=g, device=dev)
    randn = lambda *s: torch.randn(*s, generator=g, device=dev)

    means = rand(n, 3)
    means[:, :2].mul_(2.0 * c["half"]).sub_(c["half"])
    means[:, 2].mul_(c["z1"] - c["z0"]).add_(c["z0"])
    scales = torch.exp(randn(n, 3) * c["scale_sigma"] + c["scale_mu"])
    quats = torch.nn.functional.normalize(randn(n, 4), dim=1)
    t = {"means_3d": means, "means_2d": torch.zeros(n, 3, device=dev),
         "opacities": torch.sigmoid(randn(n, 1) * c["opacity_sigma"] + c["opacity_mu"])}
    if c["cov3d"]:
        w, x, y, z = quats.unbind(1)
        R = torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
                         2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
                         2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)], 1).view(n, 3, 3)
        M = R * scales[:, None, :]
        S = (M[:, :, None, :] * M[:, None, :, :]).sum(-1)
        t["cov_3d"] = torch.stack([S[:, 0, 0], S[:, 0, 1], S[:, 0, 2], S[:, 1, 1], S[:, 1, 2], S[:, 2, 2]], 1)
    else:
        t["scales"], t["rotations"] = scales, quats
    if c["colors"]:
        t["colors"] = rand(n, 3)
    else:
        shs = torch.zeros(n, 16, 3, device=dev)
        shs[:, 0].copy_(randn(n, 3) * 0.5)
        for b in range(1, (c["sh_degree"] + 1) ** 2):
            shs[:, b].copy_(randn(n, 3) * 0.05)
        t["shs"] = shs
    t = {k: v.contiguous().requires_grad_(c["backward"]) for k, v in t.items()}

    tanx, tany, view, proj, pos = _camera(c, torch.Generator().manual_seed(seed))
    inria = c["api"] == "inria"
    shape = (3, c["height"], c["width"]) if inria else (c["height"], c["width"], 3)
    fields = dict(image_height=c["height"], image_width=c["width"], tanfovx=tanx, tanfovy=tany,
                  bg=torch.ones(3, device=dev) if inria else torch.zeros(3, device=dev), scale_modifier=1.0,
                  viewmatrix=view, projmatrix=proj, sh_degree=c["sh_degree"], campos=pos, prefiltered=False,
                  debug=False)
    state = {"inria": inria, "fields": fields, "tensors": t, "backward": c["backward"],
             "v_image": randn(*shape) if c["backward"] else None, "rasterizer": None}
    if not c["new_view"]:
        state["rasterizer"] = _rasterizer(state)
    return state


def _rasterizer(state):
    if state["inria"]:
        return inria_compat.GaussianRasterizer(inria_compat.GaussianRasterizationSettings(**state["fields"]))
    return GaussianRasterizer(GaussianRasterizationSettings(max_sh_degree=3, **state["fields"]))


def _render(state):
    t = state["tensors"]
    rasterizer = state["rasterizer"] or _rasterizer(state)
    if state["inria"]:
        return rasterizer(means3D=t["means_3d"], means2D=t["means_2d"], opacities=t["opacities"], shs=t.get("shs"),
                          colors_precomp=t.get("colors"), scales=t.get("scales"), rotations=t.get("rotations"),
                          cov3D_precomp=t.get("cov_3d"))
    return rasterizer(t["means_3d"], t["means_2d"], t.get("shs"), t.get("colors"), t["opacities"], t.get("scales"),
                      t.get("rotations"), t.get("cov_3d"))


def run(state):
    if not state["backward"]:
        with torch.no_grad():
            image, radii = _render(state)
        return {"image": image, "radii": radii}
    t = state["tensors"]
    for p in t.values():
        p.grad = None
    image, radii = _render(state)
    image.backward(state["v_image"])
    out = {"v_" + k: p.grad for k, p in t.items()}
    out["image"], out["radii"] = image.detach(), radii
    return out


def work(case):
    """Inputs read once, outputs written once; the operations of the projection, of the colours and of the
    Gaussians blended at each pixel (their number is the distributions' mean, not a count)."""
    c = dict(DEFAULTS, **case)
    n, pixels = c["n"], c["width"] * c["height"]
    coeffs = (c["sh_degree"] + 1) ** 2
    shape = 24 if c["cov3d"] else 28
    moved = n * (12 + 4 + shape + (12 if c["colors"] else 12 * coeffs) + 4) + pixels * 12
    flops = n * (250 + (0 if c["colors"] else 6 * coeffs + 60)) + pixels * _blend(c)[1] * 25
    if c["backward"]:
        # again what the gradients are functions of (means, shapes, opacities), the image's gradient, and
        # every input's gradient (all 16 SH coefficients)
        moved += pixels * 12 + n * (24 + 4 + shape + (12 if c["colors"] else 192))
        flops += n * 60 + pixels * _blend(c)[1] * 72
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    """Float32 throughout, but a sum over thousands of pixels in any order, and whether a Gaussian is blended at
    a pixel at all is a comparison (alpha with 1/255, transmittance with 1e-4) that the last bit of an exponential
    decides: in a few pixels of a million one Gaussian of weight up to 1/255 is in or out.  The 2-norms hardly
    move; a single value may, by that Gaussian's share.  Radii are whole numbers from operations that round one way."""
    return {"rel": 1e-4, "max": 0.1, "differ": 0.0}
