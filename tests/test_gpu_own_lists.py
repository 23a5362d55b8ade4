"""A forward without a backward, of few tiles: every tile finds its own entries.  The image and the radii against the general
path's (whose lists, ranges and images are compared with the oracle's elsewhere), which a forward with a backward to follow takes,
and against the oracle's."""
import numpy as np
import pytest
import torch

from ds_splat import GaussianRasterizationSettings, GaussianRasterizer
from ds_splat_amd import _native, inria_compat
from ds_splat_amd.synthetic import make_scene
from helpers import set_camera
import test_gpu_pipeline

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def render_both(sc, planar=False, precomputed=False):
    """(image, radii) without and with gradients to take"""
    t = {k: (v.to(DEV) if isinstance(v, torch.Tensor) else v) for k, v in sc.items()}
    fields = dict(image_height=sc["height"], image_width=sc["width"], tanfovx=sc["tanfovx"], tanfovy=sc["tanfovy"],
                  bg=torch.tensor([0.2, 0.5, 0.8], device=DEV), scale_modifier=1.0, viewmatrix=t["viewmatrix"],
                  projmatrix=t["projmatrix"], sh_degree=sc["sh_degree"], campos=t["campos"], prefiltered=False, debug=False)
    means2d, colors, cov = torch.zeros_like(t["means_3d"]), None, None
    if precomputed:
        colors = t["shs"][:, 0].contiguous().abs()
        s2 = t["scales"][:, :1] ** 2
        cov = torch.cat([s2, 0.1 * s2, 0 * s2, s2, 0 * s2, 0.5 * s2], 1).contiguous()
    shs, scales, rots = (None, None, None) if precomputed else (t["shs"], t["scales"], t["rotations"])
    got = []
    for grad in (False, True):
        means = t["means_3d"].clone().requires_grad_(grad)
        if planar:
            r = inria_compat.GaussianRasterizer(inria_compat.GaussianRasterizationSettings(**fields))
            out = r(means3D=means, means2D=means2d, opacities=t["opacities"], shs=shs, colors_precomp=colors, scales=scales,
                    rotations=rots, cov3D_precomp=cov)
        else:
            r = GaussianRasterizer(GaussianRasterizationSettings(max_sh_degree=3, **fields))
            out = r(means, means2d, shs, colors, t["opacities"], scales, rots, cov)
        got.append(tuple(x.detach() for x in out))
    return got


def check(sc, in_parts=False, **options):
    (image, radii), (want, want_radii) = render_both(sc, **options)
    assert torch.equal(radii, want_radii)
    if in_parts:
        # (a colour is a sum of at most 10200 terms in four parts whose members differ: as many roundings of 2^-24 of at
        # most the whole sum, of either sign: sqrt(10200) 2^-24 = 6e-6 of the largest colour)
        assert not torch.isnan(image).any()
        assert float((image - want).abs().max()) <= 6e-6 * max(1.0, float(want.abs().max()))
    else:
        assert torch.equal(image, want)
    return image


def taken(sc):
    return _native.load().dsx_render_bytes(sc["n"], sc["width"], sc["height"], 0) > 0


@pytest.mark.parametrize("n,W,H,applies", [
    (1, 16, 16, True),             # (the last Gaussian emits nothing)
    (2, 1, 1, True),
    (300, 40, 40, True),
    (5000, 97, 50, True),          # tiles cut off at both edges
    (16384, 256, 256, True),       # as many tiles as there are compute units
    (16384, 256, 257, False),
    (34600, 256, 256, True),
    (34601, 256, 256, False),
    (9100, 16, 16, True),
    (9101, 16, 16, False),
])
def test_image_of_tiles_that_find_their_entries(n, W, H, applies):
    sc = make_scene("cfg0", n=n, width=W, height=H, sh_degree=1, seed=n)
    assert taken(sc) == applies
    for options in ({}, {"planar": True}, {"precomputed": True}):
        check(sc, in_parts=n > 4096 and W * H <= 256, **options)


@pytest.mark.parametrize("depths", ["spread", "equal", "layers", "nearly_equal", "two"])
@pytest.mark.parametrize("n,W,H", [(4096, 16, 16), (4097, 16, 16), (9100, 16, 16), (10200, 64, 48)])
def test_windows_of_a_tile_with_many_entries(n, W, H, depths):
    """Faint Gaussians that cover every tile: up to 4096 entries are one window, more are several; depths that are equal or nearly so
    are told apart by their last bits or by the index, and sorted by comparisons where a bin holds many."""
    sc = make_scene("cfg0", n=n, width=W, height=H, sh_degree=0, seed=n)
    g = torch.Generator().manual_seed(n)
    u = torch.rand(n, generator=g)
    sc["means_3d"][:, :2] *= 0.05
    sc["means_3d"][:, 2] = {"spread": 2.0 + 8.0 * u, "equal": 4.0 + 0.0 * u, "layers": 2.0 + (8.0 * u).floor(),
                            "nearly_equal": 4.0 + 1e-5 * u, "two": torch.where(u < 0.5, 2.0, 9.0)}[depths]
    sc["scales"] = torch.full((n, 3), 1.0) * (1.0 + torch.rand(n, 1, generator=g))
    sc["opacities"] = 0.004 + 0.004 * torch.rand(n, 1, generator=g)
    assert taken(sc)
    image = check(sc, in_parts=n > 4096)
    assert float(image.abs().max()) > 0.1


@pytest.mark.parametrize("share", [0.0, 0.5, 1.0])
@pytest.mark.parametrize("n,W,H", [(200, 70, 50), (9000, 70, 50), (3000, 16, 16)])
def test_entries_behind_the_camera_and_the_highest_tile(n, W, H, share):
    """The highest occupied tile's entries are blended by the image's last tile, and where no tile is occupied that one blends those
    of negative depth, once for every tile that they touch (the reference's last run of keys, which nothing ends)."""
    sc = make_scene("cfg0", n=n, width=W, height=H, sh_degree=0, seed=n)
    sc["projmatrix"][:, 2] = torch.tensor([0.0, 0.0, 0.0, 0.5])
    sc["projmatrix"][:, 3] = torch.tensor([0.0, 0.0, 0.0, 1.0])
    sc["means_3d"][:, :2] = 0.2 * sc["means_3d"][:, :2] - 0.35          # (the upper left of the image: its last tiles are empty)
    behind = torch.arange(n) < int(share * n)
    sc["means_3d"][behind] *= -1.0
    assert taken(sc)
    check(sc, in_parts=n > 4096)


@pytest.mark.parametrize("name,n,W,H,deg,scale_mul,bg,camera", [
    ("cfg0", 2048, 64, 64, 0, 1.0, None, "identity"),
    ("cfg0", 16384, 256, 256, 3, 2.0, (0.2, 0.4, 0.9), "rotated"),
    ("cfg0", 20000, 250, 200, 3, 2.0, None, "inside"),          # (Gaussians behind the camera)
    ("cfg4", 3000, 200, 180, 2, 0.5, (0.5, 0.1, 0.3), "anisotropic"),
    ("cfg4", 9000, 16, 16, 0, 0.5, None, "identity"),           # (one tile, several windows)
])
def test_image_vs_oracle(oracle, name, n, W, H, deg, scale_mul, bg, camera):
    sc = set_camera(make_scene(name, n=n, width=W, height=H, sh_degree=deg), camera)
    assert taken(sc)
    image, radii, _ = test_gpu_pipeline.api_run(sc, scale_mul, backward=False, bg=bg)
    want, want_radii, S, _ = test_gpu_pipeline.oracle_run(oracle, sc, scale_mul, bg=bg, backward=False)
    assert (radii.cpu().numpy() == want_radii).all() and (want_radii > 0).sum() > n // 20
    ok = S["margin"] > 1e-4
    assert ok.mean() > 0.98, ok.mean()
    np.testing.assert_allclose(image.cpu().numpy()[ok], want[ok], rtol=1e-4, atol=1e-5)


def test_a_captured_forward_without_lists_follows_its_inputs():
    """Nothing in it waits for the device, so it can be captured; every replay renders what its inputs hold by then."""
    sc = make_scene("cfg0", n=2000, width=100, height=70, sh_degree=1, seed=3)
    assert taken(sc)
    t = {k: (v.to(DEV) if isinstance(v, torch.Tensor) else v) for k, v in sc.items()}
    r = GaussianRasterizer(GaussianRasterizationSettings(
        image_height=sc["height"], image_width=sc["width"], tanfovx=sc["tanfovx"], tanfovy=sc["tanfovy"],
        bg=torch.tensor([0.2, 0.5, 0.8], device=DEV), scale_modifier=1.0, viewmatrix=t["viewmatrix"], projmatrix=t["projmatrix"],
        sh_degree=1, max_sh_degree=3, campos=t["campos"], prefiltered=False, debug=False))
    means2d = torch.zeros_like(t["means_3d"])
    run = lambda: r(t["means_3d"], means2d, t["shs"], None, t["opacities"], t["scales"], t["rotations"], None)
    with torch.no_grad():
        run()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            image, radii = run()
        seen = []
        for step in range(4):
            t["means_3d"].mul_(0.9)
            want, want_radii = run()
            image.fill_(-1.0)
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(image, want) and torch.equal(radii, want_radii)
            seen.append(want.clone())
        assert not torch.equal(seen[0], seen[3])


@pytest.mark.parametrize("n,W,H", [(960, 16, 16), (961, 16, 16), (962, 16, 16), (2500, 128, 128), (2500, 208, 80), (3000, 127, 113)])
@pytest.mark.parametrize("depths", ["spread", "equal"])
def test_quadrants_and_entries_that_a_round_holds(blend_form, n, W, H, depths):
    """Up to 960 entries of a tile are tested, sorted and staged in one go, and up to 64 tiles have a workgroup for each quadrant: at the edges
    of both, the image that the tiles' own lists give, that of the general path, and the four-wavefront form's agree."""
    sc = make_scene("cfg0", n=n, width=W, height=H, sh_degree=0, seed=n)
    if W * H == 256:
        sc["means_3d"][:, :2] *= 0.05
        sc["scales"] = torch.full((n, 3), 1.0) * (1.0 + torch.rand(n, 1, generator=torch.Generator().manual_seed(n)))
        sc["opacities"] = 0.004 + 0.02 * torch.rand(n, 1, generator=torch.Generator().manual_seed(n))
    if depths == "equal":
        sc["means_3d"][:, 2] = 4.0
    assert taken(sc)
    image = check(sc)
    (_, _), (four, _) = (blend_form(1), render_both(sc))[1]
    # (the sums' parts differ: as above)
    assert float((image - four).abs().max()) <= 6e-6 * max(1.0, float(four.abs().max()))
    assert float(image.abs().max()) > 0.1


@pytest.mark.parametrize("n", [128, 129, 130, 500, 960])
@pytest.mark.parametrize("depths", ["equal", "two", "outlier"])
def test_entries_of_one_round_whose_depths_are_alike(n, depths):
    """Up to 128 entries of a bin of depths are compared with each other, more are sorted: at the edges of both, all in one bin, in two,
    and all but one, the image is the general path's."""
    g = torch.Generator().manual_seed(n)
    sc = make_scene("cfg0", n=n, width=16, height=16, sh_degree=0, seed=n)
    sc["means_3d"][:, :2] *= 0.05
    sc["scales"] = torch.ones(n, 3) * (1.0 + torch.rand(n, 1, generator=g))
    sc["opacities"] = 0.004 + 0.02 * torch.rand(n, 1, generator=g)
    sc["means_3d"][:, 2] = 4.0
    if depths == "two":
        sc["means_3d"][::3, 2] = 6.0
    if depths == "outlier":
        sc["means_3d"][n // 2, 2] = 9.0
    assert taken(sc)
    assert float(check(sc).abs().max()) > 0.01


def test_depths_that_are_alike_take_no_longer():
    """A plane of Gaussians that faces the camera, of which each tile has hundreds of one depth, against the same ones a little apart: the
    same work but for the order (1.9 times as long where each entry is compared with all others of its depth, 1.3 as it is)."""
    n = 12000
    sc = make_scene("cfg0", n=n, width=176, height=160, sh_degree=0, seed=1)
    assert taken(sc)
    t = {k: (v.to(DEV) if isinstance(v, torch.Tensor) else v) for k, v in sc.items()}
    settings = GaussianRasterizationSettings(
        image_height=sc["height"], image_width=sc["width"], tanfovx=sc["tanfovx"], tanfovy=sc["tanfovy"], bg=t["bg"], scale_modifier=1.0,
        viewmatrix=t["viewmatrix"], projmatrix=t["projmatrix"], sh_degree=0, max_sh_degree=3, campos=t["campos"], prefiltered=False,
        debug=False)
    rasterizer = GaussianRasterizer(settings)
    apart = t["means_3d"].clone()
    apart[:, 2] = 4.0 + 0.2 * torch.rand(n, generator=torch.Generator().manual_seed(2)).to(DEV)
    plane = apart.clone()
    plane[:, 2] = 4.1
    means2d = torch.zeros_like(plane)
    best = {}
    with torch.no_grad():
        for _ in range(8):
            for name, means in (("apart", apart), ("plane", plane)):
                begin, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
                begin.record()
                for _ in range(50):
                    rasterizer(means, means2d, t["shs"], None, t["opacities"], t["scales"], t["rotations"], None)
                end.record()
                end.synchronize()
                best[name] = min(best.get(name, 1e9), begin.elapsed_time(end) / 50)
    print("us: apart %.1f, alike %.1f" % (1e3 * best["apart"], 1e3 * best["plane"]))
    assert best["plane"] < 1.6 * best["apart"], best
