"""Opacities that are no ordinary number between 0 and 1, through both directions of the blend."""
import numpy as np
import pytest
import torch

from ds_splat_amd.synthetic import make_scene
from helpers import arrays, check_grads_against_bounds, comparable_gaussians, scene_settings

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def gpu_run(sc, bins):
    from ds_splat_amd import stages
    t = {k: (v.to(DEV) if isinstance(v, torch.Tensor) else v) for k, v in sc.items()}
    cam = stages.camera_from_scene(sc, DEV, list_bin=bins)
    image, st = stages.forward(cam, t["means_3d"], t["scales"], t["rotations"], t["opacities"], t["shs"])
    final = st.final_T.clone(), st.final_idx.clone()
    o = stages.backward(cam, st, 16, t["means_3d"], t["scales"], t["rotations"], t["v_image"])
    torch.cuda.synchronize()
    return image.cpu().numpy(), final[0].cpu().numpy(), final[1].cpu().numpy(), o


@pytest.mark.parametrize("infinite", [False, True])
@pytest.mark.parametrize("bins", [1, 4])
@pytest.mark.parametrize("pixels_per_lane", [1, 4])
def test_opacities_that_no_pixel_takes(oracle, blend_form, pixels_per_lane, bins, infinite):
    """Masked and pruned Gaussians (opacity zero of either sign, below the smallest normal float, negative, below
    1/255) receive zero gradients and are never staged; an infinite opacity is blended with the clamped alpha, as
    the reference's fminf does."""
    blend_form(pixels_per_lane)
    n = 6000
    sc = make_scene("cfg0", n=n, width=323, height=197, sh_degree=1, seed=21)
    sc["scales"] = sc["scales"] * 2.0
    op = sc["opacities"]
    dead = torch.zeros(n, dtype=torch.bool)
    for start, value in ((0, 0.0), (3, -0.0), (6, 1e-39), (9, 1e-45), (12, -0.25), (15, -1e-39), (18, 1e-30), (21, 0.0039)):
        op[start::24] = value
        dead[start::24] = True
    endless = torch.tensor([100, 2000, 4001] if infinite else [], dtype=torch.long)
    assert not dead[endless].any()
    op[endless] = float("inf")
    A = arrays(sc)
    s = scene_settings(sc)
    img, radii, ost = oracle.forward(s, A["means_3d"], A["scales"], A["rotations"], A["opacities"], A["shs"])
    S = oracle.state(s, ost, n)
    B = oracle.backward(s, ost, 16, A["means_3d"], A["scales"], A["rotations"], A["opacities"], A["v_image"])
    oracle.free(ost)
    image, final_T, final_idx, o = gpu_run(sc, bins)
    ok = S["margin"] > 1e-4
    assert ok.mean() > 0.98
    assert (final_idx[ok] == S["final_idx"][ok]).all()
    np.testing.assert_allclose(image[ok], img[ok], rtol=1e-4, atol=1e-5)
    dead = dead.numpy()
    finite = np.ones(n, bool)
    finite[endless.numpy()] = False     # (their own gradients hold the infinite factor)
    marks = o["marks"].cpu().numpy()
    got = {k: o[k].cpu().numpy() for k in ("v_mean3d", "v_means2d", "v_shs", "v_opacity", "v_scale", "v_quat")}
    assert not marks[dead].any() and marks[~dead].any()
    for k, g in got.items():
        assert np.isfinite(g[finite]).all(), k
        assert (g[dead] == 0.0).all() and (B[k][dead] == 0.0).all(), k
    gok = comparable_gaussians(S, B, sc["width"], final_T, final_idx) & finite
    assert gok.mean() > 0.9
    bounds = oracle.gradient_bounds(s, 16, A["means_3d"], A["scales"], A["rotations"], S["conic"], S["cov3d"], radii,
                                    B["abs_sums"], rel=1e-4)
    check_grads_against_bounds(got, B, bounds, gok, "opacities")


def one_splat_per_tile(opacity, mean, conic, final_T=None, v_image=None, behind=None):
    """The blend stages on hand-made records: tile t of a square image holds splat t (and, behind it, splat
    tiles + t, if given).  opacity[T], mean[T, 2] from the tile's first pixel centre, conic[T, 3]; colours are 1."""
    from ds_splat_amd import stages
    tiles = opacity.numel()
    side = int(round(tiles ** 0.5))
    assert side * side == tiles
    layers = 1 if behind is None else 2
    sc = make_scene("cfg0", n=1, width=16 * side, height=16 * side, sh_degree=0)
    cam = stages.camera_from_scene(sc, DEV, list_bin=1)
    first = torch.stack([torch.arange(tiles) % side, torch.arange(tiles) // side], 1) * 16.0 + 0.5
    rec = torch.zeros(layers * tiles, 12)
    rec[:tiles, 0:2], rec[:tiles, 4:7], rec[:tiles, 7] = first + mean, conic, opacity
    rec[:, 8:11] = 1.0
    if behind is not None:
        rec[tiles:, 0:2], rec[tiles:, 4:7], rec[tiles:, 7] = first + 7.25, torch.tensor([1e-4, 0.0, 1e-4]), behind
    ids = torch.arange(layers * tiles).view(layers, tiles).t().contiguous().view(-1)
    rec, ids = rec.to(DEV), ids.to(torch.int32).to(DEV)
    ranges = torch.arange(0, layers * tiles + 1, layers, dtype=torch.int32, device=DEV)
    image, T, idx = stages.blend_fwd(cam, ranges, ids, rec)
    out = {"image": image.cpu(), "T": T.cpu(), "idx": idx.cpu(), "rec": rec.cpu(), "side": side}
    if v_image is not None:
        grads = stages.blend_bwd(cam, layers * tiles, ranges, ids, rec, T if final_T is None else final_T.to(DEV), idx,
                                 v_image.to(DEV))
        out["grads"] = grads.cpu()
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("pixels_per_lane", [1, 4])
def test_alpha_is_a_product_with_the_opacity(blend_form, pixels_per_lane):
    """Half of an opacity gives half of alpha, to the last bit (a pixel's only splat, of colour 1, shows alpha); as a
    term of the exponential's argument the halves would be rounded on their own."""
    blend_form(pixels_per_lane)
    g = torch.Generator().manual_seed(5)
    rand = lambda *s: torch.rand(*s, generator=g)
    opacity = 0.02 * 40.0 ** rand(1024)
    mean = rand(1024, 2) * 16.0 - 0.5
    a, c = 0.002 * 50.0 ** rand(1024), 0.002 * 50.0 ** rand(1024)
    conic = torch.stack([a, (rand(1024) - 0.5) * torch.sqrt(a * c), c], 1)
    whole = one_splat_per_tile(opacity, mean, conic)
    for k in (1, 2):
        part = one_splat_per_tile(opacity * 0.5 ** k, mean, conic)
        seen = part["image"][..., 0] > 0
        assert seen.float().mean() > 0.2
        assert torch.equal(part["image"][seen], whole["image"][seen] * 0.5 ** k)


@pytest.mark.parametrize("pixels_per_lane", [1, 4])
def test_opacity_gradient_of_faint_splats(blend_form, pixels_per_lane):
    """v_opacity of a pixel's only splat, from one pixel, against 64 bits.  Its rounding errors, as root mean squares
    in 1e-8 of the value: the exponent's product 2, the exponential 4, T = final_T / (1 - alpha) four of 2 to 3.5,
    two products 2.5 each: 8 together.  With the opacity's logarithm as a term of the exponent (6.6 there: half a
    unit in its last place is 24) another 9."""
    blend_form(pixels_per_lane)
    tiles, side = 1024, 32
    g = torch.Generator().manual_seed(6)
    rand = lambda *s: torch.rand(*s, generator=g)
    opacity = 0.009 + 0.003 * rand(tiles)
    # sigma = 1/2 a dx^2 with dx = 4: a product of exact factors, the same in any precision
    mean = torch.stack([torch.full((tiles,), 2.0), torch.full((tiles,), 5.0)], 1)
    a = 0.02 + 0.06 * rand(tiles)
    conic = torch.stack([a, torch.zeros(tiles), a], 1)
    v = torch.zeros(16 * side, 16 * side, 3)
    v[5::16, 6::16, 0] = 1.0                    # the pixel at (6, 5) of every tile
    out = one_splat_per_tile(opacity, mean, conic, v_image=v)
    vis = torch.exp(-0.5 * a.double() * 16.0)
    alpha = opacity.double() * vis
    assert (alpha > 1.0 / 255.0).all()
    want = {5: vis, 6: alpha}                   # (T is 1: nothing lies in front)
    for column, w in want.items():
        rms = float(((out["grads"][:, column].double() / w - 1.0) ** 2).mean().sqrt())
        print("column %d: rms relative error %.2e" % (column, rms))
        assert rms < 1.0e-7


@pytest.mark.parametrize("span", ["faint", "ordinary", "huge"])
@pytest.mark.parametrize("pixels_per_lane", [1, 4])
def test_a_pixel_is_blended_exactly_where_alpha_reaches_the_threshold(blend_form, pixels_per_lane, span):
    """The limit on sigma that an entry is staged with is the last float for which alpha, evaluated as the kernels do,
    is at least 1/255: forward and backward take the pixels that comparing alpha itself takes.  Alpha is read off a
    run with twice the opacity, whose alpha is twice as large to the last bit.  The splats' centres lie far away, so
    that sigma changes by a few floats from pixel to pixel and many floats of sigma share one alpha where it is small."""
    blend_form(pixels_per_lane)
    tiles, side = 4096, 64
    g = torch.Generator().manual_seed(7)
    rand = lambda *s: torch.rand(*s, generator=g, dtype=torch.float64)
    u = rand(tiles)
    ratio = {"faint": 1.0 + 10.0 ** (-6.0 * u), "ordinary": 2.0 * 50.0 ** u, "huge": 100.0 * 10.0 ** (38.0 * u)}[span]
    opacity = (ratio / 255.0).float()
    r = torch.log(255.0 * opacity.double())
    far = 10.0 ** (2.0 + 4.0 * rand(tiles))
    angle = 2.0 * np.pi * rand(tiles)
    direction = torch.stack([torch.cos(angle), torch.sin(angle)], 1)
    # sigma reaches r within the tile, at 7.5 pixels from its first centre along both axes
    mean = (7.5 + far[:, None] * direction).float()
    a = (2.0 * r / far ** 2).float()
    conic = torch.stack([a, torch.zeros(tiles), a], 1)
    whole = one_splat_per_tile(opacity * 2.0, mean, conic)
    alpha = whole["image"][..., 0] * 0.5
    # (twice the opacity passes nearly everywhere; the largest ones' exponential underflows first)
    assert (alpha > 0).float().mean() > (0.8 if span == "huge" else 0.9)
    takes = alpha >= torch.tensor(1.0) / 255.0
    per_tile = takes.view(side, 16, side, 16).permute(0, 2, 1, 3).reshape(tiles, 256).float().mean(1)
    assert ((per_tile > 0) & (per_tile < 1)).float().mean() > 0.5
    v = torch.ones(16 * side, 16 * side, 3)
    got = one_splat_per_tile(opacity, mean, conic, v_image=v, behind=torch.full((tiles,), 0.5))
    # the splat behind is in the lists' odd places and passes everywhere
    assert (got["idx"] % 2 == 1).all()
    T = got["T"]
    back = one_splat_per_tile(torch.zeros(tiles), mean, conic, behind=torch.full((tiles,), 0.5))["T"]
    assert ((T < back) == takes).all(), "%d pixels" % int(((T < back) != takes).sum())
    # backward: the sum of alpha over the pixels that it took, against the forward's pixels; one pixel is 1/256 of it
    # (below the clamps, which differ between the two directions)
    by_tile = torch.where(takes, alpha, torch.zeros(())).double().view(side, 16, side, 16).permute(0, 2, 1, 3).reshape(tiles, 256)
    plain = by_tile.max(1).values < 0.4
    assert plain.float().mean() > 0.9
    np.testing.assert_allclose(got["grads"][:tiles, 6].double()[plain].numpy(), by_tile.sum(1)[plain].numpy(), rtol=1e-5, atol=1e-7)
