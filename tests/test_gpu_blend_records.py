"""Records that stretch the blend kernels' arithmetic: colours that are not finite, splats of hundreds of pixels' length."""
import numpy as np
import pytest
import torch

import test_gpu_opacities as o
from ds_splat_amd.synthetic import make_scene
from helpers import arrays, comparable_gaussians, scene_settings

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("bins", [1, 4])
@pytest.mark.parametrize("pixels_per_lane", [0, 1, 4])
def test_colour_gradients_where_colours_are_not_finite(oracle, blend_form, pixels_per_lane, bins, value):
    """The gradient of a colour is a sum of alpha T v_image: it does not read the colours, and where some of them are
    infinite or NaN it is what the oracle says, for them as for all others."""
    from ds_splat_amd import stages
    blend_form(pixels_per_lane)
    n = 3000
    sc = make_scene("cfg0", n=n, width=131, height=77, sh_degree=0, seed=17)
    sc["scales"] = sc["scales"] * 0.5
    colors = torch.rand(n, 3, generator=torch.Generator().manual_seed(3))
    colors[::4, 0] = value
    colors[1::8, 1] = value
    A = arrays(sc)
    s = scene_settings(sc)
    args = A["means_3d"], A["scales"], A["rotations"], A["opacities"]
    _, radii, ost = oracle.forward(s, *args, A["shs"], colors_precomp=colors.numpy())
    S = oracle.state(s, ost, n)
    B = oracle.backward(s, ost, 16, *args, A["v_image"])
    oracle.free(ost)
    t = {k: (v.to(DEV) if isinstance(v, torch.Tensor) else v) for k, v in sc.items()}
    cam = stages.camera_from_scene(sc, DEV, list_bin=bins)
    _, st = stages.forward(cam, t["means_3d"], t["scales"], t["rotations"], t["opacities"], t["shs"],
                           colors_precomp=colors.to(DEV))
    final_T, final_idx = st.final_T.cpu().numpy(), st.final_idx.cpu().numpy()
    got = stages.backward(cam, st, 16, t["means_3d"], t["scales"], t["rotations"], t["v_image"])["v_colors"].cpu().numpy()
    ok = S["margin"] > 1e-4
    assert ok.mean() > 0.97 and (final_idx[ok] == S["final_idx"][ok]).all()
    gok = comparable_gaussians(S, B, sc["width"], final_T, final_idx)
    assert gok.mean() > 0.8 and np.isfinite(B["v_colors"]).all()
    # (the sums' bound as in gradient_bounds: their order is the atomics')
    err = np.abs(got.astype(np.float64) - B["v_colors"])
    assert (err[gok] <= 1e-4 * B["abs_sums"][gok, 6:9] + 1e-7).all(), "%d not finite" % int((~np.isfinite(got)).sum())


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
@pytest.mark.parametrize("pixels_per_lane", [1, 4])
def test_an_infinite_colour_that_no_pixel_takes(blend_form, pixels_per_lane, value):
    """A splat between four pixels of one block, too narrow for any, gets no gradient whatever its colour and wherever it stands
    in its round of staged entries (the wide splats behind it fill the rounds of 56 and of 248)."""
    from ds_splat_amd import stages
    blend_form(pixels_per_lane)
    cam = stages.camera_from_scene(make_scene("cfg0", n=1, width=16, height=16, sh_degree=0), DEV, list_bin=1)
    v_image = torch.randn(16, 16, 3, generator=torch.Generator().manual_seed(1)).to(DEV)
    for behind in (1, 55, 56, 57, 112, 248):
        k = behind + 4
        rec = torch.zeros(k, 12)
        rec[:, 0:2], rec[:, 4], rec[:, 6], rec[:, 7], rec[:, 8:11] = 8.0, 1e-3, 1e-3, 0.008, 0.5
        rec[3, 0:2], rec[3, 4], rec[3, 6], rec[3, 7], rec[3, 8] = 6.0, 100.0, 100.0, 0.9, value
        rec, ids = rec.to(DEV), torch.arange(k, dtype=torch.int32, device=DEV)
        ranges = torch.tensor([0, k], dtype=torch.int32, device=DEV)
        _, T, idx = stages.blend_fwd(cam, ranges, ids, rec)
        grads = stages.blend_bwd(cam, k, ranges, ids, rec, T, idx, v_image)[:, :9].cpu()
        assert (idx.cpu() == k - 1).any()
        assert (grads[3] == 0.0).all(), (behind, grads[3])
        assert torch.isfinite(grads).all() and (grads[0] != 0.0).any()


@pytest.mark.parametrize("length", [150.0, 800.0])
@pytest.mark.parametrize("pixels_per_lane", [0, 1, 4])
def test_a_needle_is_blended_wherever_alpha_reaches_the_threshold(blend_form, pixels_per_lane, length):
    """Splats of hundreds of pixels' length and less than one pixel's width, each in a tile far from its middle: the
    terms of its exponent, up to 1e6, cancel, so what a test of the whole tile or of a block finds lies further from
    the pixels' own exponents than a fixed slack.  With an opacity for which alpha reaches 1/255 at a pixel of
    the tile or a few, both directions take just the pixels that comparing alpha takes (4096 tiles: with the form left
    to the library, the two directions run different ones)."""
    tiles, side = 4096, 64
    g = torch.Generator().manual_seed(11)
    rand = lambda *s: torch.rand(*s, generator=g, dtype=torch.float64)
    angle, across, along = 2.0 * np.pi * rand(tiles), 20.0 * rand(tiles) - 10.0, length * (0.1 + 0.9 * rand(tiles))
    cos, sin = torch.cos(angle), torch.sin(angle)
    mean = torch.stack([7.5 + along * cos - across * sin, 7.5 + along * sin + across * cos], 1).float()
    major, minor = 1.0 / length ** 2, 1.0 / (0.3 + 0.3 * rand(tiles))
    conic = torch.stack([major * cos ** 2 + minor * sin ** 2, (major - minor) * cos * sin,
                         major * sin ** 2 + minor * cos ** 2], 1).float()
    by_tile = lambda x: x.view(side, 16, side, 16).permute(0, 2, 1, 3).reshape(tiles, 256)
    blend_form(1)       # alpha, from an opacity whose reach lies far above
    alpha = by_tile(o.one_splat_per_tile(torch.full((tiles,), 0.9), mean, conic)["image"][..., 0].contiguous())
    most = alpha.max(1).values.double()
    crossed = (most > 2.0 / 255.0) & (most < 0.88)
    assert crossed.float().mean() > 0.6
    opacity = torch.where(crossed, 0.9 * (1.0 + 1e-5) / 255.0 / most.clamp_min(1e-3), 0.0).float()
    twice = by_tile(o.one_splat_per_tile(opacity * 2.0, mean, conic)["image"][..., 0].contiguous()) * 0.5
    takes = twice >= torch.tensor(1.0) / 255.0
    assert (takes.any(1) == crossed).all()
    blend_form(pixels_per_lane)
    v = torch.ones(16 * side, 16 * side, 3)
    got = o.one_splat_per_tile(opacity, mean, conic, v_image=v)
    missed = (by_tile(got["image"][..., 0].contiguous()) > 0) != takes
    assert not missed.any(), "forward: %d tiles of %d" % (int(missed.any(1).sum()), int(crossed.sum()))
    want = torch.where(takes, twice, torch.zeros(())).double().sum(1)
    # (a pixel more or less is 1/255 of colour 1: from sums of up to 16 pixels)
    np.testing.assert_allclose(got["grads"][:, 6].double().numpy(), want.numpy(), rtol=1e-5, atol=1e-7)


def sums_in_64_bits(rec, v_image, bg, final_T, final_idx):
    """The nine sums of every entry, and the sums of their terms' magnitudes, back to front from what the forward
    left, all entries in the one list of every pixel.  Also the pixels where a decision is closer than 32 bits tell."""
    h, w = final_T.shape
    y, x = torch.meshgrid(torch.arange(h) + 0.5, torch.arange(w) + 0.5, indexing="ij")
    v, T, last = v_image.double(), final_T.double().clone(), final_idx
    behind = (v * bg.double()).sum(-1)
    n = rec.shape[0]
    sums, terms, close = torch.zeros(n, 9).double(), torch.zeros(n, 9).double(), torch.zeros(h, w, dtype=torch.bool)
    for i in range(n - 1, -1, -1):
        mx, my, _, _, a, b, c, opacity, red, green, blue, _ = rec[i].double()
        dx, dy = x - mx, y - my
        sigma = 0.5 * (a * dx * dx + c * dy * dy) + b * dx * dy
        vis = torch.exp(-sigma)
        close |= ((opacity * vis * 255.0 - 1.0).abs() < 1e-4) | (sigma.abs() < 1e-6)
        takes = (opacity * vis >= 1.0 / 255.0) & (sigma >= 0.0) & (i <= last)
        alpha = torch.where(takes, (opacity * vis).clamp(max=0.99), torch.zeros(()).double())
        T = T / (1.0 - alpha)
        ahead = v @ torch.stack([red, green, blue]) - behind
        behind = behind + alpha * ahead
        vw = torch.where(takes, vis * T * ahead, torch.zeros(()).double())
        s = opacity * vw
        for j, t in enumerate((s * (a * dx + b * dy), s * (b * dx + c * dy), -0.5 * s * dx * dx, -s * dx * dy,
                               -0.5 * s * dy * dy, vw, alpha * T * v[..., 0], alpha * T * v[..., 1], alpha * T * v[..., 2])):
            sums[i, j], terms[i, j] = t.sum(), t.abs().sum()
    return sums, terms, close


@pytest.mark.parametrize("kind", ["faint", "clamped", "stopping", "wild"])
@pytest.mark.parametrize("n", [1, 2, 55, 57, 113, 247, 249, 500])
@pytest.mark.parametrize("pixels_per_lane", [0, 1, 4])
def test_backward_sums_against_64_bits(blend_form, pixels_per_lane, n, kind):
    """Around the rounds of 56 and of 248 entries, odd and even: rounds that no pixel's last entry lies in, rounds where
    pixels end or alpha reaches the clamp, and an upstream gradient whose products with zero must stay out of the sums."""
    from ds_splat_amd import stages
    blend_form(pixels_per_lane)
    g = torch.Generator().manual_seed(n)
    rand = lambda *s: torch.rand(*s, generator=g)
    h, w = 30, 43
    rec = torch.zeros(n, 12)
    rec[:, 0], rec[:, 1], rec[:, 3] = rand(n) * (w + 8) - 4, rand(n) * (h + 8) - 4, 50.0
    turn, major, minor = rand(n) * 3.14159, 1.0 / (1.0 + 9.0 * rand(n)) ** 2, 1.0 / (0.7 + rand(n)) ** 2
    cos, sin = torch.cos(turn), torch.sin(turn)
    rec[:, 4], rec[:, 5] = major * cos ** 2 + minor * sin ** 2, (major - minor) * cos * sin
    rec[:, 6] = major * sin ** 2 + minor * cos ** 2
    rec[:, 7] = 0.02 + (0.05 if kind == "faint" else 0.9) * rand(n)
    if kind == "clamped":
        rec[:, 7] = torch.where(rand(n) < 0.02, 0.999, 0.05)
    rec[:, 8:11] = rand(n, 3)
    v_image = torch.randn(h, w, 3, generator=g)
    if kind == "wild":
        v_image[17:, 20:] *= 1e13
    scene = make_scene("cfg0", n=1, width=w, height=h, sh_degree=0)
    cam = stages.camera_from_scene(scene, DEV, list_bin=1, bg=torch.tensor([0.3, 0.1, 0.8]))
    tiles = ((h + 15) // 16) * ((w + 15) // 16)
    ids = torch.arange(n, dtype=torch.int32).repeat(tiles).to(DEV)
    ranges = (torch.arange(tiles + 1, dtype=torch.int32) * n).to(DEV)
    _, final_T, final_idx = stages.blend_fwd(cam, ranges, ids, rec.to(DEV))
    tile_of = torch.arange(h)[:, None] // 16 * ((w + 15) // 16) + torch.arange(w)[None] // 16
    args = torch.tensor([0.3, 0.1, 0.8]), final_T.cpu(), final_idx.cpu() - tile_of * n
    close = sums_in_64_bits(rec, v_image, *args)[2]
    assert close.float().mean() < 0.2
    v_image[close] = 0.0
    want, terms, _ = sums_in_64_bits(rec, v_image, *args)
    got = stages.blend_bwd(cam, n, ranges, ids, rec.to(DEV), final_T, final_idx, v_image.to(DEV))[:, :9].cpu().double()
    # (T is rebuilt over up to 500 entries, three roundings of 6e-8 each, and starts from one that the forward left)
    assert ((got - want).abs() <= 1e-4 * terms + 1e-7).all(), float(((got - want).abs() / (terms + 1e-3)).max())


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_an_infinite_colour_that_no_pixel_takes_where_tiles_are_few(blend_form, value):
    """The same with the form that the library chooses for a few tiles."""
    test_an_infinite_colour_that_no_pixel_takes(blend_form, 0, value)


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
@pytest.mark.parametrize("n", [57, 130, 300])
@pytest.mark.parametrize("pixels_per_lane", [0, 1, 4])
def test_a_pixels_gradient_that_is_not_finite(blend_form, pixels_per_lane, n, value):
    """An infinite or NaN upstream gradient at a pixel that some entries took and at one that none took: it is in the sums
    of those that took it; those of all others, in the same block's list or not, are what they are without it."""
    from ds_splat_amd import stages
    blend_form(pixels_per_lane)
    g = torch.Generator().manual_seed(n)
    rand = lambda *s: torch.rand(*s, generator=g)
    h, w = 30, 43
    rec = torch.zeros(n, 12)
    rec[:, 0], rec[:, 1], rec[:, 3] = rand(n) * 0.7 * w, rand(n) * 0.7 * h, 50.0
    rec[:, 4] = rec[:, 6] = 0.6 + rand(n)                               # (a pixel or two wide)
    rec[:, 7], rec[:, 8:11] = 0.02 + 0.3 * rand(n), rand(n, 3)
    # one in the empty part, which takes some pixels of its block and not the one at (36, 26)
    rec[n // 2, :2], rec[n // 2, 4], rec[n // 2, 6], rec[n // 2, 7] = torch.tensor([38.3, 26.3]), 3.0, 3.0, 0.5
    cam = stages.camera_from_scene(make_scene("cfg0", n=1, width=w, height=h, sh_degree=0), DEV, list_bin=1,
                                   bg=torch.tensor([0.3, 0.1, 0.8]))
    tiles = ((h + 15) // 16) * ((w + 15) // 16)
    ids = torch.arange(n, dtype=torch.int32).repeat(tiles).to(DEV)
    ranges = (torch.arange(tiles + 1, dtype=torch.int32) * n).to(DEV)
    _, final_T, final_idx = stages.blend_fwd(cam, ranges, ids, rec.to(DEV))
    tile_of = torch.arange(h)[:, None] // 16 * ((w + 15) // 16) + torch.arange(w)[None] // 16
    args = torch.tensor([0.3, 0.1, 0.8]), final_T.cpu(), final_idx.cpu() - tile_of * n
    v_image = torch.randn(h, w, 3, generator=g)
    close = sums_in_64_bits(rec, v_image, *args)[2]
    assert close.float().mean() < 0.2
    v_image[close] = 0.0
    untouched, touched = (final_T.cpu() == 1.0) & ~close, (final_T.cpu() < 0.99) & ~close
    assert untouched[26, 36] and final_T[26, 38] < 1.0
    y, x = torch.nonzero(touched)[len(torch.nonzero(touched)) // 2].tolist()
    # (the 64-bit sums without the two; who took them, from an upstream gradient of theirs alone)
    alone = torch.zeros_like(v_image)
    alone[26, 36], alone[y, x], v_image[26, 36], v_image[y, x] = 1.0, 1.0, 0.0, 0.0
    want, terms, _ = sums_in_64_bits(rec, v_image, *args)
    others = sums_in_64_bits(rec, alone, *args)[1][:, 6] == 0.0
    v_image[26, 36], v_image[y, x] = value, value                       # (the first: by nobody)
    got = stages.blend_bwd(cam, n, ranges, ids, rec.to(DEV), final_T, final_idx, v_image.to(DEV))[:, :9].cpu().double()
    assert 0 < int((~others).sum()) < n // 2 and others[n // 2]
    # (T over up to 300 entries, as above)
    assert ((got - want).abs() <= 1e-4 * terms + 1e-7)[others].all(), int((~torch.isfinite(got[others])).any(1).sum())
    assert not torch.isfinite(got[~others]).all(1).any()


@pytest.mark.parametrize("opacity", [0.99, 0.9900001, 1.0, 2.0, 2.5, 300.0])
@pytest.mark.parametrize("n, where", [(2, 1), (57, 3), (250, 249)])
@pytest.mark.parametrize("pixels_per_lane", [0, 1, 4])
def test_sums_where_one_opacity_lies_at_a_limit_of_the_walks(blend_form, pixels_per_lane, n, where, opacity):
    """Rounds of the backward whose alphas stay below the clamp, rounds that reach it, and rounds with an opacity beyond 2 take different
    walks: one opacity on either side of each limit among ordinary ones, in the first round and in a later one."""
    from ds_splat_amd import stages
    blend_form(pixels_per_lane)
    g = torch.Generator().manual_seed(n)
    rand = lambda *s: torch.rand(*s, generator=g)
    h, w = 16, 16
    rec = torch.zeros(n, 12)
    rec[:, 0], rec[:, 1], rec[:, 3] = rand(n) * w, rand(n) * h, 50.0
    rec[:, 4] = rec[:, 6] = 0.02 + 0.2 * rand(n)
    rec[:, 7], rec[:, 8:11] = 0.01 + 0.03 * rand(n), rand(n, 3)
    rec[where, :2], rec[where, 7] = torch.tensor([8.5, 7.5]), opacity    # (on a pixel's centre but for the sign of sigma)
    bg = torch.tensor([0.3, 0.1, 0.8])
    cam = stages.camera_from_scene(make_scene("cfg0", n=1, width=w, height=h, sh_degree=0), DEV, list_bin=1, bg=bg)
    ids, ranges = torch.arange(n, dtype=torch.int32).to(DEV), torch.tensor([0, n], dtype=torch.int32).to(DEV)
    _, final_T, final_idx = stages.blend_fwd(cam, ranges, ids, rec.to(DEV))
    v_image = torch.randn(h, w, 3, generator=g)
    args = bg, final_T.cpu(), final_idx.cpu()
    close = sums_in_64_bits(rec, v_image, *args)[2]
    assert close.float().mean() < 0.2
    v_image[close] = 0.0
    want, terms, _ = sums_in_64_bits(rec, v_image, *args)
    assert (terms[where] > 0).all()
    got = stages.blend_bwd(cam, n, ranges, ids, rec.to(DEV), final_T, final_idx, v_image.to(DEV))[:, :9].cpu().double()
    # (as above: T over up to 250 entries)
    assert ((got - want).abs() <= 1e-4 * terms + 1e-7).all(), float(((got - want).abs() / (terms + 1e-3)).max())


@pytest.mark.parametrize("n, where", [(1, 0), (64, 63), (65, 64), (150, 3), (150, 70), (150, 149)])
def test_alpha_is_clamped_in_the_rounds_that_need_it(blend_form, n, where):
    """One opaque splat on a pixel's centre among faint ones, in any round of 64 staged entries: the forms of the
    forward, of which only one leaves the clamp out of the other rounds, give the same bits, and the pixel's
    transmittance is what 1 - 0.999 leaves of it."""
    from ds_splat_amd import stages
    cam = stages.camera_from_scene(make_scene("cfg0", n=1, width=16, height=16, sh_degree=0), DEV, list_bin=1)
    rec = torch.zeros(n, 12)
    rec[:, 0:2], rec[:, 4], rec[:, 6], rec[:, 7], rec[:, 8:11] = 8.0, 1e-3, 1e-3, 0.008, 0.5
    rec[where, 0:2], rec[where, 4], rec[where, 6], rec[where, 7] = 5.51, 0.5, 0.5, 1.0
    rec, ids = rec.to(DEV), torch.arange(n, dtype=torch.int32, device=DEV)
    ranges = torch.tensor([0, n], dtype=torch.int32, device=DEV)
    got = []
    for form in (1, 4):
        blend_form(form)
        got.append([x.cpu() for x in stages.blend_fwd(cam, ranges, ids, rec)])
    assert all(torch.equal(a, b) for a, b in zip(*got))
    faint = 0.008 * np.exp(-0.5e-3 * 2 * 2.5 ** 2)
    # (1 - 0.999 in 32 bits, to a unit in the last place of 0.999)
    np.testing.assert_allclose(got[1][1][5, 5], 1e-3 * (1.0 - faint) ** (n - 1), rtol=1e-4)
