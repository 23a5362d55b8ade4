"""What the blend stages promise, in the forms that the library chooses for images of a few tiles (sixteen wavefronts a tile or
a quadrant in the forward, one for each 4x4 block in the backward), which no forced form is: the other files' checks, at most 256 tiles at
a time."""
import functools

import pytest
import torch

import test_gpu_kernel_edges
import test_gpu_opacities
import test_gpu_pipeline
import test_gpu_stages
from ds_splat_amd.synthetic import make_scene

pytestmark = pytest.mark.gpu
FEW = 256


@pytest.mark.parametrize("n,W,H,scale_mul", [(20000, 256, 256, 2.0), (4000, 200, 120, 6.0), (300, 33, 17, 4.0)])
def test_blend_fwd_vs_oracle(oracle, blend_form, n, W, H, scale_mul):
    test_gpu_stages.test_blend_fwd_vs_oracle(oracle, n, W, H, scale_mul, 0, blend_form)


@pytest.mark.parametrize("n,W,H,scale_mul,bg", [(20000, 256, 256, 2.0, (0, 0, 0)), (4000, 200, 120, 6.0, (0.3, 0.6, 0.1)),
                                                (300, 33, 17, 4.0, (1, 1, 1))])
def test_blend_bwd_vs_oracle(oracle, blend_form, n, W, H, scale_mul, bg):
    test_gpu_stages.test_blend_bwd_vs_oracle(oracle, n, W, H, scale_mul, bg, 0, blend_form)


@pytest.mark.parametrize("n,W,H,deg,scale_mul,bg,camera", [
    (16384, 256, 256, 3, 2.0, (0.2, 0.4, 0.9), "rotated"), (9000, 250, 246, 2, 2.0, None, "inside"),
    (6000, 121, 100, 3, 1.5, (0.5, 0.1, 0.3), "anisotropic")])
def test_api_forward_backward_vs_oracle(oracle, blend_form, list_bin, n, W, H, deg, scale_mul, bg, camera):
    test_gpu_pipeline.test_api_forward_backward_vs_oracle(oracle, "cfg0", n, W, H, deg, scale_mul, bg, camera, 1, 0, blend_form,
                                                          list_bin)


@pytest.mark.parametrize("n,W,H,scale_mul", [(1500, 250, 246, 0.1), (1500, 250, 246, 0.5), (1500, 170, 90, 0.5)])
def test_large_gaussians_vs_oracle(oracle, blend_form, list_bin, n, W, H, scale_mul):
    """Gaussians that cover some tiles or many: on both sides of the pairs up to which each block has a wavefront."""
    test_gpu_pipeline.test_api_forward_backward_vs_oracle(oracle, "cfg4", n, W, H, 2, scale_mul, None, "identity", 1, 0, blend_form,
                                                          list_bin)


@pytest.mark.parametrize("W,H", [(211, 197), (64, 48)])
def test_channel_first_image(oracle, blend_form, list_bin, W, H):
    test_gpu_kernel_edges.test_channel_first_image_in_every_blend_form(oracle, blend_form, list_bin, 0, 1, W, H)


@pytest.mark.parametrize("infinite", [False, True])
def test_opacities_that_no_pixel_takes(oracle, blend_form, monkeypatch, infinite):
    monkeypatch.setattr(test_gpu_opacities, "make_scene",
                        lambda name, **of: make_scene(name, **dict(of, width=203, height=149)))
    test_gpu_opacities.test_opacities_that_no_pixel_takes(oracle, blend_form, 0, 1, infinite)


def few_at_a_time(one_splat_per_tile, opacity, mean, conic, final_T=None, v_image=None, behind=None):
    """test_gpu_opacities.one_splat_per_tile, FEW tiles in a call."""
    tiles, few = opacity.numel(), 16
    side = int(round(tiles ** 0.5))
    apart = lambda x, s: x.view(s, 16, s, 16, -1).permute(0, 2, 1, 3, 4).reshape(s * s, 16, 16, -1)
    together = lambda x, s: x.view(s, s, 16, 16, -1).permute(0, 2, 1, 3, 4).reshape(16 * s, 16 * s, -1)
    assert few * few == FEW and tiles % FEW == 0 and final_T is None
    parts = []
    for first in range(0, tiles, FEW):
        of = slice(first, first + FEW)
        parts.append(one_splat_per_tile(
            opacity[of], mean[of], conic[of], behind=None if behind is None else behind[of],
            v_image=None if v_image is None else together(apart(v_image, side)[of].contiguous(), few).contiguous()))
    out = {"side": side}
    for key in ("image", "T", "idx"):
        whole = together(torch.cat([apart(p[key].contiguous(), few) for p in parts]), side)
        out[key] = whole if key == "image" else whole[..., 0]
    if v_image is not None:
        layers = 1 if behind is None else 2
        out["grads"] = torch.cat([p["grads"].view(layers, FEW, -1) for p in parts], 1).reshape(layers * tiles, -1)
    return out


@pytest.fixture
def few_tiles(monkeypatch):
    monkeypatch.setattr(test_gpu_opacities, "one_splat_per_tile",
                        functools.partial(few_at_a_time, test_gpu_opacities.one_splat_per_tile))


def test_alpha_is_a_product_with_the_opacity(blend_form, few_tiles):
    test_gpu_opacities.test_alpha_is_a_product_with_the_opacity(blend_form, 0)


def test_opacity_gradient_of_faint_splats(blend_form, few_tiles):
    test_gpu_opacities.test_opacity_gradient_of_faint_splats(blend_form, 0)


@pytest.mark.parametrize("span", ["faint", "ordinary", "huge"])
def test_a_pixel_is_blended_exactly_where_alpha_reaches_the_threshold(blend_form, few_tiles, span):
    test_gpu_opacities.test_a_pixel_is_blended_exactly_where_alpha_reaches_the_threshold(blend_form, 0, span)


@pytest.mark.parametrize("W,H", [(64, 64), (150, 70)])       # (a workgroup for each quadrant, and for each tile)
@pytest.mark.parametrize("pixels_per_lane", [0, 1, 4])
@pytest.mark.parametrize("n", [1_000_037, 3_000_005])
def test_an_accumulator_of_zeros_is_whole_and_no_more(blend_form, monkeypatch, pixels_per_lane, n, W, H):
    """DSX_PREPARE_ZEROS: whichever form prepares it, nothing of what lay in the records and the marks is left (the conics may be there),
    and nothing behind the accumulator's bytes is touched (a number of Gaussians that sixteen does not divide)."""
    from ds_splat_amd import _native, stages
    PREPARE_ZEROS = 0x800
    blend_form(pixels_per_lane)
    dev = torch.device("cuda:0")
    sc = make_scene("cfg0", n=n, width=W, height=H, sh_degree=0, seed=3)
    t = {k: (v.to(dev) if isinstance(v, torch.Tensor) else v) for k, v in sc.items()}
    cam = stages.camera_from_scene(sc, dev, list_bin=1)
    cam.c.list_bin |= PREPARE_ZEROS
    monkeypatch.setattr(stages.CameraArgs, "list_bin", property(lambda self: self.c.list_bin & 0xff))
    size, guard = int(_native.load().dsx_grads_bytes(n)) // 4, 4096
    whole = torch.full((size + guard,), float("nan"), device=dev)
    poison = whole.view(torch.int32)[0].item()
    monkeypatch.setattr(stages, "new_accumulator", lambda m, device: whole[:size])
    image, st = stages.forward(cam, t["means_3d"], t["scales"], t["rotations"], t["opacities"], t["shs"], prepare_grads=True)
    torch.cuda.synchronize()
    assert torch.isfinite(image).all() and float(image.max()) > 0
    records, marks = stages.accumulator_views(whole[:size], n)
    assert not records[:, :9].any() and not marks.any()
    conics = st.splats[:, 4:7]
    assert bool(((records[:, 9:] == 0).all(1) | (records[:, 9:] == conics).all(1)).all())
    assert bool((whole.view(torch.int32)[size:] == poison).all())
