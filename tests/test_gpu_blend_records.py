"""Records that stretch the blend kernels' arithmetic: colours that are not finite."""
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
