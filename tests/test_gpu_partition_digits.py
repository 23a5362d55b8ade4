"""The partition of the pairs by list, on both sides of the numbers of pairs up to which it takes one digit."""
import pytest
import torch

from ds_splat_amd.synthetic import make_scene

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def forward(W, H, bins, means, scales, **scene):
    from ds_splat_amd import stages
    n = means.shape[0]
    sc = make_scene("cfg0", n=n, width=W, height=H, sh_degree=0, **scene)
    cam = stages.camera_from_scene(sc, DEV, list_bin=bins)
    image, st = stages.forward(cam, means, scales, sc["rotations"].to(DEV), sc["opacities"].to(DEV), sc["shs"].to(DEV))
    assert torch.isfinite(image).all()
    return cam, st


@pytest.mark.parametrize("more", [0, 1])
@pytest.mark.parametrize("W,H,bins,lists,each", [
    (640, 400, 1, 1000, 12000),      # ten bits: 12 M pairs
    (640, 640, 1, 1600, 5000),       # eleven: 8 M
    (1600, 1120, 2, 1750, 2000),     # eleven, lists per bin: 3.5 M
])
def test_lists_at_the_most_pairs_of_one_digit(W, H, bins, lists, each, more):
    """Gaussians that cover the whole image: every list is the depth order of them all."""
    each += more
    g = torch.Generator().manual_seed(each)
    n = each + 1                     # (the last one emits nothing)
    means = torch.zeros(n, 3)
    means[:, 2] = 2.0 + 8.0 * torch.rand(n, generator=g)
    cam, st = forward(W, H, bins, means.to(DEV), torch.full((n, 3), 30.0, device=DEV))
    assert st.num_keys == lists * each
    order = torch.sort(means[:each, 2], stable=True).indices.to(torch.int32).to(DEV)
    assert torch.equal(st.ids.view(lists, each), order.expand(lists, each))
    tiles = cam.num_tiles
    assert torch.equal(st.ranges, torch.arange(tiles + 1, dtype=torch.int32, device=DEV) * each)
    if bins > 1:
        words = st.sorted_ids[st.num_keys:].view(lists, each)
        slots = torch.arange(1, lists + 1, dtype=torch.int32, device=DEV)
        assert torch.equal(words & 0xffff, slots[:, None].expand(lists, each))
        assert bool(((words >> 16) == (words[:, :1] >> 16)).all())


@pytest.mark.parametrize("W,H,scale", [(512, 390, 0.5), (512, 390, 1.0), (512, 512, 0.35), (512, 512, 0.6), (700, 700, 0.5),
                                       (745, 700, 0.5)])    # (2068 tiles: twelve bits)
def test_lists_of_many_pairs_equal_the_64_bit_route(W, H, scale):
    """Large Gaussians, some of them behind the camera, against a sort of 64-bit keys."""
    from ds_splat_amd import stages
    n = 60_000
    sc = make_scene("cfg4", n=n, width=W, height=H, sh_degree=0, seed=W + H)
    means = sc["means_3d"].clone()
    means[:500, 2] *= -1.0
    cam, st = forward(W, H, 1, means.to(DEV), (scale * sc["scales"]).to(DEV))
    k = st.num_keys
    print("%d pairs" % k)
    tiles = st.splats[:, 11].view(torch.int32).to(torch.int64).clone()
    tiles[-1] = 0
    assert k == int(tiles.sum()) > 1_000_000
    sums = torch.cat([tiles, torch.zeros((-n) % 256, dtype=torch.int64, device=DEV)]).view(-1, 256).sum(1).to(torch.int32)
    stages.scan_u32(sums)
    keys, ids = stages.emit_keys(cam, n, k, st.splats, sums)
    stages.sort_pairs(keys, ids, cam.num_tiles)
    assert torch.equal(ids, st.sorted_ids) and torch.equal(stages.tile_ranges(keys, cam.num_tiles), st.ranges)
