"""Kernels that are chosen by size, at the sizes where the choice and their tiles end."""
import numpy as np
import pytest
import torch

import test_gpu_pipeline
import test_gpu_stages
from ds_splat_amd.synthetic import make_scene
from helpers import comparable_gaussians

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("depths", ["spread", "equal", "ties", "culled"])
@pytest.mark.parametrize("n", [1, 255, 2048, 2049, 4097, 16383, 16384, 16385])
def test_depth_order_of_few_gaussians(n, depths):
    """The depth order is the stable order of the depth bits, its block offsets are the exclusive sums of the tile
    counts in that order."""
    from ds_splat_amd import stages
    sc = make_scene("cfg0", n=n, width=200, height=120, seed=5)
    means = sc["means_3d"].clone()
    if depths == "equal":
        means[:, 2] = 4.0
    elif depths == "ties":
        means[::7, 2] = means[::7, 2].round()
    elif depths == "culled":
        means[:, 0] += 1e4
    cam = stages.camera_from_scene(sc, DEV, list_bin=1)
    order = stages.new_order(cam, n, DEV)
    splats, radii, _, _ = stages.project_fwd(cam, means.to(DEV), sc["scales"].to(DEV), sc["rotations"].to(DEV),
                                             sc["opacities"].to(DEV), sc["shs"].to(DEV), order=order)
    keys = order[:4 * n].cpu().numpy().view(np.uint32).copy()
    perm, offsets = stages.depth_order(cam, n, order)
    perm, offsets = perm.cpu().numpy().astype(np.int64), offsets.cpu().numpy().astype(np.int64)
    assert (keys == 0xffffffff).all() == (depths == "culled" or n == 1)   # (the last Gaussian emits nothing)
    assert (perm == np.argsort(keys, kind="stable")).all()
    touched = splats[:, 11].contiguous().view(torch.int32).cpu().numpy().astype(np.int64)
    touched[keys == 0xffffffff] = 0
    sums = np.add.reduceat(touched[perm], np.arange(0, n, 256))
    assert (offsets[:len(sums)] == np.cumsum(sums) - sums).all()


@pytest.mark.parametrize("bin_side", [1, 2, 8])
@pytest.mark.parametrize("n,W,H,scale_mul,flip,giants", [
    (3, 48, 40, 0.1, 0, 0),               # runs shorter than a thread's four outputs
    (257, 100, 70, 0.2, 5, 0),            # a block of 256 Gaussians and one more
    (700, 300, 200, 1.0, 90, 2),          # shares that end inside a Gaussian's run, behind the camera and in front
    (400, 140000, 64, 20.0, 0, 3),        # rectangles of 8750 columns: their ends need more than 13 bits
])
def test_emission_of_four_pairs_to_a_thread(oracle, list_bin, bin_side, n, W, H, scale_mul, flip, giants):
    if bin_side == 1:
        test_gpu_stages.test_tile_lists_bit_exact(oracle, list_bin, n, W, H, scale_mul, flip, giants=giants)
    else:
        test_gpu_stages.test_binned_tile_lists_vs_oracle(oracle, list_bin, bin_side, n, W, H, scale_mul, flip, giants,
                                                         "identity")


@pytest.mark.parametrize("n,W,H,scale_mul,flip,bin_side", [
    (3000, 240, 272, 3.0, 40, 1),         # 255 tiles: eight bits, the last of them; 256: nine
    (3000, 256, 256, 3.0, 40, 1),
    (3000, 112, 1168, 3.0, 40, 1),        # 511 and 512: nine and ten
    (3000, 512, 256, 3.0, 40, 1),
    (3000, 528, 496, 3.0, 40, 1),         # 1023 and 1024: ten and eleven (two digits a thread)
    (3000, 512, 512, 3.0, 40, 1),
    (1, 512, 512, 1.0, 0, 1),
    (3000, 368, 1424, 3.0, 40, 1),        # 2047: eleven, the last of them
    (9000, 512, 512, 3.0, 40, 1),         # 2, 4, 8 and 12 keys a thread and more tiles than compute units
    (20000, 512, 512, 3.0, 40, 1),
    (40000, 512, 512, 3.0, 40, 1),
    (90000, 512, 512, 3.0, 40, 1),
    (131072, 512, 512, 1.0, 40, 1),       # one digit up to here, two beyond
    (131073, 512, 512, 1.0, 40, 1),
    (131073, 256, 512, 1.0, 40, 1),
    (20000, 1920, 1080, 3.0, 40, 4),      # bins: 510, 920 and 2040 lists
    (20000, 1280, 720, 3.0, 40, 2),
    (20000, 1920, 1080, 3.0, 40, 2),
])
def test_partition_by_one_wide_digit(oracle, list_bin, n, W, H, scale_mul, flip, bin_side):
    """Lists of nine to eleven bits: one pass where eight bits a pass would take two, at the edges of the widths and of
    the rule that says for how many Gaussians; ids, ranges and masks bit for bit the oracle's."""
    if bin_side == 1:
        test_gpu_stages.test_tile_lists_bit_exact(oracle, list_bin, n, W, H, scale_mul, flip)
    else:
        test_gpu_stages.test_binned_tile_lists_vs_oracle(oracle, list_bin, bin_side, n, W, H, scale_mul, flip, 0, "identity")


@pytest.mark.parametrize("depths", ["uniform", "octaves", "too_many_octaves", "equal", "both_signs", "none"])
@pytest.mark.parametrize("n", [262144, 262145, 530001])
def test_depth_order_over_a_known_range(n, depths):
    """The depth order inside a whole forward: by buckets where the depths have one sign and are neither thin nor wide, else in
    three digits where they lie within sixteen octaves and have one sign, else in four."""
    from ds_splat_amd import stages
    sc = make_scene("cfg0", n=n, width=64, height=48, seed=9)
    g = torch.Generator().manual_seed(n)
    u = torch.rand(n, generator=g)
    means = torch.zeros(n, 3)
    means[:, 2] = {"uniform": 2.0 + 18.0 * u, "octaves": 0.02 * 2.0 ** (14.5 * u), "both_signs": 3.0 + u,
                   "too_many_octaves": 0.015 * 2.0 ** (17.0 * u), "equal": 4.0 + 0.0 * u, "none": 2.0 + u}[depths]
    if depths == "both_signs":       # (a mirrored point behind the camera passes the frustum test)
        sc["projmatrix"][2, 2], sc["projmatrix"][3, 2] = -sc["projmatrix"][2, 2].abs(), sc["projmatrix"][3, 2].abs()
        sc["projmatrix"][:, 2] = torch.tensor([0.0, 0.0, 0.0, 0.5])
        sc["projmatrix"][:, 3] = torch.tensor([0.0, 0.0, 0.0, 1.0])
        means[::3, 2] *= -1.0
    if depths == "none":
        means[:, 0] = 1e4
    scales = (means[:, 2:].abs() * 1e-3).expand(n, 3).contiguous()
    cam = stages.camera_from_scene(sc, DEV, list_bin=1)
    seen = {}

    def look(order, n_, k):
        perm, offsets = stages.depth_order_view(n_, order)
        seen["perm"], seen["offsets"] = perm.cpu().numpy().astype(np.int64), offsets.cpu().numpy().astype(np.int64)

    _, st = stages.forward(cam, means.to(DEV), scales.to(DEV), sc["rotations"].to(DEV), sc["opacities"].to(DEV),
                           sc["shs"].to(DEV), after_project=look)
    touched = st.splats[:, 11].contiguous().view(torch.int32).cpu().numpy().astype(np.int64)
    touched[-1] = 0
    bits = st.splats[:, 2].contiguous().view(torch.int32).cpu().numpy().view(np.uint32)
    keys = np.where(touched > 0, bits, np.uint32(0xffffffff))
    emitting = keys != 0xffffffff
    assert emitting.sum() == (0 if depths == "none" else n - 1)
    if depths == "both_signs":
        assert (keys[emitting] >> 31).any() and not (keys[emitting] >> 31).all()
    if emitting.any() and depths != "both_signs":
        span = int(keys[emitting].max() >> 16) - int(keys[emitting].min() >> 16) + 1
        assert (span << 16 >= 1 << 27) == (depths == "too_many_octaves")
    perm = np.argsort(keys, kind="stable")
    assert (seen["perm"] == perm).all()
    sums = np.add.reduceat(touched[perm], np.arange(0, n, 256))
    assert (seen["offsets"] == np.concatenate([[0], np.cumsum(sums)])).all()


@pytest.mark.parametrize("out", ["third", "first_half", "last_half", "nearly_all", "in_runs"])
@pytest.mark.parametrize("n,bins", [(262145, 1), (530001, 1), (3200000, 4)])
def test_depth_order_of_a_cloud_that_is_partly_out_of_sight(n, bins, out):
    """A whole forward puts the Gaussians that emit nothing behind the others, by index, and the others alone are sorted: the order,
    the offsets and the pairs that are emitted are what they are without that.  (The launches that order by buckets here; the
    first digit pass, which does so too, in the next test.)"""
    from ds_splat_amd import stages
    sc = make_scene("cfg0", n=n, width=96, height=64, sh_degree=0, seed=9)
    g = torch.Generator().manual_seed(n)
    i = torch.arange(n)
    gone = {"third": torch.rand(n, generator=g) < 0.35, "first_half": i < n // 2, "last_half": i >= n // 2,
            "nearly_all": i % 50000 != 7, "in_runs": (i // 5000) % 2 == 0}[out]
    means = torch.zeros(n, 3)
    means[:, 2] = 2.0 + 18.0 * torch.rand(n, generator=g)
    means[::11, 2] = 5.0                                       # ties
    means[gone, 0] = 1e4
    scales = (means[:, 2:] * 1e-3).expand(n, 3).contiguous()
    cam = stages.camera_from_scene(sc, DEV, list_bin=bins)
    seen = {}

    def look(order, n_, k):
        perm, offsets = stages.depth_order_view(n_, order)
        seen["perm"], seen["offsets"] = perm.cpu().numpy().astype(np.int64), offsets.cpu().numpy().astype(np.int64)

    _, st = stages.forward(cam, means.to(DEV), scales.to(DEV), sc["rotations"].to(DEV), sc["opacities"].to(DEV),
                           sc["shs"].to(DEV), after_project=look)
    touched = st.splats[:, 11].contiguous().view(torch.int32).cpu().numpy().astype(np.int64)
    touched[-1] = 0
    bits = st.splats[:, 2].contiguous().view(torch.int32).cpu().numpy().view(np.uint32)
    keys = np.where(touched > 0, bits, np.uint32(0xffffffff))
    emitting = int((keys != 0xffffffff).sum())
    assert emitting == int((~gone[:-1]).sum()) and 0 < emitting < n - 1
    perm = np.argsort(keys, kind="stable")
    assert (seen["perm"] == perm).all()
    if bins == 1:
        sums = np.add.reduceat(touched[perm], np.arange(0, n, 256))
        assert (seen["offsets"] == np.concatenate([[0], np.cumsum(sums)])).all()
        assert (np.bincount(st.sorted_ids.cpu().numpy(), minlength=n) == touched).all()
    else:
        assert set(np.unique(st.ids.cpu().numpy()).tolist()) == set(np.nonzero(touched)[0].tolist())


@pytest.mark.parametrize("out", ["third", "first_half", "last_half", "nearly_all", "in_runs"])
@pytest.mark.parametrize("n", [262145, 530001, 3200000])
def test_digit_passes_over_a_cloud_that_is_partly_out_of_sight(n, out):
    """The first digit pass puts the Gaussians that emit nothing behind the others, by index, and the others alone go through the
    rest (what runs where the buckets do not, and with other limits on the waits)."""
    from ds_splat_amd import stages
    sc = make_scene("cfg0", n=64, width=96, height=64, sh_degree=0, seed=9)
    g = torch.Generator().manual_seed(n)
    i = torch.arange(n)
    gone = {"third": torch.rand(n, generator=g) < 0.35, "first_half": i < n // 2, "last_half": i >= n // 2,
            "nearly_all": i % 50000 != 7, "in_runs": (i // 5000) % 2 == 0}[out]
    means = torch.zeros(n, 3)
    means[:, 2] = 2.0 + 18.0 * torch.rand(n, generator=g)
    means[::11, 2] = 5.0                                       # ties
    means[gone, 0] = 1e6
    rotations, opacities, shs = torch.zeros(n, 4), torch.full((n, 1), 0.5), torch.zeros(n, 16, 3)
    rotations[:, 0] = 1.0
    cam = stages.camera_from_scene(sc, DEV, list_bin=1)
    order = stages.new_order(cam, n, DEV)
    splats, _, _, _ = stages.project_fwd(cam, *(x.to(DEV) for x in (means, (means[:, 2:] * 1e-2).expand(n, 3).contiguous(), rotations,
                                                                    opacities, shs)), order=order)
    keys = order[:4 * n].view(torch.int32).cpu().numpy().view(np.uint32).copy()
    assert int((keys != 0xffffffff).sum()) == int((~gone[:-1]).sum())
    perm, offsets = (x.cpu().numpy().astype(np.int64) for x in stages.depth_order_bounded(cam, n, order, sort_polls=1 << 17))
    # (the tiles of the first digit pass count themselves in the fourth word before the flag)
    assert int(order.view(torch.int32)[stages.sort_flag_indices(cam, n, 0, order, None)[0] - 4].item()) > 0
    want = np.argsort(keys, kind="stable")
    assert (perm == want).all()
    touched = splats[:, 11].contiguous().view(torch.int32).cpu().numpy().astype(np.int64)
    touched[keys == 0xffffffff] = 0
    assert (offsets == np.concatenate([[0], np.cumsum(np.add.reduceat(touched[want], np.arange(0, n, 256)))])).all()


@pytest.mark.parametrize("polls", [-1, 0])
@pytest.mark.parametrize("bins", [1, 4])
@pytest.mark.parametrize("n,seen", [(24577, 1.0), (28673, 0.5), (262145, 0.3), (530001, 1.0), (1300001, 0.6)])
def test_block_offsets_of_workgroups_that_do_not_wait(n, seen, bins, polls):
    """A workgroup that does not look for another's sum, or finds it missing, adds up the other's rectangles itself: the
    offsets are those of workgroups that wait, where the last share, the last run and the last Gaussian that emits end anywhere."""
    from ds_splat_amd import stages
    sc = make_scene("cfg0", n=n, width=520, height=300, sh_degree=0, seed=9)
    means = sc["means_3d"].clone()
    gone = torch.rand(n, generator=torch.Generator().manual_seed(n)) >= seen
    means[gone, 0] = 1e4
    cam = stages.camera_from_scene(sc, DEV, list_bin=bins)
    order = stages.new_order(cam, n, DEV)
    splats, _, _, _ = stages.project_fwd(cam, means.to(DEV), sc["scales"].to(DEV), sc["rotations"].to(DEV),
                                         sc["opacities"].to(DEV), sc["shs"].to(DEV), order=order)
    again = order.clone()
    perm, offsets = (x.clone() for x in stages.depth_order_bounded(cam, n, order))
    perm2, offsets2 = stages.depth_order_bounded(cam, n, again, offset_polls=polls)
    assert torch.equal(perm, perm2) and torch.equal(offsets, offsets2)
    assert int(offsets[-1]) > 0 and bool((offsets[1:] >= offsets[:-1]).all())
    if bins == 1:
        touched = splats[:, 11].contiguous().view(torch.int32).to(torch.int64)
        touched[-1] = 0
        assert int(offsets[-1]) == int(touched.sum())


@pytest.mark.parametrize("n,W", [(24577, 520), (24577, 4200), (530001, 520), (530001, 4200)])
def test_a_depth_sort_that_gives_up_stays_inside_its_buffer(n, W):
    """Tiles that do not look at their predecessors' statuses: with four digits and three, rectangles carried and
    gathered (beyond 255 columns of tiles), the places that their keys take, and those of what later passes make of
    the places that nobody wrote, lie inside the buffer, and the flag says that the order is wrong."""
    from ds_splat_amd import stages
    sc = make_scene("cfg0", n=n, width=W, height=40, sh_degree=0, seed=9)
    means = sc["means_3d"].clone()
    means[torch.rand(n, generator=torch.Generator().manual_seed(n)) < 0.6, 0] = 1e4
    cam = stages.camera_from_scene(sc, DEV, list_bin=1)
    size, guard = stages.new_order(cam, n, DEV).numel(), 1 << 22
    buffer = torch.full((size + guard,), 0xfe, dtype=torch.uint8, device=DEV)
    order = buffer[:size]
    stages.project_fwd(cam, means.to(DEV), sc["scales"].to(DEV), sc["rotations"].to(DEV), sc["opacities"].to(DEV),
                       sc["shs"].to(DEV), order=order)
    keys = order[:4 * n].cpu().numpy().view(np.uint32).copy()
    perm, _ = stages.depth_order_bounded(cam, n, order, sort_polls=-1)
    flag = int(order.view(torch.int32)[stages.sort_flag_indices(cam, n, 0, order, None)[0]].item())
    assert bool((buffer[size:] == 0xfe).all())
    assert flag == 1 and not (perm.cpu().numpy() == np.argsort(keys, kind="stable")).all()


@pytest.mark.parametrize("pixels_per_lane", [1, 4])
def test_bin_lists_beyond_two_to_the_thirty(blend_form, pixels_per_lane):
    """Positions of a bin's list that a 32-bit byte offset does not reach: the same lists, moved behind 2^30 others,
    give the same image and gradients (the places they would be mistaken for hold other Gaussians)."""
    from ds_splat_amd import stages
    blend_form(pixels_per_lane)
    sc = make_scene("cfg0", n=5000, width=160, height=112, sh_degree=0, seed=4)
    cam = stages.camera_from_scene(sc, DEV, list_bin=4)
    t = {k: (v.to(DEV) if isinstance(v, torch.Tensor) else v) for k, v in sc.items()}
    n = sc["n"]
    image, st = stages.forward(cam, t["means_3d"], t["scales"] * 2.0, t["rotations"], t["opacities"], t["shs"])
    grads = stages.blend_bwd(cam, n, st.lists, st.sorted_ids, st.splats, st.final_T, st.final_idx, t["v_image"])
    k, ahead = st.num_keys, 1 << 30
    if torch.cuda.mem_get_info()[0] < 12 * ahead:
        pytest.skip("needs 12 GiB of free GPU memory")
    moved = torch.empty(2 * (ahead + k), dtype=torch.int32, device=DEV)
    moved[:k], moved[ahead + k:ahead + 2 * k] = st.ids.flip(0), st.sorted_ids[k:].flip(0)
    moved[ahead:ahead + k], moved[2 * ahead + k:] = st.ids, st.sorted_ids[k:]
    lists = st.lists.clone()
    stages.split_lists(cam, lists)["bins"].add_(ahead)
    image2, T2, idx2 = stages.blend_fwd(cam, lists, moved, st.splats)
    assert torch.equal(image2, image) and torch.equal(T2, st.final_T) and torch.equal(idx2, st.final_idx)
    grads2 = stages.blend_bwd(cam, n, lists, moved, st.splats, T2, idx2, t["v_image"])
    # (the same terms; float atomics add them in another order)
    assert torch.allclose(grads2[:, :9], grads[:, :9], rtol=1e-3, atol=1e-4 * float(grads[:, :9].abs().max()))
    assert float(grads[:, :9].abs().max()) > 0


@pytest.mark.parametrize("bins", [1, 4])
@pytest.mark.parametrize("pixels_per_lane", [1, 4])
@pytest.mark.parametrize("W,H", [(323, 197), (64, 48)])
def test_channel_first_image_in_every_blend_form(oracle, blend_form, list_bin, pixels_per_lane, bins, W, H):
    """The adaptor's image and gradients (planes of the image stored and read by the blend kernels, background
    composited) from both forms of the kernels and both kinds of lists, where planes and rows end inside a quad of
    lanes and inside a tile, and where they do not."""
    from ds_splat_amd import inria_compat
    blend_form(pixels_per_lane)
    list_bin(bins)
    bg = np.array([0.3, 0.6, 0.1], np.float32)
    sc = make_scene("cfg1", n=12000, width=W, height=H, sh_degree=1, seed=31)
    t = {k: (v.to(DEV) if isinstance(v, torch.Tensor) else v) for k, v in sc.items()}
    p = dict(means=t["means_3d"].clone(), means2d=torch.zeros_like(t["means_3d"]), shs=t["shs"].clone(),
             opac=t["opacities"].clone(), scales=t["scales"] * 2.0, rots=t["rotations"].clone())
    p = {k: v.requires_grad_(True) for k, v in p.items()}
    settings = inria_compat.GaussianRasterizationSettings(
        image_height=H, image_width=W, tanfovx=sc["tanfovx"], tanfovy=sc["tanfovy"], bg=torch.from_numpy(bg).to(DEV),
        scale_modifier=1.0, viewmatrix=t["viewmatrix"], projmatrix=t["projmatrix"], sh_degree=1, campos=t["campos"])
    color, radii = inria_compat.GaussianRasterizer(settings)(
        means3D=p["means"], means2D=p["means2d"], opacities=p["opac"], shs=p["shs"], scales=p["scales"],
        rotations=p["rots"])
    color.backward(t["v_image"].permute(2, 0, 1))
    torch.cuda.synchronize()
    img_o, radii_o, S, B = test_gpu_pipeline.oracle_run(oracle, sc, 2.0, bg=bg)
    assert color.shape == (3, H, W) and color.is_contiguous() and (radii.cpu().numpy() == radii_o).all()
    ok = S["margin"] > 1e-4
    assert ok.mean() > 0.98
    want = img_o + S["final_T"][..., None] * bg
    np.testing.assert_allclose(color.detach().permute(1, 2, 0).cpu().numpy()[ok], want[ok], rtol=1e-4, atol=1e-5)
    fT, fidx, _ = test_gpu_pipeline.gpu_forward_state(sc, 2.0)
    gok = comparable_gaussians(S, B, W, fT, fidx)
    assert gok.mean() > 0.8
    test_gpu_pipeline.check_grads(p, B, gok, "channel first %d %d" % (pixels_per_lane, bins))


@pytest.mark.parametrize("depths", ["spread", "ties"])
@pytest.mark.parametrize("n", [18433, 24575, 24576, 24577])
def test_depth_order_up_to_twelve_tiles_of_keys(n, depths):
    """The same with 37 to 49 workgroups of 512 ranks, of which the last has one rank, all but one or all."""
    test_depth_order_of_few_gaussians(n, depths)


@pytest.mark.parametrize("kind,n,W,H", [
    ("round", 1, 16, 16),        # (the last Gaussian emits nothing)
    ("round", 57, 33, 17),       # a round of 56 entries and none; tiles cut off at both edges
    ("round", 66, 16, 16),       # a round of 64 entries and one more
    ("round", 250, 64, 64),      # the workgroup form's round of 248 and one more
    ("round", 962, 16, 16),      # the round of 960 of sixteen wavefronts and one more
    ("opaque", 2500, 21, 35),    # pixels that stop in the first round of several, and in the middle of four entries
    ("thin", 250, 131, 77),      # long splats at all angles: blocks that their middles and their ends reach
    ("tiny", 6000, 97, 50),      # splats that reach one block or two
    ("black", 2000, 80, 61),     # colours of zero: an entry that is nobody's must not be taken for one that is
    ("clamped", 900, 70, 50),    # opacities at and above the clamps of both directions
])
@pytest.mark.parametrize("bins", [1, 4])
@pytest.mark.parametrize("pixels_per_lane", [0, 1, 4])  # (0: sixteen wavefronts per tile, for lists per tile)
def test_entries_in_the_lists_of_the_blocks_that_they_reach(oracle, blend_form, pixels_per_lane, bins, kind, n, W, H):
    """Image, last indices and gradients of every form against the oracle, which walks every entry for every pixel: an
    entry that were missing in a block's list would be missing in its pixels."""
    import test_gpu_opacities as o
    blend_form(pixels_per_lane)
    sc = make_scene("cfg0", n=n, width=W, height=H, sh_degree=0, seed=n)
    g = torch.Generator().manual_seed(n)
    sc["scales"] = sc["scales"] * 2.0
    if kind == "round":
        sc["opacities"] = sc["opacities"] * 0.1     # (no pixel stops: every entry is walked)
        sc["means_3d"][:, :2] *= 0.3
    elif kind == "thin":
        # (up to 15 pixels, widths below one: the exponent's terms, up to 1/2 3.3 15^2 = 370, cancel and cost alpha
        # 370 2^-24 = 2e-5 of itself for each rounding)
        sc["scales"] = torch.exp(torch.randn(n, 1, generator=g) * 0.3 - 1.8) * torch.tensor([[1.0, 0.02, 0.02]])
    elif kind == "tiny":
        sc["scales"] = sc["scales"] * 0.1
    elif kind == "black":
        sc["shs"][:, 0] = -5.0
    elif kind == "clamped":
        sc["opacities"] = torch.tensor([0.98, 0.99, 0.995, 0.999, 1.0])[torch.randint(5, (n, 1), generator=g)]
    A = o.arrays(sc)
    s = o.scene_settings(sc)
    img, radii, ost = oracle.forward(s, A["means_3d"], A["scales"], A["rotations"], A["opacities"], A["shs"])
    S = oracle.state(s, ost, n)
    B = oracle.backward(s, ost, 16, A["means_3d"], A["scales"], A["rotations"], A["opacities"], A["v_image"])
    oracle.free(ost)
    image, final_T, final_idx, out = o.gpu_run(sc, bins)
    ok = S["margin"] > 1e-4
    assert ok.mean() > 0.97
    assert (final_idx[ok] == S["final_idx"][ok]).all()
    np.testing.assert_allclose(image[ok], img[ok], rtol=1e-4, atol=1e-5)
    gok = comparable_gaussians(S, B, W, final_T, final_idx)
    assert gok.mean() > 0.8
    bounds = oracle.gradient_bounds(s, 16, A["means_3d"], A["scales"], A["rotations"], S["conic"], S["cov3d"], radii,
                                    B["abs_sums"], rel=1e-4)
    got = {k: out[k].cpu().numpy() for k in ("v_mean3d", "v_means2d", "v_shs", "v_opacity", "v_scale", "v_quat")}
    o.check_grads_against_bounds(got, B, bounds, gok, kind)


@pytest.mark.parametrize("depths", ["uniform", "two", "layers", "nearly_equal", "cluster", "seldom", "one", "both_signs"])
@pytest.mark.parametrize("n", [512, 513, 1537, 40961, 131072, 131073])
def test_depth_order_and_counts_in_one_launch(n, depths):
    """Up to 131072 Gaussians a workgroup finds its own 512 ranks: where a bin of the range holds many more keys than that, or keys
    that differ in the last bits only, or hardly any key emits, or the range goes beyond the largest number there is; and just beyond.
    Order, offsets, and the lists, ranges and histograms of tiles and of bins are those of the digit passes."""
    from ds_splat_amd import stages
    W, H = 200, 120
    sc = make_scene("cfg0", n=n, width=W, height=H, sh_degree=0, seed=9)
    u = torch.rand(n, generator=torch.Generator().manual_seed(n))
    means = torch.zeros(n, 3)
    means[:, 2] = {"two": torch.where(u < 0.5, 2.0, 19.0), "layers": 2.0 + (u * 20.0).floor(), "nearly_equal": 4.0 + u * 1e-5,
                   "cluster": torch.where(u < 0.9, 4.0 + u * 1e-4, 2.0 + 18.0 * u)}.get(depths, 2.0 + 18.0 * u)
    if depths == "both_signs":       # (a mirrored point behind the camera passes the frustum test)
        sc["projmatrix"][:, 2] = torch.tensor([0.0, 0.0, 0.0, 0.5])
        sc["projmatrix"][:, 3] = torch.tensor([0.0, 0.0, 0.0, 1.0])
        means[::3, 2] *= -1.0
    if depths == "seldom":
        means[u > 0.01, 0] = 1e4
    if depths == "one":
        means[torch.arange(n) != n // 3, 0] = 1e4
    scales = (means[:, 2:].abs() * 1e-2).expand(n, 3).contiguous()
    for bins in (1, 4):
        cam = stages.camera_from_scene(sc, DEV, list_bin=bins)
        order = stages.new_order(cam, n, DEV)
        splats, _, _, _ = stages.project_fwd(cam, means.to(DEV), scales.to(DEV), sc["rotations"].to(DEV),
                                             sc["opacities"].to(DEV), sc["shs"].to(DEV), order=order)
        keys = order[:4 * n].cpu().numpy().view(np.uint32).copy()
        again = order.clone()
        perm, offsets = (x.clone() for x in stages.depth_order(cam, n, order))
        perm2, offsets2 = stages.depth_order_bounded(cam, n, again, sort_polls=1 << 17)      # (the digit passes)
        emitting = keys != 0xffffffff
        assert emitting.any()
        if depths == "both_signs":
            assert keys[emitting].max() >> 31 and not keys[emitting].min() >> 31 and not emitting[-1]
        assert (perm.cpu().numpy() == np.argsort(keys, kind="stable")).all()
        assert torch.equal(perm, perm2) and torch.equal(offsets, offsets2)
        if bins == 1:
            touched = splats[:, 11].contiguous().view(torch.int32).to(torch.int64)
            touched[-1] = 0
            assert int(offsets[-1]) == int(touched.sum())
        k = int(offsets[-1])
        ids, lists = stages.tile_lists(cam, n, k, order, return_lists=True)
        ids2, lists2 = stages.tile_lists(cam, n, k, again, return_lists=True)
        ready = cam.num_tiles + 2 + (0 if bins == 1 else 2 + -(-W // 64) * -(-H // 64))
        assert torch.equal(ids, ids2) and torch.equal(lists[:ready], lists2[:ready])


@pytest.mark.parametrize("bins", [1, 2, 8])
@pytest.mark.parametrize("n,W,H", [
    (2000, 3840, 2160), (21888, 3840, 2160), (21889, 3840, 2160), (131072, 3840, 2160),     # (32777 cells)
    (17825, 2700, 2300), (17826, 2700, 2300), (9675, 1920, 1080), (9676, 1920, 1080), (5760, 400, 300), (5761, 400, 300),
    (6001, 16, 4000)])
def test_counts_of_large_images_beside_the_order(n, W, H, bins):
    """Up to 131072 Gaussians the tiles are counted beside the order: by one workgroup up to 5500 Gaussians and one more for every two
    of the grid's cells, by several beyond, on grids whose cells and tiles fill no whole rounds of its threads.  Ranges, histograms and
    lists are those of the launches that the digit passes have beside them."""
    from ds_splat_amd import stages
    sc = make_scene("cfg0", n=n, width=W, height=H, sh_degree=0, seed=n)
    sc["means_3d"][:, :2] *= 1.5                  # (some out of sight, many cut off at the edges)
    sc["means_3d"][::97] *= -1.0
    cam = stages.camera_from_scene(sc, DEV, list_bin=bins)
    order = stages.new_order(cam, n, DEV)
    splats, _, _, _ = stages.project_fwd(cam, *(sc[k].to(DEV) for k in ("means_3d", "scales", "rotations", "opacities", "shs")),
                                         order=order)
    again = order.clone()
    perm, offsets = (x.clone() for x in stages.depth_order(cam, n, order))
    perm2, offsets2 = stages.depth_order_bounded(cam, n, again, sort_polls=1 << 17)      # (the digit passes)
    assert torch.equal(perm, perm2) and torch.equal(offsets, offsets2)
    k = int(offsets[-1])
    ids, lists = stages.tile_lists(cam, n, k, order, return_lists=True)
    ids2, lists2 = stages.tile_lists(cam, n, k, again, return_lists=True)
    ready = cam.num_tiles + 2 + (0 if bins == 1 else 2 + -(-W // (16 * bins)) * -(-H // (16 * bins)))
    assert k > n // 4 and torch.equal(ids, ids2) and torch.equal(lists[:ready], lists2[:ready])
    touched = splats[:, 11].contiguous().view(torch.int32).to(torch.int64)
    touched[-1] = 0
    assert int(lists[cam.num_tiles]) == int(touched.sum())


@pytest.mark.parametrize("depths", ["uniform", "layers", "octaves", "seldom", "one", "runs", "two", "thin", "cloud"])
@pytest.mark.parametrize("n", [131073, 262145, 524289, 1048577, 2097153, 3145729, 4194305])
def test_depth_order_by_buckets(n, depths):
    """From 131073 Gaussians on the order is made by buckets: each number of keys to a workgroup and of bins, where hardly any key
    emits, whole stretches do not, and where hundreds of depths are equal (which a bucket sorts another way).  Order and offsets are
    those of the digit passes, which are also what runs where a bin holds too many keys or the range is thin."""
    from ds_splat_amd import stages
    W, H = 200, 120
    sc = make_scene("cfg0", n=64, width=W, height=H, sh_degree=0, seed=9)
    u = torch.rand(n, generator=torch.Generator().manual_seed(n))
    layers = n // 700                 # (700 keys to a layer; with the depth, 128 layers at least)
    means = torch.zeros(n, 3)
    means[:, 2] = {"two": torch.where(u < 0.5, 2.0, 19.0), "thin": 4.0 + 0.01 * u, "octaves": 0.02 * 2.0 ** (14.5 * u),
                   "cloud": torch.where(u < 0.9, 4.0 + 0.1 * u, 0.02 * 2.0 ** (14.5 * u)),
                   "layers": 2.0 + (u * layers).floor() * (18.0 / layers)}.get(depths, 2.0 + 18.0 * u)
    index = torch.arange(n)
    gone = {"seldom": index % 100 != 7, "one": index != n // 3, "runs": (index // 3000) % 2 == 0}.get(depths, index < 0)
    means[gone, 0] = 1e6
    scales = (means[:, 2:].abs() * 1e-2).expand(n, 3).contiguous()
    rotations, opacities, shs = torch.zeros(n, 4), torch.full((n, 1), 0.5), torch.zeros(n, 16, 3)
    rotations[:, 0] = 1.0
    for bins in (1, 4):
        cam = stages.camera_from_scene(sc, DEV, list_bin=bins)
        order = stages.new_order(cam, n, DEV)
        splats, _, _, _ = stages.project_fwd(cam, means.to(DEV), scales.to(DEV), rotations.to(DEV), opacities.to(DEV),
                                             shs.to(DEV), order=order)
        keys = order[:4 * n].view(torch.int32).cpu().numpy().view(np.uint32).copy()
        again = order.clone()
        perm, offsets = (x.clone() for x in stages.depth_order_bounded(cam, n, order))
        # (the tiles of a first digit pass count themselves in the fourth word before the flag)
        tiles = int(order.view(torch.int32)[stages.sort_flag_indices(cam, n, 0, order, None)[0] - 4].item())
        assert (tiles == 0) == (depths not in ("two", "thin", "one", "cloud"))
        perm2, offsets2 = stages.depth_order_bounded(cam, n, again, sort_polls=1 << 17)      # (the digit passes)
        assert (keys != 0xffffffff).any()
        assert torch.equal(perm, perm2) and torch.equal(offsets, offsets2)
        if bins == 1:
            assert (perm.cpu().numpy() == np.argsort(keys, kind="stable")).all()
            touched = splats[:, 11].contiguous().view(torch.int32).to(torch.int64)
            touched[-1] = 0
            assert int(offsets[-1]) == int(touched.sum())


@pytest.mark.parametrize("n", [8388608, 8388609])
def test_depth_order_where_there_are_as_many_buckets_as_can_be(n):
    """4096 buckets of 2048 are the most: with one Gaussian more the digit passes run."""
    from ds_splat_amd import stages
    sc = make_scene("cfg0", n=64, width=200, height=120, sh_degree=0, seed=9)
    cam = stages.camera_from_scene(sc, DEV, list_bin=1)
    g = torch.Generator(device=DEV)
    g.manual_seed(n)
    means = torch.zeros(n, 3, device=DEV)
    means[:, 2] = 2.0 + 18.0 * torch.rand(n, generator=g, device=DEV)
    scales = (means[:, 2:] * 1e-2).expand(n, 3).contiguous()
    rotations, opacities, shs = torch.zeros(n, 4, device=DEV), torch.full((n, 1), 0.5, device=DEV), torch.zeros(n, 16, 3, device=DEV)
    rotations[:, 0] = 1.0
    order = stages.new_order(cam, n, DEV)
    splats, _, _, _ = stages.project_fwd(cam, means, scales, rotations, opacities, shs, order=order)
    keys = order[:4 * n].view(torch.int32).to(torch.int64) & 0xffffffff
    assert int((keys == 0xffffffff).sum()) == 1
    perm, offsets = stages.depth_order_bounded(cam, n, order)
    tiles = int(order.view(torch.int32)[stages.sort_flag_indices(cam, n, 0, order, None)[0] - 4].item())
    assert (tiles == 0) == (n == 8388608)
    want = torch.sort(keys, stable=True)[1]
    assert torch.equal(perm.to(torch.int64), want)
    touched = splats[:, 11].contiguous().view(torch.int32).to(torch.int64)
    touched[-1] = 0
    blocks = torch.nn.functional.pad(touched[want], (0, -n % 256)).view(-1, 256).sum(1).cumsum(0)
    assert int(offsets[0]) == 0 and torch.equal(offsets[1:].to(torch.int64), blocks)


@pytest.mark.parametrize("gone", ["none", "two_of_three", "all_but_300", "all"])
@pytest.mark.parametrize("n", [140001, 262145])
def test_block_offsets_of_depths_of_both_signs_and_what_emits_nothing(n, gone):
    """Four digit passes, behind which the offsets are summed over those that emit only: the others lie behind them and add nothing."""
    from ds_splat_amd import stages
    sc = make_scene("cfg0", n=64, width=200, height=120, sh_degree=0, seed=9)
    sc["projmatrix"][:, 2] = torch.tensor([0.0, 0.0, 0.0, 0.5])         # (a mirrored point behind the camera passes the frustum test)
    sc["projmatrix"][:, 3] = torch.tensor([0.0, 0.0, 0.0, 1.0])
    cam = stages.camera_from_scene(sc, DEV, list_bin=1)
    means = torch.zeros(n, 3)
    means[:, 2] = 2.0 + 18.0 * torch.rand(n, generator=torch.Generator().manual_seed(n))
    means[::2, 2] *= -1.0
    index = torch.arange(n)
    means[{"none": index < 0, "two_of_three": index % 3 != 1, "all_but_300": (index < 5000) | (index >= 5300), "all": index >= 0}[gone], 0] = 1e6
    rotations, opacities, shs = torch.zeros(n, 4), torch.full((n, 1), 0.5), torch.zeros(n, 16, 3)
    rotations[:, 0] = 1.0
    order = stages.new_order(cam, n, DEV)
    splats, _, _, _ = stages.project_fwd(cam, *(x.to(DEV) for x in (means, (means[:, 2:].abs() * 1e-2).expand(n, 3).contiguous(),
                                                                    rotations, opacities, shs)), order=order)
    keys = order[:4 * n].view(torch.int32).cpu().numpy().view(np.uint32).copy()
    assert (keys != 0xffffffff).any() == (gone != "all")
    perm, offsets = (x.cpu().numpy().astype(np.int64) for x in stages.depth_order_bounded(cam, n, order))
    want = np.argsort(keys, kind="stable")
    assert (perm == want).all()
    touched = splats[:, 11].contiguous().view(torch.int32).cpu().numpy().astype(np.int64)
    touched[keys == 0xffffffff] = 0
    assert (offsets == np.concatenate([[0], np.cumsum(np.add.reduceat(touched[want], np.arange(0, n, 256)))])).all()


@pytest.mark.parametrize("n,crowd,buckets", [
    (200001, 2900, True), (200001, 3200, True), (200001, 3600, None), (200001, 3900, None), (200001, 3970, None), (200001, 4050, False),
    (600001, 1900, True), (600001, 2500, True), (600001, 3900, None), (600001, 4050, False),
    (1100000, 3000, True), (3000000, 400000, False), (4200001, 3000, True), (4200001, 100000, False)])
def test_depth_order_by_buckets_of_a_crowded_bin(n, crowd, buckets):
    """A bin of the range may hold up to what a bucket has room for (4032 keys) less what else its bucket gets, which the launch that
    fills the buckets finds out before it does; beyond, it counts the digits of the passes instead.  Order and offsets are the
    same, whichever way they are made; crowd: depths that are equal (some more lie in the same bin); buckets: certainly or not."""
    from ds_splat_amd import stages
    sc = make_scene("cfg0", n=64, width=200, height=120, sh_degree=0, seed=9)
    cam = stages.camera_from_scene(sc, DEV, list_bin=1)
    u = torch.rand(n, generator=torch.Generator().manual_seed(n + crowd))
    means = torch.zeros(n, 3)
    means[:, 2] = 2.0 + 18.0 * u
    means[torch.randperm(n, generator=torch.Generator().manual_seed(crowd))[:crowd], 2] = 7.0
    means[n // 5::11, 0] = 1e6            # (some emit nothing)
    means[means[:, 2] == 7.0, 0] = 0.0
    scales = (means[:, 2:].abs() * 1e-2).expand(n, 3).contiguous()
    rotations, opacities, shs = torch.zeros(n, 4), torch.full((n, 1), 0.5), torch.zeros(n, 16, 3)
    rotations[:, 0] = 1.0
    order = stages.new_order(cam, n, DEV)
    stages.project_fwd(cam, *(x.to(DEV) for x in (means, scales, rotations, opacities, shs)), order=order)
    keys = order[:4 * n].view(torch.int32).cpu().numpy().view(np.uint32).copy()
    again = order.clone()
    perm, offsets = (x.clone() for x in stages.depth_order_bounded(cam, n, order))
    # (the tiles of a first digit pass count themselves in the fourth word before the flag)
    tiles = int(order.view(torch.int32)[stages.sort_flag_indices(cam, n, 0, order, None)[0] - 4].item())
    assert buckets is None or (tiles == 0) == buckets
    perm2, offsets2 = stages.depth_order_bounded(cam, n, again, sort_polls=1 << 17)      # (the digit passes)
    assert torch.equal(perm, perm2) and torch.equal(offsets, offsets2)
    assert (perm.cpu().numpy() == np.argsort(keys, kind="stable")).all()


@pytest.mark.parametrize("skip", [0, 8])
@pytest.mark.parametrize("n", [3000, 131072, 200001])
def test_depth_order_of_a_buffer_that_is_aligned_to_eight_bytes(n, skip):
    """The `order` buffer may begin at any multiple of eight bytes (as include/dsx.h says), whichever kernels order it."""
    from ds_splat_amd import stages
    sc = make_scene("cfg0", n=n, width=200, height=120, seed=5)
    cam = stages.camera_from_scene(sc, DEV, list_bin=1)
    room = torch.empty(stages.new_order(cam, n, DEV).numel() + 16, dtype=torch.uint8, device=DEV)
    order = room[skip:skip + room.numel() - 16]
    assert room.data_ptr() % 16 == 0 and order.data_ptr() % 16 == skip
    splats, _, _, _ = stages.project_fwd(cam, sc["means_3d"].to(DEV), sc["scales"].to(DEV), sc["rotations"].to(DEV),
                                         sc["opacities"].to(DEV), sc["shs"].to(DEV), order=order)
    keys = order[:4 * n].cpu().numpy().view(np.uint32).copy()
    perm, offsets = (x.cpu().numpy().astype(np.int64) for x in stages.depth_order_bounded(cam, n, order))
    want = np.argsort(keys, kind="stable")
    assert (keys != 0xffffffff).sum() > n // 2 and (perm == want).all()
    touched = splats[:, 11].contiguous().view(torch.int32).cpu().numpy().astype(np.int64)
    touched[keys == 0xffffffff] = 0
    sums = np.add.reduceat(touched[want], np.arange(0, n, 256))
    assert (offsets == np.concatenate([[0], np.cumsum(sums)])).all()
