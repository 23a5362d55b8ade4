"""What torch's autograd machinery and a user's program do around a call: cameras written over, hooks on saved
tensors, recomputation, tracing, transforms of functions."""
import pytest
import torch
import torch.utils.checkpoint

from ds_splat_amd.synthetic import make_scene
from helpers import set_camera

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# image and gradients of two runs of one scene: the same terms, the gradients' added by float atomics in another order
RTOL, ATOL = 1e-3, 1e-4


def scene(camera="rotated"):
    sc = set_camera(make_scene("cfg0", n=3000, width=96, height=80, sh_degree=2, seed=7), camera)
    t = {k: (v.to(DEV) if isinstance(v, torch.Tensor) else v) for k, v in sc.items()}
    leaves = [t["means_3d"], torch.zeros_like(t["means_3d"]), t["shs"], t["opacities"], t["scales"] * 2.0, t["rotations"]]
    return sc, t, [x.clone().requires_grad_(True) for x in leaves]


def rasterizer(t, view=None, proj=None):
    from ds_splat import GaussianRasterizationSettings, GaussianRasterizer
    return GaussianRasterizer(GaussianRasterizationSettings(
        image_height=t["height"], image_width=t["width"], tanfovx=t["tanfovx"], tanfovy=t["tanfovy"], bg=t["bg"],
        scale_modifier=1.0, viewmatrix=t["viewmatrix"] if view is None else view,
        projmatrix=t["projmatrix"] if proj is None else proj, sh_degree=2, max_sh_degree=3, campos=t["campos"],
        prefiltered=False, debug=False))


def call(r, leaves):
    means, means2d, shs, opac, scales, rots = leaves
    return r(means, means2d, shs, None, opac, scales, rots, None)[0]


def wanted():
    _, t, leaves = scene()
    image = call(rasterizer(t), leaves)
    image.backward(t["v_image"])
    assert all(float(x.grad.abs().max()) > 0 for x in leaves)
    return image.detach(), [x.grad for x in leaves]


def check_grads(got, want):
    for g, w in zip(got, want):
        assert torch.allclose(g, w, rtol=RTOL, atol=ATOL * max(1.0, float(w.abs().max())))


def test_the_camera_may_be_written_over_before_the_backward():
    image_w, grads_w = wanted()
    _, t, leaves = scene()
    view, proj = t["viewmatrix"].clone(), t["projmatrix"].clone()
    image = call(rasterizer(t, view, proj), leaves)
    view.copy_(torch.eye(4))
    proj.zero_()
    image.backward(t["v_image"])
    assert torch.equal(image, image_w)
    check_grads([x.grad for x in leaves], grads_w)


def test_the_backgrounds_memory_may_be_another_one_at_the_backward():
    image_w, grads_w = wanted()
    _, t, leaves = scene()
    image = call(rasterizer(t), leaves)
    t["bg"].data, t["campos"].data = t["bg"].clone(), t["campos"].clone()
    image.backward(t["v_image"])
    check_grads([x.grad for x in leaves], grads_w)


@pytest.mark.parametrize("form", ["by_columns", "flat", "strided", "double"])
def test_forms_of_the_camera_matrices(form):
    image_w, grads_w = wanted()
    _, t, leaves = scene()

    def as_form(m):
        if form == "by_columns":
            return m.t().contiguous().t()
        if form == "flat":      # (transposing a vector leaves it: it holds the row-major matrix itself)
            return m.t().contiguous().view(16)
        if form == "strided":
            return torch.stack([m, m], 2)[:, :, 0]
        return m.double()

    image = call(rasterizer(t, as_form(t["viewmatrix"]), as_form(t["projmatrix"])), leaves)
    image.backward(t["v_image"])
    assert torch.equal(image, image_w)
    check_grads([x.grad for x in leaves], grads_w)
    with pytest.raises(RuntimeError):
        call(rasterizer(t, t["viewmatrix"][None]), leaves)


def test_saved_tensors_may_be_kept_on_the_host():
    image_w, grads_w = wanted()
    _, t, leaves = scene()
    with torch.autograd.graph.save_on_cpu():
        image = call(rasterizer(t), leaves)
    image.backward(t["v_image"])
    assert torch.equal(image, image_w)
    check_grads([x.grad for x in leaves], grads_w)


@pytest.mark.parametrize("reentrant", [False, True])
def test_recomputation_under_checkpointing(reentrant):
    image_w, grads_w = wanted()
    _, t, leaves = scene()
    r = rasterizer(t)
    image = torch.utils.checkpoint.checkpoint(lambda *xs: call(r, xs), *leaves, use_reentrant=reentrant)
    image.backward(t["v_image"])
    assert torch.equal(image, image_w)
    check_grads([x.grad for x in leaves], grads_w)


def test_tracing_is_refused():
    _, t, leaves = scene()
    with pytest.raises(RuntimeError):
        torch.jit.trace(lambda *xs: call(rasterizer(t), xs), tuple(x.detach() for x in leaves), check_trace=False)


def test_tangents_and_transforms_are_refused():
    import torch.autograd.forward_ad as fwd
    _, t, leaves = scene()
    plain = [x.detach() for x in leaves]
    r = rasterizer(t)
    for grad_mode in (True, False):
        with torch.set_grad_enabled(grad_mode), fwd.dual_level():
            dual = [fwd.make_dual(plain[0], torch.ones_like(plain[0]))] + plain[1:]
            with pytest.raises((RuntimeError, NotImplementedError)):
                call(r, dual)
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda m: call(r, [m] + plain[1:]).sum())(plain[0])
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda m: call(r, [m] + plain[1:]))(plain[0][None])


def test_counts_belong_to_the_call_that_waits_for_them():
    """A call that was begun and given up (an allocation failed) writes its counts all the same; the next call of
    the thread waits for its own."""
    import ctypes
    from ds_splat_amd import _native as N, stages
    lib, stream = N.load(), torch.cuda.current_stream().cuda_stream
    ptr = lambda x: ctypes.c_void_p(x.data_ptr() if x is not None else None)
    kept = []

    def begin(n, scale_mul):
        sc = make_scene("cfg0", n=n, width=256, height=192, seed=3)
        cam = stages.camera_from_scene(sc, torch.device(DEV), list_bin=2)
        t = [sc[k].to(DEV) for k in ("means_3d", "scales", "rotations", "opacities", "shs")]
        t[1] = t[1] * scale_mul
        order = stages.new_order(cam, n, DEV)
        bufs = [torch.empty((n, N.SPLAT_FLOATS), device=DEV), torch.empty(n, dtype=torch.int32, device=DEV),
                torch.empty(int(lib.dsx_num_blocks(n)), dtype=torch.int32, device=DEV)]
        kept.append((cam, t, order, bufs))
        N.check(lib.dsx_forward_project_begin(cam.ref, n, *map(ptr, t), ptr(None), ptr(None), ptr(bufs[0]),
                                              ptr(bufs[1]), ptr(None), ptr(bufs[2]), ptr(order), order.numel(),
                                              ptr(None), stream))
        return cam

    def counts(cam, n):
        two = (ctypes.c_int64 * 2)()
        N.check(lib.dsx_forward_project_counts(cam.ref, n, ctypes.byref(two), stream))
        return two[0], two[1]

    want = counts(begin(5000, 1.0), 5000)
    other = counts(begin(60000, 2.0), 60000)
    assert 0 < want[0] <= want[1] < other[0]
    for _ in range(20):
        begin(60000, 2.0)
        assert counts(begin(5000, 1.0), 5000) == want
    torch.cuda.synchronize()


@pytest.mark.parametrize("opacity_shape", [(-1, 1), (-1,)])
def test_functions_derived_from_the_rasterizers(opacity_shape):
    """DsRasterizerFunction is an autograd function: one derived from it, as it is or with an output more, gives the
    image and gradients of the call itself."""
    from ds_splat_amd import DsRasterizerFunction

    class Plain(DsRasterizerFunction):
        pass

    class WithTransmittance(DsRasterizerFunction):
        @staticmethod
        def forward(ctx, *args):
            image, radii, final_T = DsRasterizerFunction.run_forward(ctx, *args)
            ctx.mark_non_differentiable(radii, final_T)
            return image, radii, final_T

        @staticmethod
        def backward(ctx, v_image, _, __):
            return DsRasterizerFunction.backward(ctx, v_image, None)

    assert issubclass(DsRasterizerFunction, torch.autograd.Function)
    image_w, grads_w = wanted()
    for function in (DsRasterizerFunction, Plain, WithTransmittance):
        _, t, leaves = scene()
        means, means2d, shs, opac, scales, rots = leaves
        none = torch.empty(0, device=DEV)
        out = function.apply(means, means2d, shs, none, opac.reshape(opacity_shape), scales, rots, none,
                             rasterizer(t).settings_for_cpp_code)
        out[0].backward(t["v_image"], retain_graph=True)
        assert torch.equal(out[0], image_w)
        check_grads([x.grad for x in leaves], grads_w)
        out[0].backward(t["v_image"])                         # (the prepared accumulator serves the first one only)
        check_grads([x.grad for x in leaves], [2.0 * g for g in grads_w])
        with pytest.raises(RuntimeError):
            out[0].backward(t["v_image"])
        assert len(out) == 2 or float((out[2] - 1.0).abs().max()) > 0.01
