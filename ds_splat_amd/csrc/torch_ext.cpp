// PyTorch binding over the C ABI of libdsx (include/dsx.h): it owns no kernels.  It plays the role of
// the reference's pybind module ds_splat_cuda (cpp/rasterizer_python.cpp:3-23), of the tensor
// plumbing in cpp/rasterizer_torch.cu:170-316 and of the autograd function in ds_splat/rasterizer.py:7-117:
// check the inputs, allocate the outputs as torch tensors, hand raw device pointers and the current
// stream to the library.  All of it is native: a small scene's forward takes the device 50 us, and
// the same steps in Python took the host as long.
#include <torch/extension.h>

#include <ATen/FuncTorchTLS.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include <algorithm>
#include <stdexcept>
#include <string>
#include <vector>

#include "dsx.h"

namespace
{

using OptTensor = c10::optional<at::Tensor>;

void check(int status)
{
    if(status != DSX_OK)
        throw std::runtime_error(dsx_error_string(status));
}

void require(bool ok, const char* message)
{
    if(!ok)
        throw std::runtime_error(message);
}

bool given(const OptTensor& t)
{
    return t.has_value() && t->defined() && t->numel() > 0;
}

const float* fptr(const OptTensor& t)
{
    return given(t) ? t->data_ptr<float>() : nullptr;
}

void* current_stream(const at::Device& dev)
{
    return c10::hip::getCurrentHIPStream(dev.index()).stream();
}

// What a render call is told besides the Gaussians.
struct Settings
{
    int64_t height, width;
    double tanfovx, tanfovy, scale_modifier;
    int64_t sh_degree, max_sh_degree;
    at::Tensor view, proj; // transposed, as the API's users hold them
    at::Tensor campos, bg;
    int64_t list_bin; // tiles per side of the bins of the tile lists (0: the library's choice)
    bool planar;      // [3,H,W] with the background composited instead of [H,W,3] without
};

struct Camera
{
    at::Tensor view, proj, campos, bg; // float32, on the device: kept alive for the call
    dsx_camera c;
    int32_t bin;  // of c.list_bin, without the flags
    bool planar;
};

// A matrix as the library takes it: 16 floats and whether they go by columns.  What the user holds is the
// transpose; a tensor that is itself the transposed view of a contiguous one needs no copy either.
at::Tensor matrix_of(const at::Tensor& t, const at::Device& dev, bool& by_columns)
{
    at::Tensor m = t.to(dev, at::kFloat);
    require(m.numel() == 16, "camera tensors must be 4x4, 4x4, [3], [3]");
    const bool square = m.dim() == 2 && m.size(0) == 4;
    if(square && m.is_contiguous())
    {
        by_columns = true;
        return m;
    }
    by_columns = false;
    if(square && m.stride(0) == 1 && m.stride(1) == 4)
        return m;
    return m.t().contiguous(); // (any other shape: what the reference's transposition makes of it, or its error)
}

// kept_view: the forward's copy of the view matrix, for the backward (which does not look at the projection
// matrix); null: both matrices as the settings hold them
Camera make_camera(const Settings& s, const at::Device& dev, const float* kept_view = nullptr)
{
    Camera cam;
    bool view_by_columns = false, proj_by_columns = false;
    if(kept_view == nullptr)
    {
        cam.view = matrix_of(s.view, dev, view_by_columns);
        cam.proj = matrix_of(s.proj, dev, proj_by_columns);
    }
    cam.campos = s.campos.to(dev, at::kFloat).contiguous();
    cam.bg = s.bg.to(dev, at::kFloat).contiguous();
    require(cam.campos.numel() >= 3 && cam.bg.numel() >= 3 && !(s.planar && cam.bg.numel() != 3),
            "camera tensors must be 4x4, 4x4, [3], [3]");
    cam.c.image_height = (int32_t)s.height;
    cam.c.image_width = (int32_t)s.width;
    cam.c.tanfovx = (float)s.tanfovx;
    cam.c.tanfovy = (float)s.tanfovy;
    cam.c.scale_modifier = (float)s.scale_modifier;
    cam.c.sh_degree = (int32_t)s.sh_degree;
    cam.c.max_sh_degree = (int32_t)s.max_sh_degree;
    cam.c.view = kept_view ? kept_view : cam.view.data_ptr<float>();
    cam.c.proj = kept_view ? kept_view : cam.proj.data_ptr<float>();
    cam.c.campos = cam.campos.data_ptr<float>();
    cam.c.bg = cam.bg.data_ptr<float>();
    require(s.list_bin == 0 || s.list_bin == 1 || s.list_bin == 2 || s.list_bin == 4 || s.list_bin == 8,
            "list_bin must be 0 (the library's choice), 1, 2, 4 or 8 tiles a side");
    cam.c.list_bin = (int32_t)s.list_bin | (view_by_columns ? DSX_VIEW_BY_COLUMNS : 0) |
                     (proj_by_columns ? DSX_PROJ_BY_COLUMNS : 0) | (s.planar ? DSX_PLANAR_IMAGE : 0) | DSX_PREPARE_ZEROS;
    cam.bin = (int32_t)s.list_bin;
    cam.planar = s.planar;
    return cam;
}

// The Gaussians of a call, in the API's order.
struct Inputs
{
    at::Tensor means3d, means2d;
    OptTensor shs, colors;
    at::Tensor opacities;
    OptTensor scales, quats, cov3d;
};

// The checks of rasterizer_forward_deepsense, cpp/rasterizer_torch.cu:176-190 and :124-129, and CHECK_INPUT,
// cpp/gsplat/bindings.h:9-16.
void check_input(const at::Tensor& t, const char* name)
{
    if(!t.is_cuda())
        throw std::runtime_error(std::string(name) + " must be a CUDA tensor");
    if(!t.is_contiguous())
        throw std::runtime_error(std::string(name) + " must be contiguous");
}

bool usable(const OptTensor& t)
{
    return t->is_contiguous() && t->is_cuda();
}

void check_float(const OptTensor& t, const char* name)
{
    if(given(t) && t->scalar_type() != at::kFloat)
        throw std::runtime_error(std::string(name) + " must be float32");
}

void validate(const Inputs& in, const Settings& s)
{
    check_input(in.means3d, "means_3d");
    check_input(in.means2d, "means_2d");
    check_input(in.opacities, "opacities");
    require(!given(in.shs) || usable(in.shs), "shs error");
    require(!given(in.scales) || usable(in.scales), "scales error");
    require(!given(in.quats) || usable(in.quats), "rotations error");
    require(given(in.cov3d) ? usable(in.cov3d)
                            : given(in.scales) && given(in.quats) && in.scales->size(0) == in.quats->size(0),
            "cov3D error");
    require(given(in.colors) ? usable(in.colors) : given(in.shs), "SHS error");
    check_float(in.means3d, "means_3d");
    check_float(in.opacities, "opacities");
    check_float(in.shs, "shs");
    check_float(in.scales, "scales");
    check_float(in.quats, "rotations");
    check_float(in.cov3d, "cov3D_precomp");
    check_float(in.colors, "colors_precomp");
    const int64_t n = in.means3d.numel() / 3;
    require(in.opacities.numel() == n, "opacities must have one entry per Gaussian");
    if(given(in.shs))
    {
        require(s.sh_degree >= 0 && s.sh_degree <= 3 && s.max_sh_degree == 3,
                "sh_degree must be in [0, 3] and max_sh_degree must be 3");
        const int64_t coeff = (s.sh_degree + 1) * (s.sh_degree + 1), most = (s.max_sh_degree + 1) * (s.max_sh_degree + 1);
        require(in.shs->dim() == 3 && in.shs->size(0) == n && in.shs->size(1) >= coeff && in.shs->size(1) == most &&
                    in.shs->size(2) == 3,
                "shs must have shape [N, (max_sh_degree+1)^2, 3]");
    }
    require(!given(in.scales) || (in.scales->numel() == 3 * n && given(in.quats) && in.quats->numel() == 4 * n),
            "scales must be [N,3] and rotations [N,4]");
    require(!given(in.cov3d) || in.cov3d->numel() == 6 * n, "cov3D_precomp must be [N,6]");
    require(!given(in.colors) || in.colors->numel() == 3 * n, "colors_precomp must be [N,3]");
}

// The user's matrices may be written over between a forward and its backward (one camera buffer for many views):
// the projection kernel keeps a copy of the one that the backward needs behind its records.
constexpr int64_t kViewRecords = (16 + DSX_SPLAT_FLOATS - 1) / DSX_SPLAT_FLOATS;

// What the forward leaves for the backward.
struct Rendered
{
    at::Tensor image, radii;
    at::Tensor splats;      // f32 [N + kViewRecords,12]: the records, then the view matrix that they were made with
    at::Tensor sorted_ids;  // i32 [dsx_sorted_ids_count(K)]
    at::Tensor ranges;      // i32 [dsx_ranges_count]
    at::Tensor final_T, final_idx;
    at::Tensor grads;       // the backward's accumulator, prepared by the blend kernel (or undefined)
    int64_t k = 0;
};

// image_only: what the image and the radii do not need need not be there
Rendered render(const Camera& cam, const Inputs& in, bool prepare_backward, bool image_only = false)
{
    const at::Device dev = in.means3d.device();
    const int64_t n = in.means3d.numel() / 3;
    const int32_t W = cam.c.image_width, H = cam.c.image_height, bin = cam.bin;
    const auto f32 = at::TensorOptions().dtype(at::kFloat).device(dev);
    const auto i32 = at::TensorOptions().dtype(at::kInt).device(dev);
    const auto u8 = at::TensorOptions().dtype(at::kByte).device(dev);
    void* s = current_stream(dev);

    Rendered r;
    r.radii = at::empty({n}, i32);
    auto new_image = [&] { return cam.planar ? at::empty({3, H, W}, f32) : at::empty({H, W, 3}, f32); };
    if(const size_t bytes = image_only ? dsx_render_bytes(n, W, H, bin) : 0)
    {
        at::Tensor scratch = at::empty({(int64_t)bytes}, u8);
        r.image = new_image();
        check(dsx_render(&cam.c, n, in.means3d.data_ptr<float>(), fptr(in.scales), fptr(in.quats), in.opacities.data_ptr<float>(),
                         fptr(in.shs), fptr(in.cov3d), fptr(in.colors), r.radii.data_ptr<int32_t>(), r.image.data_ptr<float>(),
                         scratch.data_ptr(), bytes, s));
        return r;
    }
    r.splats = at::empty({n + kViewRecords, DSX_SPLAT_FLOATS}, f32);
    // scratch of the first half: the projection's block sums and, behind them, the depth order
    const size_t sums_bytes = ((size_t)std::max<int64_t>(dsx_num_blocks(n), 1) * 4 + 255) & ~(size_t)255;
    const size_t order_bytes = dsx_order_bytes(n, W, H, bin);
    at::Tensor scratch = at::empty({(int64_t)(sums_bytes + order_bytes)}, u8);
    uint32_t* bs = reinterpret_cast<uint32_t*>(scratch.data_ptr());
    void* order = static_cast<char*>(scratch.data_ptr()) + sums_bytes;
    check(dsx_forward_project_begin(&cam.c, n, in.means3d.data_ptr<float>(), fptr(in.scales), fptr(in.quats),
                                    in.opacities.data_ptr<float>(), fptr(in.shs), fptr(in.cov3d), fptr(in.colors),
                                    r.splats.data_ptr<float>(), r.radii.data_ptr<int32_t>(), nullptr, bs, order,
                                    order_bytes,
                                    prepare_backward ? r.splats.data_ptr<float>() + n * DSX_SPLAT_FLOATS : nullptr, s));
    // (while the device counts the pairs: everything whose size does not depend on their number)
    r.ranges = at::empty({dsx_ranges_count(W, H, bin)}, i32);
    r.image = new_image();
    r.final_T = at::empty({H, W}, f32);
    r.final_idx = at::empty({H, W}, i32);
    if(prepare_backward && n > 0)
        r.grads = at::empty({(int64_t)(dsx_grads_bytes(n) / 4)}, f32);
    int64_t counts[2];
    check(dsx_forward_project_counts(&cam.c, n, counts, s));
    r.k = counts[0];
    r.sorted_ids = at::empty({dsx_sorted_ids_count(r.k, W, H, bin)}, i32);
    const size_t ws_bytes = dsx_workspace_bytes(n, r.k, W, H, bin);
    at::Tensor ws = at::empty({(int64_t)std::max<size_t>(ws_bytes, 1)}, u8);
    check(dsx_forward_finish(&cam.c, n, r.k, r.splats.data_ptr<float>(), order, r.sorted_ids.data_ptr<int32_t>(),
                             r.ranges.data_ptr<int32_t>(), r.image.data_ptr<float>(), r.final_T.data_ptr<float>(),
                             r.final_idx.data_ptr<int32_t>(), ws.data_ptr(), ws_bytes,
                             r.grads.defined() ? r.grads.data_ptr<float>() : nullptr, s));
    return r;
}

// v_mean3d[N,3], v_means2d[N,3], v_shs[N,B,3] (undefined when num_bases == 0), v_colors[N,3],
// v_opacity[N,1], v_scale[N,3], v_quat[N,4], v_cov3d[N,6].  Bit i of `wanted` asks for the i-th
// of them; the others are neither allocated nor written and come back undefined.
std::vector<at::Tensor> differentiate(const Camera& cam, int64_t k, int64_t num_bases, const at::Tensor& means3d,
                                      const OptTensor& scales, const OptTensor& quats, const OptTensor& cov3d,
                                      const at::Tensor& splats, const at::Tensor& radii, const at::Tensor& ranges,
                                      const at::Tensor& sorted_ids, const at::Tensor& final_T,
                                      const at::Tensor& final_idx, const at::Tensor& v_image, at::Tensor prepared,
                                      int64_t wanted)
{
    const at::Device dev = means3d.device();
    const int64_t n = means3d.numel() / 3;
    const auto f32 = at::TensorOptions().dtype(at::kFloat).device(dev);
    require(v_image.is_contiguous() && v_image.scalar_type() == at::kFloat &&
                v_image.numel() == (int64_t)cam.c.image_height * cam.c.image_width * 3 && v_image.device() == dev,
            "v_image must be a float32 tensor of the image's shape, on its device");
    auto out = [&](int bit, std::initializer_list<int64_t> shape) {
        return (wanted >> bit) & 1 ? at::empty(shape, f32) : at::Tensor();
    };
    auto ptr = [](const at::Tensor& t) { return t.defined() ? t.data_ptr<float>() : nullptr; };
    if(num_bases <= 0 || !((wanted >> 2) & 1))
        num_bases = 0;
    at::Tensor v_mean3d = out(0, {n, 3}), v_means2d = out(1, {n, 3});
    at::Tensor v_shs = num_bases > 0 ? at::empty({n, num_bases, 3}, f32) : at::Tensor();
    at::Tensor v_colors = out(3, {n, 3}), v_opacity = out(4, {n, 1});
    at::Tensor v_scale = out(5, {n, 3}), v_quat = out(6, {n, 4}), v_cov3d = out(7, {n, 6});
    // the accumulator that the forward prepared (sums zeroed, conics in place; good for one
    // backward), or a new one that the call fills
    const bool is_prepared = prepared.defined();
    at::Tensor grads = is_prepared ? prepared : at::empty({(int64_t)(dsx_grads_bytes(n) / 4)}, f32);
    check(dsx_backward(&cam.c, n, k, (int32_t)num_bases, means3d.data_ptr<float>(), fptr(scales), fptr(quats),
                       splats.data_ptr<float>(), fptr(cov3d), radii.data_ptr<int32_t>(), ranges.data_ptr<int32_t>(),
                       sorted_ids.numel() ? sorted_ids.data_ptr<int32_t>() : nullptr, final_T.data_ptr<float>(),
                       final_idx.data_ptr<int32_t>(), v_image.data_ptr<float>(), grads.data_ptr<float>(),
                       is_prepared ? 1 : 0, ptr(v_mean3d), ptr(v_means2d), ptr(v_shs), ptr(v_colors), ptr(v_opacity),
                       ptr(v_scale), ptr(v_quat), ptr(v_cov3d), current_stream(dev)));
    return {v_mean3d, v_means2d, v_shs, v_colors, v_opacity, v_scale, v_quat, v_cov3d};
}

// What the autograd node keeps besides its saved tensors.
struct NodeState : torch::CustomClassHolder
{
    Settings settings;   // (no address is kept: the tensors' memory may be another one by then)
    at::Tensor prepared; // the accumulator, until a backward has used it
    int64_t k = 0, num_bases = 0;
    std::vector<int64_t> opacity_shape;
    int edge[8]; // which of the node's inputs the i-th of the eight tensors is (-1: not given)
};

// The reference maps shs.size(-2) in {1,4,9,16} to a degree (anything else to 3), cpp/rasterizer_torch.cu:224-239,
// and gsplat/sh.cuh:18-29 maps the degree back to the number of bases.
int64_t bases_of(const OptTensor& shs)
{
    if(!given(shs))
        return 0;
    const int64_t b = shs->size(-2);
    return b == 1 || b == 4 || b == 9 || b == 16 ? b : 16;
}

class Rasterize : public torch::autograd::Function<Rasterize>
{
public:
    static torch::autograd::variable_list forward(torch::autograd::AutogradContext* ctx, const at::Tensor& means3d,
                                                  const at::Tensor& means2d, const OptTensor& shs,
                                                  const OptTensor& colors, const at::Tensor& opacities,
                                                  const OptTensor& scales, const OptTensor& quats,
                                                  const OptTensor& cov3d, const Settings& settings)
    {
        const Inputs in{means3d, means2d, shs, colors, opacities, scales, quats, cov3d};
        c10::DeviceGuard guard(means3d.device());
        auto state = c10::make_intrusive<NodeState>();
        Rendered r = render(make_camera(settings, means3d.device()), in, true);
        state->settings = settings;
        state->settings.view = state->settings.proj = at::Tensor(); // (the records hold the copy)
        state->prepared = r.grads;
        state->k = r.k;
        state->num_bases = bases_of(shs);
        state->opacity_shape = opacities.sizes().vec();
        const bool present[8] = {true, true, shs.has_value() && shs->defined(), colors.has_value() && colors->defined(), true,
                                 scales.has_value() && scales->defined(), quats.has_value() && quats->defined(),
                                 cov3d.has_value() && cov3d->defined()};
        for(int i = 0, e = 0; i < 8; ++i)
            state->edge[i] = present[i] ? e++ : -1;
        // the reference also keeps the 3-D covariances (cpp/rasterizer_torch.cu:207); the backward here
        // rebuilds them from scales and rotations, or reads the ones that were passed in
        ctx->save_for_backward({means3d, scales.value_or(at::Tensor()), quats.value_or(at::Tensor()),
                                cov3d.value_or(at::Tensor()), r.splats, r.radii, r.ranges, r.sorted_ids, r.final_T,
                                r.final_idx});
        ctx->saved_data["state"] = c10::IValue::make_capsule(state);
        ctx->mark_non_differentiable({r.radii});
        // no zero tensors for outputs that take no gradient (autograd would fill an int32[N] of zeros
        // for radii before every backward: a kernel launch in the middle of the step)
        ctx->set_materialize_grads(false);
        return {r.image, r.radii};
    }

    static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                   torch::autograd::variable_list grad_outputs)
    {
        torch::autograd::variable_list out(9);
        if(!grad_outputs[0].defined()) // nothing flows into the image (gradients are not materialised)
            return out;
        auto holder = ctx->saved_data["state"].toCapsule();
        NodeState& state = *static_cast<NodeState*>(holder.get());
        const auto saved = ctx->get_saved_variables();
        c10::DeviceGuard guard(saved[0].device());
        // the reference computes all eight gradients and autograd drops those of inputs that take
        // none (cpp/rasterizer_torch.cu:315, ds_splat/rasterizer.py:112); here the kernel is told
        // which ones are wanted and writes no others
        int64_t wanted = 0;
        for(int i = 0; i < 8; ++i)
            if(state.edge[i] >= 0 && ctx->needs_input_grad((size_t)state.edge[i]))
                wanted |= 1ll << i;
        at::Tensor prepared;
        std::swap(prepared, state.prepared); // good for one backward: it leaves sums behind
        const Camera camera = make_camera(state.settings, saved[0].device(),
                                          saved[4].data_ptr<float>() + saved[0].numel() / 3 * DSX_SPLAT_FLOATS);
        std::vector<at::Tensor> g =
            differentiate(camera, state.k, state.num_bases, saved[0], saved[1], saved[2], saved[3], saved[4],
                          saved[5], saved[6], saved[7], saved[8], saved[9], grad_outputs[0].contiguous(), prepared, wanted);
        if(g[4].defined() && g[4].sizes() != at::IntArrayRef(state.opacity_shape))
            g[4] = g[4].reshape(state.opacity_shape);
        std::copy(g.begin(), g.end(), out.begin());
        return out;
    }
};

// (image, radii).  Optional tensors may be None or empty.
std::tuple<at::Tensor, at::Tensor> forward(const at::Tensor& means3d, const at::Tensor& means2d, const OptTensor& shs,
                                           const OptTensor& colors, const at::Tensor& opacities, const OptTensor& scales,
                                           const OptTensor& quats, const OptTensor& cov3d, int64_t height, int64_t width,
                                           double tanfovx, double tanfovy, double scale_modifier, int64_t sh_degree,
                                           int64_t max_sh_degree, const at::Tensor& view, const at::Tensor& proj,
                                           const at::Tensor& campos, const at::Tensor& bg, int64_t list_bin, bool planar)
{
    const Settings settings{height, width, tanfovx, tanfovy, scale_modifier, sh_degree, max_sh_degree, view, proj,
                            campos, bg, list_bin, planar};
    const Inputs in{means3d, means2d, shs, colors, opacities, scales, quats, cov3d};
    validate(in, settings);
    // Without a gradient to take the node is passed by; transforms of functions and tangents of forward-mode
    // differentiation are not: torch refuses them at the node.
    if(const auto& transforms = at::functorch::functorchTLSAccessor())
        transforms->checkSupportsCppAutogradFunction();
    const bool grad_mode = at::GradMode::is_enabled();
    auto needs_node = [grad_mode](const OptTensor& t) {
        return t.has_value() && t->defined() && ((grad_mode && t->requires_grad()) || t->_fw_grad(0).defined());
    };
    if(!(needs_node(means3d) || needs_node(means2d) || needs_node(shs) || needs_node(colors) || needs_node(opacities) ||
         needs_node(scales) || needs_node(quats) || needs_node(cov3d)))
    {
        c10::DeviceGuard guard(means3d.device());
        Rendered r = render(make_camera(settings, means3d.device()), in, false, true);
        return {r.image, r.radii};
    }
    auto out = Rasterize::apply(means3d, means2d, shs, colors, opacities, scales, quats, cov3d, settings);
    return {out[0], out[1]};
}

// The two directions for an autograd function written in Python (DsRasterizerFunction and what derives from it): what
// the forward leaves, and the gradients from it.
std::tuple<at::Tensor, at::Tensor, at::Tensor, at::Tensor, at::Tensor, at::Tensor, at::Tensor, at::Tensor, int64_t>
render_parts(const at::Tensor& means3d, const at::Tensor& means2d, const OptTensor& shs, const OptTensor& colors,
             const at::Tensor& opacities, const OptTensor& scales, const OptTensor& quats, const OptTensor& cov3d,
             int64_t height, int64_t width, double tanfovx, double tanfovy, double scale_modifier, int64_t sh_degree,
             int64_t max_sh_degree, const at::Tensor& view, const at::Tensor& proj, const at::Tensor& campos,
             const at::Tensor& bg, int64_t list_bin, bool prepare_backward)
{
    const Settings settings{height, width, tanfovx, tanfovy, scale_modifier, sh_degree, max_sh_degree, view, proj,
                            campos, bg, list_bin, false};
    const Inputs in{means3d, means2d, shs, colors, opacities, scales, quats, cov3d};
    validate(in, settings);
    c10::DeviceGuard guard(means3d.device());
    Rendered r = render(make_camera(settings, means3d.device()), in, prepare_backward);
    return {r.image, r.radii, r.splats, r.sorted_ids, r.ranges, r.final_T, r.final_idx, r.grads, r.k};
}

std::vector<at::Tensor> backward_of_parts(const at::Tensor& means3d, const OptTensor& shs, const OptTensor& scales,
                                          const OptTensor& quats, const OptTensor& cov3d, const at::Tensor& splats,
                                          const at::Tensor& radii, const at::Tensor& ranges, const at::Tensor& sorted_ids,
                                          const at::Tensor& final_T, const at::Tensor& final_idx,
                                          const at::Tensor& v_image, const OptTensor& prepared, int64_t k, int64_t wanted,
                                          int64_t height, int64_t width, double tanfovx, double tanfovy,
                                          double scale_modifier, int64_t sh_degree, int64_t max_sh_degree,
                                          const at::Tensor& campos, const at::Tensor& bg, int64_t list_bin)
{
    const Settings settings{height, width, tanfovx, tanfovy, scale_modifier, sh_degree, max_sh_degree, at::Tensor(),
                            at::Tensor(), campos, bg, list_bin, false};
    c10::DeviceGuard guard(means3d.device());
    require(splats.size(0) == means3d.numel() / 3 + kViewRecords, "splats must be what render returned");
    const Camera camera = make_camera(settings, means3d.device(),
                                      splats.data_ptr<float>() + means3d.numel() / 3 * DSX_SPLAT_FLOATS);
    return differentiate(camera, k, bases_of(shs), means3d, scales, quats, cov3d, splats, radii, ranges, sorted_ids,
                         final_T, final_idx, v_image, prepared.value_or(at::Tensor()), wanted);
}

} // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m)
{
    m.doc() = "torch binding of libdsx (gfx950 3D-Gaussian-Splatting rasterizer)";
    // (torch's own wrappers: errors come back as torch's exceptions, and a Python exception that a hook on saved
    // tensors raises, as recomputation under checkpointing does, passes through as it is)
    m.def("forward", torch::wrap_pybind_function_no_gil(forward), "projection, tile lists and blend; differentiable");
    m.def("render", torch::wrap_pybind_function_no_gil(render_parts),
          "the forward without a node: (image, radii, splats, sorted_ids, ranges, final_T, final_idx, grads, k)");
    m.def("backward", torch::wrap_pybind_function_no_gil(backward_of_parts), "the eight gradients from what render left");
    m.def("version", []() { return dsx_version(); });
}
