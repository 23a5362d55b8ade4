"""Python surface of the rasterizer: the same names, field order, argument order, returned
tensors and error behaviour as the reference's ``ds_splat/rasterizer.py`` (:7-194), on top of
the gfx950 library.

    from ds_splat import GaussianRasterizationSettings, GaussianRasterizer

``GaussianRasterizer(settings)(means_3d, means_2d, shs, colors_precomp, opacities, scales,
rotations, cov_3d_precomp)`` returns ``(image[H, W, 3], radii[N] int32)``; the image is HWC and
the background is not composited.  Backward returns gradients for the eight tensor inputs in
that order: v_means3d[N,3], v_means2d[N,3] (pixel units, third column zero), v_shs[N,B,3],
v_colors[N,3], v_opacity[N,1], v_scales[N,3], v_rotations[N,4], v_cov3d[N,6].
"""
from dataclasses import dataclass

import torch

from . import _native


class DsRasterizerFunction(torch.autograd.Function):
    """The differentiable call under ``GaussianRasterizer``.  ``raster_settings`` is what
    ``GaussianRasterizer.settings_for_cpp_code`` returns.

    ``DsRasterizerFunction.apply`` itself goes to the native autograd node (csrc/torch_ext.cpp: checks, forward and
    node without Python).  ``forward`` and ``backward`` are for functions derived from this one, whose ``apply`` is
    torch's: the same kernels, with the tensors kept on ``ctx``."""

    @classmethod
    def apply(cls, *args, **kwargs):
        return _apply(*args, **kwargs) if cls is DsRasterizerFunction else super().apply(*args, **kwargs)

    @staticmethod
    def forward(ctx, means_3d, means_2d, shs, colors_precomp, opacities, scales, rotations, cov_3d_precomp,
                raster_settings):
        image, radii, _ = DsRasterizerFunction.run_forward(ctx, means_3d, means_2d, shs, colors_precomp, opacities,
                                                           scales, rotations, cov_3d_precomp, raster_settings)
        return image, radii

    @staticmethod
    def run_forward(ctx, means_3d, means_2d, shs, colors_precomp, opacities, scales, rotations, cov_3d_precomp,
                    raster_settings):
        """The forward proper; also returns final_T (for functions that composite a background)."""
        s = raster_settings
        scalars = (int(s.image_height), int(s.image_width), float(s.tanfovx), float(s.tanfovy),
                   float(s.scale_modifier), int(s.sh_degree), int(s.max_sh_degree))
        list_bin = _native.default_list_bin()
        image, radii, splats, sorted_ids, ranges, final_T, final_idx, ctx.prepared_grads, k = \
            _native.load_torch_ext().render(means_3d, means_2d, shs, colors_precomp, opacities, scales, rotations,
                                            cov_3d_precomp, *scalars, s.view_matrix.t(), s.proj_matrix.t(), s.campos,
                                            s.bg, list_bin, any(ctx.needs_input_grad[:8]))
        ctx.num_keys, ctx.cam = k, scalars + (s.campos, s.bg, list_bin)
        ctx.save_for_backward(means_3d, shs, scales, rotations, cov_3d_precomp, splats, radii, ranges, sorted_ids,
                              final_T, final_idx)
        ctx.opacity_shape = opacities.shape
        ctx.mark_non_differentiable(radii)
        ctx.set_materialize_grads(False)
        return image, radii, final_T

    @staticmethod
    def backward(ctx, rendered_img_grad, _):
        if rendered_img_grad is None:   # nothing flows into the image (gradients are not materialised)
            return (None,) * 9
        wanted = sum(1 << i for i in range(8) if ctx.needs_input_grad[i])
        prepared, ctx.prepared_grads = ctx.prepared_grads, None   # good for one backward: it leaves sums behind
        grads = list(_native.load_torch_ext().backward(*ctx.saved_tensors, rendered_img_grad.contiguous(), prepared,
                                                       ctx.num_keys, wanted, *ctx.cam))
        if grads[4] is not None:
            grads[4] = grads[4].reshape(ctx.opacity_shape)
        return (*grads, None)


def _apply(means_3d, means_2d, shs, colors_precomp, opacities, scales, rotations, cov_3d_precomp, raster_settings):
    s = raster_settings
    return _render(means_3d, means_2d, shs, colors_precomp, opacities, scales, rotations, cov_3d_precomp, s,
                   s.view_matrix.t(), s.proj_matrix.t(), s.max_sh_degree, False)


def _render(means_3d, means_2d, shs, colors_precomp, opacities, scales, rotations, cov_3d_precomp, s, viewmatrix,
            projmatrix, max_sh_degree, planar):
    """``s``: any object with the scalar settings, ``campos`` and ``bg``; the matrices as the API's users hold them
    (transposed).  planar: the image is channel-first and has the background composited."""
    if torch.jit.is_tracing():  # (nothing but the allocations would be recorded)
        raise RuntimeError("the rasterizer cannot be recorded by torch.jit.trace")
    return _native.load_torch_ext().forward(
        means_3d, means_2d, shs, colors_precomp, opacities, scales, rotations, cov_3d_precomp, int(s.image_height),
        int(s.image_width), float(s.tanfovx), float(s.tanfovy), float(s.scale_modifier), int(s.sh_degree),
        int(max_sh_degree), viewmatrix, projmatrix, s.campos, s.bg, _native.default_list_bin(), planar)


@dataclass
class GaussianRasterizationSettings:
    image_height: int
    image_width: int
    tanfovx: float
    tanfovy: float
    bg: torch.Tensor
    scale_modifier: float
    viewmatrix: torch.Tensor
    projmatrix: torch.Tensor
    sh_degree: int
    max_sh_degree: int
    campos: torch.Tensor
    prefiltered: bool
    debug: bool


class _NativeSettings:
    """Plays the role of ``ds_splat_cuda.RasterizationSettings`` (cpp/rasterizer_python.cpp:5-19):
    the thirteen fields, with the two matrices already transposed to row-major."""
    __slots__ = ("image_height", "image_width", "tanfovx", "tanfovy", "bg", "scale_modifier", "view_matrix",
                 "proj_matrix", "sh_degree", "max_sh_degree", "campos", "prefiltered", "debug")


class GaussianRasterizer(torch.nn.Module):
    def __init__(self, raster_settings: GaussianRasterizationSettings):
        super().__init__()
        self._settings = raster_settings
        self._native_cache = None

    @property
    def settings_for_cpp_code(self):
        # the reference transposes both matrices on every call (ds_splat/rasterizer.py:147-148);
        # the result is kept here for as long as the settings hold the same, unmodified tensors.
        # The cache entry keeps the tensors themselves (compared with `is`: an address alone could
        # be a new tensor in a freed one's place) and their version counters; tensors without one
        # (created under torch.inference_mode) are transposed on every call.
        rs = self._settings
        try:
            versions = (rs.viewmatrix._version, rs.projmatrix._version)
        except RuntimeError:
            return self._build_native_settings()
        scalars = (rs.image_height, rs.image_width, rs.tanfovx, rs.tanfovy, rs.scale_modifier, rs.sh_degree,
                   rs.max_sh_degree, rs.prefiltered, rs.debug)
        c = self._native_cache
        if (c is not None and c[0] is rs and c[1] is rs.viewmatrix and c[2] is rs.projmatrix and c[3] is rs.bg
                and c[4] is rs.campos and c[5] == versions and c[6] == scalars):
            return c[7]
        s = self._build_native_settings()
        self._native_cache = (rs, rs.viewmatrix, rs.projmatrix, rs.bg, rs.campos, versions, scalars, s)
        return s

    def _build_native_settings(self):
        s = _NativeSettings()
        s.image_height = self._settings.image_height
        s.image_width = self._settings.image_width
        s.tanfovx = self._settings.tanfovx
        s.tanfovy = self._settings.tanfovy
        s.bg = self._settings.bg
        s.scale_modifier = self._settings.scale_modifier
        s.view_matrix = self._settings.viewmatrix.t().contiguous()
        s.proj_matrix = self._settings.projmatrix.t().contiguous()
        s.sh_degree = self._settings.sh_degree
        s.max_sh_degree = self._settings.max_sh_degree
        s.campos = self._settings.campos
        s.prefiltered = self._settings.prefiltered
        s.debug = self._settings.debug
        return s

    def forward(self, means_3d, means_2d, shs, colors_precomp, opacities, scales, rotations, cov_3d_precomp):
        # (the binding takes the matrices as they are: no transposed copies on the way)
        s = self._settings
        return _render(means_3d, means_2d, shs, colors_precomp, opacities, scales, rotations, cov_3d_precomp, s,
                       s.viewmatrix, s.projmatrix, s.max_sh_degree, False)
