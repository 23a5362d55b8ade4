"""Adaptor with the calling convention of the original 3DGS rasterizer
(graphdeco-inria/diff-gaussian-rasterization), for trainers written against it:

    from ds_splat_amd.inria_compat import GaussianRasterizationSettings, GaussianRasterizer
    color, radii = GaussianRasterizer(settings)(means3D=..., means2D=..., opacities=..., shs=...,
                                                scales=..., rotations=...)

Differences from ``ds_splat.GaussianRasterizer`` (ds_splat/rasterizer.py:132-194 of the
reference), which this wraps:
  * keyword arguments in the original order (``opacities`` third, everything after optional);
  * the image comes back channel-first, ``[3, H, W]``, with the background composited:
    ``color = image + final_T * bg``.  The backward of the wrapped rasterizer already contains
    the gradient of exactly that term (cpp/gsplat/backward.cu:156-168 of the reference carries
    ``-T_final * ra * bg . v_out`` although its forward never adds the background), so the
    composited forward and the unchanged backward are consistent;
  * the settings tuple has no ``max_sh_degree`` (it is 3).
"""
from typing import NamedTuple

import torch

from .rasterizer import _render


class GaussianRasterizationSettings(NamedTuple):
    image_height: int
    image_width: int
    tanfovx: float
    tanfovy: float
    bg: torch.Tensor
    scale_modifier: float
    viewmatrix: torch.Tensor
    projmatrix: torch.Tensor
    sh_degree: int
    campos: torch.Tensor
    prefiltered: bool = False
    debug: bool = False


class GaussianRasterizer(torch.nn.Module):
    def __init__(self, raster_settings):
        super().__init__()
        self.raster_settings = raster_settings

    def forward(self, means3D, means2D, opacities, shs=None, colors_precomp=None, scales=None, rotations=None,
                cov3D_precomp=None):
        if (shs is None) == (colors_precomp is None):
            raise Exception("Please provide excatly one of either SHs or precomputed colors!")
        if ((scales is None or rotations is None) and cov3D_precomp is None) or \
                ((scales is not None or rotations is not None) and cov3D_precomp is not None):
            raise Exception("Please provide exactly one of either scale/rotation pair or precomputed 3D covariance!")
        s = self.raster_settings
        # (final_T reaches the image only through its product with the background, whose gradient the backward
        # kernel already accounts for; the blend kernels write and read the channel-first image themselves)
        return _render(means3D, means2D, shs, colors_precomp, opacities, scales, rotations, cov3D_precomp, s,
                       s.viewmatrix, s.projmatrix, 3, True)
