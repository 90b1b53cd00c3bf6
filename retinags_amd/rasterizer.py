"""Host-side mirror of the reference's rasterizer module
(K/diff_gaussian_rasterization_half_gaussian/__init__.py with
K = rasterization_kernels/diff-gaussian-rasterization-half-gaussian): the same
names, argument order, return values and error behaviour, driving PyTorch-ROCm
tensors through the C ABI of librgs_gfx950.so.

PyTorch only provides device memory, the current stream and the autograd graph here; every
stage of the rasterizer runs in the HIP library, and the steps around its calls (workspaces,
argument tables, autograd nodes) are csrc/host.cpp.
"""
from __future__ import annotations

import ctypes as C
from typing import NamedTuple

import torch
import torch.nn as nn

from ._capi import lib, check, ptr
from . import _host
from ._host import GeometryStage  # noqa: F401


def cpu_deep_copy_tuple(input_tuple):
    copied_tensors = [item.cpu().clone() if isinstance(item, torch.Tensor) else item for item in input_tuple]
    return tuple(copied_tensors)


class GaussianRasterizationSettings(NamedTuple):
    """K/diff_gaussian_rasterization_half_gaussian/__init__.py:166-181, field for field."""
    image_height: int
    image_width: int
    tanfovx: float
    tanfovy: float
    bg: torch.Tensor
    scale_modifier: float
    viewmatrix: torch.Tensor
    projmatrix: torch.Tensor
    projmatrix_inv: torch.Tensor
    range_low: torch.Tensor
    range_up: torch.Tensor
    sh_degree: int
    campos: torch.Tensor
    prefiltered: bool
    debug: bool


def _dev_f32(t: torch.Tensor, device, name: str) -> torch.Tensor:
    """Contiguous fp32 tensor on `device`; the reference calls .contiguous() on every
    argument (K/rasterize_points.cu:99-121)."""
    if not isinstance(t, torch.Tensor):
        raise TypeError(f"{name} must be a tensor")
    if t.numel() == 0:
        return t
    if t.device != device or t.dtype != torch.float32:
        t = t.to(device=device, dtype=torch.float32)
    return t.contiguous()


_EMPTY = torch.Tensor([])  # stands for an absent input, as in the reference (it becomes a null pointer)


def _stream_ptr(device) -> C.c_void_p:
    return C.c_void_p(torch.cuda.current_stream(device).cuda_stream)


def _rasterize_forward(bg, means3D, colors_precomp, opacities, scales, rotations, scale_modifier, cov3Ds_precomp,
                       viewmatrix, projmatrix, projmatrix_inv, range_low, range_up, tanfovx, tanfovy, image_height,
                       image_width, sh, sh_degree, campos, prefiltered, debug):
    """Counterpart of RasterizeGaussiansCUDA_hgs (K/rasterize_points.cu:35-125): allocates the
    outputs and the three workspaces, runs the forward, returns the same 8-tuple."""
    return _host.rasterize_forward(bg, means3D, colors_precomp, opacities, scales, rotations, float(scale_modifier),
                                   cov3Ds_precomp, viewmatrix, projmatrix, projmatrix_inv, range_low, range_up,
                                   float(tanfovx), float(tanfovy), int(image_height), int(image_width), sh, int(sh_degree),
                                   campos, bool(prefiltered), bool(debug))


def _gradient_outputs(P, M, device, scratch=()):
    """The eight dense gradient tensors of K/rasterize_points.cu:165-174, uninitialised (the library
    writes every row of them: those of Gaussians that were not rendered as zeros), and the
    backward's scratch for the per-Gaussian sums (the library clears it).  Each is an allocation of
    its own: what a caller keeps, a leaf's .grad or the means2D gradient for densification
    statistics, holds nothing else.  `scratch` names those of the eight that the caller
    hands to nobody (the colour gradient when the colours come from SH, the covariance gradient
    when it comes from scale and rotation): they are not made at all (None), and the library
    does not write them.  The backward nodes make the same arrays without coming here, unless
    another function has been put in the place of this one: that one is asked."""
    return _host.gradient_outputs(P, M, device, scratch)


_host.set_original_gradient_outputs(_gradient_outputs)


def _rasterize_backward(bg, means3D, radii, colors_precomp, scales, rotations, scale_modifier, cov3Ds_precomp,
                        viewmatrix, projmatrix, projmatrix_inv, range_low, range_up, tanfovx, tanfovy, grad_color,
                        grad_depth, grad_alpha, sh, sh_degree, campos, geomBuffer, num_rendered, binningBuffer,
                        imgBuffer, alpha, debug):
    """Counterpart of RasterizeGaussiansBackwardCUDA_hgs (K/rasterize_points.cu:127-220);
    returns the same 8 tensors in the same order."""
    return _host.rasterize_backward(bg, means3D, radii, colors_precomp, scales, rotations, float(scale_modifier),
                                    cov3Ds_precomp, viewmatrix, projmatrix, projmatrix_inv, range_low, range_up,
                                    float(tanfovx), float(tanfovy), grad_color, grad_depth, grad_alpha, sh, int(sh_degree),
                                    campos, geomBuffer, int(num_rendered), binningBuffer, imgBuffer, alpha, bool(debug))


def _mark_visible(means3D, viewmatrix, projmatrix):
    """Counterpart of markVisible_hgs (K/rasterize_points.cu:222-241)."""
    device = means3D.device
    if not means3D.is_cuda:
        raise RuntimeError("the rasterizer needs its inputs on a GPU (device memory)")
    P = int(means3D.shape[0])
    present = torch.zeros((P,), dtype=torch.bool, device=device)
    if P != 0:
        means3D = _dev_f32(means3D, device, "means3D")
        viewmatrix = _dev_f32(viewmatrix, device, "viewmatrix")
        projmatrix = _dev_f32(projmatrix, device, "projmatrix")
        with torch.cuda.device(device):
            check(lib.rgs_mark_visible(P, ptr(means3D), ptr(viewmatrix), ptr(projmatrix), ptr(present),
                                       _stream_ptr(device)))
    return present


def rasterize_gaussians(means3D, means2D, sh, colors_precomp, opacities, scales, rotations, cov3Ds_precomp,
                        raster_settings, geometry=None):
    return _RasterizeGaussians.apply(means3D, means2D, sh, colors_precomp, opacities, scales, rotations,
                                     cov3Ds_precomp, raster_settings, geometry)


def _forward_in_debug(args, run):
    """A forward in debug mode: its arguments are kept aside and written to a file if it fails."""
    cpu_args = cpu_deep_copy_tuple(args)  # copy them before they can be corrupted
    try:
        return run()
    except Exception as ex:
        torch.save(cpu_args, "snapshot_fw.dump")
        print("\nAn error occured in forward. Please forward snapshot_fw.dump for debugging.")
        raise ex


def _backward_in_debug(args, run):
    """The backward of a call in debug mode: its arguments are kept aside and written to a file if it fails."""
    cpu_args = cpu_deep_copy_tuple(args)
    try:
        return run()
    except Exception as ex:
        torch.save(cpu_args, "snapshot_bw.dump")
        print("\nAn error occured in backward. Writing snapshot_bw.dump for debugging.\n")
        raise ex


class _RasterizeGaussians(torch.autograd.Function):
    """K/diff_gaussian_rasterization_half_gaussian/__init__.py:44-164: forward and backward of one call as an autograd
    function.  apply() goes through the native one (RasterizeCall of csrc/host.cpp), which does the same without coming back
    to Python; forward and backward are for those who call them or derive from them, and a derived class's apply() runs them."""

    @classmethod
    def apply(cls, means3D, means2D, sh, colors_precomp, opacities, scales, rotations, cov3Ds_precomp, raster_settings,
              geometry=None):
        if cls is not _RasterizeGaussians:
            return super().apply(means3D, means2D, sh, colors_precomp, opacities, scales, rotations, cov3Ds_precomp,
                                 raster_settings, geometry)
        run = lambda: _host.rasterize(means3D, means2D, sh, colors_precomp, opacities, scales, rotations, cov3Ds_precomp,
                                      raster_settings, geometry)
        if not raster_settings.debug or geometry is not None:
            return run()
        return _forward_in_debug(_forward_arguments(means3D, sh, colors_precomp, opacities, scales, rotations, cov3Ds_precomp,
                                                    raster_settings), run)

    @staticmethod
    def forward(ctx, means3D, means2D, sh, colors_precomp, opacities, scales, rotations, cov3Ds_precomp,
                raster_settings, geometry=None):
        if geometry is not None:
            outs = _host.rasterize_forward_from_stage(geometry, means3D, raster_settings)
        else:
            args = _forward_arguments(means3D, sh, colors_precomp, opacities, scales, rotations, cov3Ds_precomp, raster_settings)
            run = lambda: _rasterize_forward(*args)
            outs = _forward_in_debug(args, run) if raster_settings.debug else run()
        num_rendered, color, depth, alpha, radii, geomBuffer, binningBuffer, imgBuffer = outs

        ctx.set_materialize_grads(False)  # an output that took no part in the loss comes back as None, not as a tensor of zeros
        ctx.raster_settings = raster_settings
        ctx.num_rendered = num_rendered
        ctx.save_for_backward(colors_precomp, means3D, scales, rotations, cov3Ds_precomp, radii, sh, geomBuffer,
                              binningBuffer, imgBuffer, alpha)
        ctx.mark_non_differentiable(radii)
        return color, radii, depth, alpha

    @staticmethod
    def backward(ctx, grad_color, grad_radii, grad_depth, grad_alpha):
        rs = ctx.raster_settings
        (colors_precomp, means3D, scales, rotations, cov3Ds_precomp, radii, sh, geomBuffer, binningBuffer, imgBuffer,
         alpha) = ctx.saved_tensors
        # The reference's C++ side always receives dense tensors; here an absent depth / alpha gradient goes down as a null
        # pointer, which the library takes as zero.
        if grad_color is None:
            grad_color = torch.zeros((3,) + tuple(alpha.shape[1:]), dtype=alpha.dtype, device=alpha.device)
        args = (rs.bg, means3D, radii, colors_precomp, scales, rotations, rs.scale_modifier, cov3Ds_precomp, rs.viewmatrix,
                rs.projmatrix, rs.projmatrix_inv, rs.range_low, rs.range_up, rs.tanfovx, rs.tanfovy, grad_color,
                _EMPTY if grad_depth is None else grad_depth, _EMPTY if grad_alpha is None else grad_alpha, sh, rs.sh_degree,
                rs.campos, geomBuffer, ctx.num_rendered, binningBuffer, imgBuffer, alpha, rs.debug)
        run = lambda: _rasterize_backward(*args)
        (grad_means2D, grad_colors_precomp, grad_opacities, grad_means3D, grad_cov3Ds_precomp, grad_sh, grad_scales,
         grad_rotations) = _backward_in_debug(args, run) if rs.debug else run()
        return (grad_means3D, grad_means2D, grad_sh if sh.numel() else None,
                grad_colors_precomp if colors_precomp.numel() else None, grad_opacities,
                grad_scales if scales.numel() else None, grad_rotations if rotations.numel() else None,
                grad_cov3Ds_precomp if cov3Ds_precomp.numel() else None, None, None)


def _forward_arguments(means3D, sh, colors_precomp, opacities, scales, rotations, cov3Ds_precomp, rs):
    """The arguments of the reference's C++ forward in its order (K/rasterize_points.cu:35-58)."""
    return (rs.bg, means3D, colors_precomp, opacities, scales, rotations, rs.scale_modifier, cov3Ds_precomp, rs.viewmatrix,
            rs.projmatrix, rs.projmatrix_inv, rs.range_low, rs.range_up, rs.tanfovx, rs.tanfovy, rs.image_height, rs.image_width,
            sh, rs.sh_degree, rs.campos, rs.prefiltered, rs.debug)


def rasterize_frame(rasterizers, inputs, streams=None, workspaces=None):
    """All layers of a frame through one call.  `rasterizers`: K GaussianRasterizer (their settings share the
    camera and the image size); `inputs`: K dicts with the keyword arguments of GaussianRasterizer.forward
    (means3D, means2D, opacities, shs / colors_precomp, scales + rotations / cov3D_precomp); `streams`: None,
    or for every layer the handle of a HIP stream; the first that is not the current stream takes memory-bound work
    beside the kernels of the current one: the backward runs the per-Gaussian part of the layers whose blend is done
    on it (the caller's stream waits for it); every forward stage runs on the current stream.  `workspaces`: None, or a
    list that receives per layer (num_rendered, geomBuffer, binningBuffer, imgBuffer), the rest of the 8-tuple a single
    forward call returns (K/rasterize_points.cu:124).  Returns K tuples (color, radii, depth, alpha), the results of K
    forward calls, and differentiates like them."""
    return _rasterize_layers([rz.raster_settings for rz in rasterizers], inputs, streams, workspaces)


def _rasterize_layers(settings, inputs, streams=None, workspaces=None, strips=None):
    """rasterize_frame from the layers' settings.  `strips`: a list that receives what the compositor can use of each layer
    (see _host.composite).  A layer's "sh_parts", of all layers or of none: the further parts of SH rows of which "shs" holds
    the first coefficients (see _host.rasterize_frame)."""
    flat = []
    split = None if not any("sh_parts" in kw for kw in inputs) else [kw["sh_parts"] for kw in inputs]
    for kw in inputs:
        shs, colors_precomp, scales, rotations, cov3D = _checked_inputs(kw.get("shs"), kw.get("colors_precomp"), kw.get("scales"),
                                                                        kw.get("rotations"), kw.get("cov3D_precomp"))
        flat += (kw["means3D"], kw["means2D"], shs, colors_precomp, kw["opacities"], scales, rotations, cov3D)
    return _host.rasterize_frame(settings, flat, streams, workspaces, strips, split)


def _checked_inputs(shs, colors_precomp, scales, rotations, cov3D_precomp):
    """The five inputs of which a call takes some, empty tensors for those that are absent."""
    if (shs is None and colors_precomp is None) or (shs is not None and colors_precomp is not None):
        raise Exception('Please provide excatly one of either SHs or precomputed colors!')

    if ((scales is None or rotations is None) and cov3D_precomp is None) or \
            ((scales is not None or rotations is not None) and cov3D_precomp is not None):
        raise Exception('Please provide exactly one of either scale/rotation pair or precomputed 3D covariance!')
    return (_EMPTY if shs is None else shs, _EMPTY if colors_precomp is None else colors_precomp,
            _EMPTY if scales is None else scales, _EMPTY if rotations is None else rotations,
            _EMPTY if cov3D_precomp is None else cov3D_precomp)


class GaussianRasterizer(nn.Module):
    """K/diff_gaussian_rasterization_half_gaussian/__init__.py:183-232."""

    def __init__(self, raster_settings):
        super().__init__()
        self.raster_settings = raster_settings

    def markVisible(self, positions):
        # Mark visible points (based on frustum culling for camera) with a boolean
        with torch.no_grad():
            raster_settings = self.raster_settings
            visible = _mark_visible(positions, raster_settings.viewmatrix, raster_settings.projmatrix)
        return visible

    def forward(self, means3D, means2D, opacities, shs=None, colors_precomp=None, scales=None, rotations=None,
                cov3D_precomp=None, geometry=None):
        """As the reference's forward.  `geometry`, if given, is what enqueue_geometry returned for
        these same inputs: the call then only waits for that stage and goes on from there."""
        shs, colors_precomp, scales, rotations, cov3D_precomp = _checked_inputs(shs, colors_precomp, scales, rotations,
                                                                                cov3D_precomp)
        return rasterize_gaussians(means3D, means2D, shs, colors_precomp, opacities, scales, rotations, cov3D_precomp,
                                   self.raster_settings, geometry)

    def enqueue_geometry(self, means3D, opacities, shs=None, colors_precomp=None, scales=None, rotations=None,
                         cov3D_precomp=None, instance_bound=None) -> GeometryStage:
        """Starts the first half of a forward call (preprocess and instance count) on the current
        stream and returns without waiting for it.  No counterpart in the reference, whose forward
        always blocks on the count (K/cuda_rasterizer_hgs/rasterizer_impl.cu:287): a caller that
        renders several submodels on separate streams enqueues every geometry stage first and
        then calls forward(..., geometry=stage) for each, on the stream the stage was enqueued
        on, so that the host's wait for one count no longer holds back the other submodels.

        instance_bound: room for that many (Gaussian, tile) instances is set aside and the forward
        does not wait for the count at all (the reference grows its buffers on demand instead,
        K/rasterize_points.cu:27-33).  The caller must then ask stage.within_bound() after the
        forward has been issued (at the end of the iteration is early enough) and, if it is
        false, repeat the forward with a bound of at least stage.instances()."""
        shs, colors_precomp, scales, rotations, cov3D_precomp = _checked_inputs(shs, colors_precomp, scales, rotations,
                                                                                cov3D_precomp)
        if instance_bound is not None:
            instance_bound = int(instance_bound)
            if instance_bound < 0:
                raise ValueError("instance_bound must not be negative")
        return _host.enqueue_geometry(means3D, shs, colors_precomp, opacities, scales, rotations, cov3D_precomp,
                                      self.raster_settings, instance_bound)
