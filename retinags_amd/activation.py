"""From a submodel's stored parameters to the tensors its renderer and neighbours see, in one kernel
each way (rgs_activate_forward / rgs_activate_backward, include/rgs.h): what the get_* properties of
the reference's Gaussian model compute with one tensor operation each
(scene/gaussian_nn_module.py:373-394).  The autograd function is Activate of csrc/host_training.cpp."""
from __future__ import annotations

from typing import Optional

import torch

from . import _host
from .sharing import SharedGSInfo


def activate_gaussians(xyz: torch.Tensor, features_dc: torch.Tensor, features_rest: torch.Tensor, scaling: torch.Tensor,
                       rotation: torch.Tensor, opacity: torch.Tensor, means2D: Optional[torch.Tensor] = None,
                       spare_rows: int = 0) -> SharedGSInfo:
    """The SharedGSInfo that gather_local_SharedGSInfo builds from a model's properties
    (parallel_utils/basic_parallel_trainer/result_aggregator.py:40-52).  means3D is xyz itself, as
    in the reference; means2D is the caller's screen-space placeholder (zeros if absent).
    spare_rows: room behind every activated tensor, which sharing.merge_shared(append=True) needs
    (xyz and means2D must then bring their own)."""
    shs, scales, rotations, opacities = _host.activate(features_dc, features_rest, scaling, rotation, opacity, int(spare_rows))
    if means2D is None:
        meta = torch.empty((int(xyz.shape[0]), 1), dtype=torch.float32, device=xyz.device)
        means2D = _host.screen_placeholder(meta, int(spare_rows)).requires_grad_(xyz.requires_grad)
    return SharedGSInfo(xyz, means2D, opacities, scales, rotations, shs)
