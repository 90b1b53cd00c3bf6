"""Image loss of a training iteration on the GPU: (1 - lambda) L1 + lambda (1 - SSIM) with its
gradient in two kernels (rgs_l1_ssim_forward / rgs_l1_ssim_backward, include/rgs.h), under the
names of the reference's utils/loss_utils.py.  The autograd function is L1SSIM of csrc/host_training.cpp."""
from __future__ import annotations

from typing import Tuple

import torch

from . import _host


def l1_ssim_loss(image: torch.Tensor, gt: torch.Tensor, lambda_dssim: float = 0.2) -> Tuple[torch.Tensor, torch.Tensor]:
    """(loss, Ll1) of loss_local (parallel_utils/basic_parallel_trainer/trainer4tree_partition.py:
    449-450): loss = (1 - lambda_dssim) * l1_loss + lambda_dssim * (1 - ssim); differentiable in
    `image`.  Ll1 is returned for logging, detached."""
    loss, parts = _host.l1_ssim(image, gt, float(lambda_dssim))
    return loss, parts[1]


def l1_loss(network_output: torch.Tensor, gt: torch.Tensor) -> torch.Tensor:
    """utils/loss_utils.py:17-18 (value only; train through l1_ssim_loss)."""
    with torch.no_grad():
        return _host.l1_ssim(network_output, gt, 0.0)[1][1]


def ssim(img1: torch.Tensor, img2: torch.Tensor) -> torch.Tensor:
    """utils/loss_utils.py:39-63 with its defaults (window 11, mean over everything); value only."""
    with torch.no_grad():
        return _host.l1_ssim(img1, img2, 1.0)[1][2]
