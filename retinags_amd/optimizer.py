"""Adam with the update of every tensor of a submodel in one kernel launch (rgs_adam_step,
include/rgs.h).  A torch.optim.Optimizer, so parameter groups, per-group learning rates, the
state dictionary ("step", "exp_avg", "exp_avg_sq" per parameter: what the reference's
densification edits, scene/gaussian_nn_module.py:588-635) and zero_grad work as with
torch.optim.Adam, which the reference uses with eps = 1e-15 (scene/gaussian_nn_module.py:443)."""
from __future__ import annotations

import torch

from . import _host


class Adam(torch.optim.Optimizer):
    def __init__(self, params, lr: float = 1e-3, betas=(0.9, 0.999), eps: float = 1e-8):
        if lr < 0 or eps < 0 or not 0 <= betas[0] < 1 or not 0 <= betas[1] < 1:
            raise ValueError("invalid Adam hyper-parameter")
        super().__init__(params, dict(lr=lr, betas=betas, eps=eps))

    @torch.no_grad()
    def step(self, closure=None):
        loss = None
        if closure is not None:
            with torch.enable_grad():
                loss = closure()
        _host.adam_step(self.param_groups, self.state)
        return loss

    def zero_grad(self, set_to_none: bool = True):
        if not set_to_none:
            return super().zero_grad(set_to_none=False)
        for group in self.param_groups:
            for p in group["params"]:
                p.grad = None
