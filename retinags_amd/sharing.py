"""Boundary straddlers: what every submodel lends to its neighbours, and a submodel's merged
input (its own Gaussians first, then the lent ones in ascending lender id).

Host side of rgs_straddler_select / rgs_merge_rows / rgs_merge_rows_backward (include/rgs.h).
It does what gather_SharedGSInfo_pool + merge_SharedGSInfo do in the reference
(parallel_utils/basic_parallel_trainer/result_aggregator.py:55-160, 263-288) for submodels that
live on one GPU, without materialising a (source, destination) tensor set per pair: the
selection yields row lists, the merge reads the sources through them once, and the backward
adds the gradients of lent rows straight onto the lender's gradients.  The steps are in
csrc/host_training.cpp (select_straddlers, MergeShared).
"""
from __future__ import annotations

from typing import Dict, List, Optional, Sequence, Tuple

import numpy as np
import torch

from . import _capi, _host

FIELDS = ("means3D", "means2D", "opacity", "scales", "rotations", "shs")


class SharedGSInfo:
    """The six tensors a submodel shows its renderer and its neighbours
    (parallel_utils/basic_parallel_trainer/task_utils.py:230-247): activated values, N rows each."""

    def __init__(self, means3D: torch.Tensor, means2D: torch.Tensor, opacity: torch.Tensor, scales: torch.Tensor,
                 rotations: torch.Tensor, shs: torch.Tensor) -> None:
        self.means3D = means3D
        self.means2D = means2D
        self.opacity = opacity
        self.scales = scales
        self.rotations = rotations
        self.shs = shs

    def fields(self) -> List[torch.Tensor]:
        return [getattr(self, n) for n in FIELDS]

    def __len__(self) -> int:
        return int(self.means3D.shape[0])


class StraddlerTable:
    """counts[src, dst] lent rows and, for each pair with any, their row numbers within the
    source (ascending, uint32 stored as int32 on the device)."""

    def __init__(self, counts: np.ndarray, rows: Dict[Tuple[int, int], torch.Tensor], own: List[int]) -> None:
        self.counts = counts
        self.rows = rows
        self.own = own

    def merged_size(self, dst: int) -> int:
        return self.own[dst] + int(self.counts[:, dst].sum())


def _require_device_rows(t: torch.Tensor, width, name: str) -> None:
    if not t.is_cuda:
        raise RuntimeError(f"{name} must be a device tensor: there is no host implementation")
    if t.dtype != torch.float32 or not t.is_contiguous():
        raise RuntimeError(f"{name} must be contiguous float32")
    if tuple(t.shape[1:]) != tuple(width):
        raise RuntimeError(f"{name} has shape {tuple(t.shape)}, expected (N, {', '.join(map(str, width))})")


def select_straddlers(models: Sequence[SharedGSInfo], box_low, box_up, capacity: Optional[int] = None) -> StraddlerTable:
    """models[m] is submodel m with box (box_low[m], box_up[m]) in world units, (K,3) each.
    One pass over every submodel's means and scales; one device-to-host copy for all counts."""
    K = len(models)
    if K > _capi.MAX_SHARE_BOXES:
        raise RuntimeError(f"{K} submodels: at most {_capi.MAX_SHARE_BOXES} per call")
    if capacity is not None and int(capacity) < 0:
        raise RuntimeError(f"a capacity of {capacity} rows: it must not be negative")
    low = np.ascontiguousarray(np.asarray(box_low, dtype=np.float32).reshape(K, 3))
    up = np.ascontiguousarray(np.asarray(box_up, dtype=np.float32).reshape(K, 3))
    own = [len(m) for m in models]
    for m in models:
        _require_device_rows(m.means3D, (3,), "means3D")
        _require_device_rows(m.scales, (3,), "scales")
    counts, rows = _host.select_straddlers([m.means3D for m in models], [m.scales for m in models],
                                           low.ravel().tolist() + up.ravel().tolist(), -1 if capacity is None else int(capacity))
    return StraddlerTable(np.array(counts, dtype=np.int64).reshape(K, K), rows, own)


def _lent_to(dst: int, table: StraddlerTable) -> List[Tuple[int, torch.Tensor, int]]:
    """(source, row list, count) of the rows lent to dst, in merge order."""
    return [(src, table.rows[(src, dst)], int(table.counts[src, dst])) for src in range(len(table.own))
            if src != dst and table.counts[src, dst] > 0]


def merge_shared(models: Sequence[SharedGSInfo], table: StraddlerTable, reuse_gradients: bool = False,
                 append: bool = False) -> List[SharedGSInfo]:
    """Every submodel's merged input (merge_SharedGSInfo, result_aggregator.py:263-288, for all
    destinations), differentiable with respect to every field of every submodel.

    append: instead of copying a submodel's own rows into new arrays, write the lent rows into
    the memory right behind them and return tensors over both.  Every field of every submodel
    must then sit in an allocation with that much room behind its rows (with_spare_rows makes
    such tensors); the merged tensors alias the submodel's own, and the room behind is
    overwritten by every merge.  Autograd does not know of that aliasing (the merged tensors are
    built over the inputs' storage, so the inputs' version counters do not guard them): the
    inputs must not be updated in place, and no other merge may run, between this call and the
    backward of everything that was rendered from its result.

    reuse_gradients: the backward returns the incoming gradient buffers of the merged arrays,
    with the borrowers' rows added in place, instead of copies.  Only for callers that do not
    read the merged arrays' gradients afterwards (no retain_grad on them)."""
    for m in models:
        for name, width in (("means3D", (3,)), ("means2D", (3,)), ("opacity", (1,)), ("scales", (3,)), ("rotations", (4,))):
            _require_device_rows(getattr(m, name), width, name)
        _require_device_rows(m.shs, tuple(models[0].shs.shape[1:]), "shs")
    flat = [t for m in models for t in m.fields()]
    outs = _host.merge_shared(table.own, [_lent_to(d, table) for d in range(len(models))], bool(reuse_gradients), bool(append), flat)
    return [SharedGSInfo(*outs[6 * m:6 * m + 6]) for m in range(len(models))]


def with_spare_rows(t: torch.Tensor, spare: int) -> torch.Tensor:
    """A copy of t (N rows) at the start of an allocation of N + spare rows, for merge_shared(append=True)."""
    room = torch.empty((t.shape[0] + spare,) + tuple(t.shape[1:]), dtype=t.dtype, device=t.device)
    room[:t.shape[0]].copy_(t)
    return room[:t.shape[0]]
