"""Front-to-back compositing of per-submodel partial images, forward and backward, as
one fused HIP pass each.  Host-side mirror of blender_render_result
(parallel_utils/basic_parallel_trainer/result_aggregator.py:193-260): the same ordering
rule (ascending value of the relation vector, negative = not related), the same three
outputs (render, depth, alpha) and the same gradients torch autograd produces for the
reference's cat / cumprod / sum expression.  The autograd function is Composite of
csrc/host.cpp.
"""
from __future__ import annotations

from typing import Dict, Optional, Sequence

import torch

from . import _capi, _host


def composite_partial_images(images: Sequence[torch.Tensor], depths: Sequence[torch.Tensor],
                             alphas: Sequence[torch.Tensor], background: Optional[torch.Tensor] = None):
    """Composite K partial images that are already in front-to-back order.
    images[k]: (3,H,W); depths[k], alphas[k]: (1,H,W).  Returns (image, depth, alpha).
    More than MAX_COMPOSITE inputs are folded in groups: compositing is associative in
    (image, depth, alpha) when the inner groups use a black background."""
    return _composite(images, depths, alphas, background, None)


def _composite(images, depths, alphas, background, strips):
    """composite_partial_images; strips[k], if the list is given: what the rasterizer says of layer k beside its planes."""
    K = len(images)
    if K == 0 or len(depths) != K or len(alphas) != K:
        raise RuntimeError("composite_partial_images needs K >= 1 images, depths and alphas")
    images, depths, alphas = list(images), list(depths), list(alphas)
    if K > _capi.MAX_COMPOSITE:
        strips = None
    while len(images) > _capi.MAX_COMPOSITE:
        n = _capi.MAX_COMPOSITE
        img, dep, alp = _host.composite(None, images[:n] + depths[:n] + alphas[:n])
        images, depths, alphas = [img] + images[n:], [dep] + depths[n:], [alp] + alphas[n:]
    return _host.composite(background, images + depths + alphas, strips)


def blender_render_result(render_results: Dict[int, dict], relation_vector, background: Optional[torch.Tensor],
                          strips: Optional[Dict[int, tuple]] = None):
    """Same contract as the reference function of this name
    (parallel_utils/basic_parallel_trainer/result_aggregator.py:193-260) for one camera on
    one GPU: `render_results` maps submodel id -> {"render","depth","alpha"} (what
    render4renderinfo returns), `relation_vector[model_id]` is the compositing rank of that
    submodel or a negative value when it is not related to the camera.  Returns a dict with
    "render", "depth", "alpha".  A missing background draws a random colour, like the
    reference (:256).
    strips: for results that come straight from rasterize_frame, what it handed out under that name by submodel id; planes
    are then not read where their submodel shows nothing."""
    if isinstance(relation_vector, torch.Tensor):
        relation_vector = relation_vector.cpu().numpy()
    related = [(int(relation_vector[m]), m) for m in render_results if relation_vector[m] >= 0]
    num_related = int(sum(1 for v in relation_vector if v >= 0))
    if len(related) != num_related:
        raise RuntimeError("NUM_RELATED mis-match")
    related.sort(key=lambda x: x[0])
    pk = [render_results[m] for _, m in related]
    device = pk[0]["render"].device
    bkg = background if background is not None else torch.rand((3,), device=device)
    image, depth, alpha = _composite([p["render"] for p in pk], [p["depth"] for p in pk], [p["alpha"] for p in pk], bkg,
                                     None if strips is None else [strips[m] for _, m in related])
    return {"render": image, "depth": depth, "alpha": alpha}


def partial_image_package(render: torch.Tensor, depth: torch.Tensor, alpha: torch.Tensor) -> torch.Tensor:
    """The (5,H,W) tensor in which the reference ships a partial image or its gradient between ranks
    (RenderResult.zip_content / zip_grad, parallel_utils/basic_parallel_trainer/task_utils.py:156-163,
    187-195): colour, depth, alpha stacked.  The rasterizer and the compositor's backward of this
    package already write the three into one such block, so this returns that block itself when it is
    given them (no copy), and concatenates otherwise."""
    base = render._base
    if (base is not None and depth._base is base and alpha._base is base and tuple(base.shape) == (5,) + tuple(render.shape[1:])
            and base.is_contiguous() and render.data_ptr() == base.data_ptr()
            and depth.data_ptr() == base[3:4].data_ptr() and alpha.data_ptr() == base[4:5].data_ptr()):
        return base.detach()
    with torch.no_grad():
        return torch.cat([render, depth, alpha], dim=0).to(dtype=torch.float32)


def unpack_partial_image(package: torch.Tensor):
    """Views of a (5,H,W) package: colour (3,H,W), depth (1,H,W), alpha (1,H,W)
    (RenderResult.unzip_content / unzip_grad, task_utils.py:176-185, 206-214, without the copies)."""
    if package.dim() != 3 or package.shape[0] != 5:
        raise RuntimeError("a partial-image package has shape (5, H, W)")
    return package[0:3], package[3:4], package[4:5]
