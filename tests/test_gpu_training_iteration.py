"""A whole training iteration on the GPU (share boundary Gaussians, render the submodels, composite,
L1 + SSIM loss, backward to every submodel's own Gaussians, Adam) against the chain of CPU checkers
for its gradients, and over a few iterations for what it is for: the loss goes down."""
import numpy as np
import pytest
import torch

from helpers import GRAD_TOL, IMAGE_TOL, np32, oracle_settings, orc, rel_l2, scenes
from oracle import sharing_oracle as so
from oracle import training_oracle as to

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
NAMES = ("means3D", "means2D", "opacity", "scales", "rotations", "shs")


def _setup(spare=0.0):
    from retinags_amd.harness import partition, pipeline
    scene, cam, _ = scenes.make_config("C1", shrink=150, resolution_scale=0.25)
    scene["scales"] = scene["scales"] * 2.0      # more boundary straddlers at this size
    part = partition.partition_scene(scene["xyz"], scene["scales"], 2)
    rel = partition.relation_vector(part, cam)
    models = pipeline.owned_models_from_partition(scene, part, DEV, spare)
    return scene, cam, part, rel, models


def test_gradients_of_one_iteration_against_the_checker_chain():
    from retinags_amd import sharing
    from retinags_amd.harness import pipeline
    from retinags_amd.loss import l1_ssim_loss
    scene, cam, part, rel, models = _setup()
    K = len(models)
    H, W = cam.image_height, cam.image_width
    gen = torch.Generator().manual_seed(9)
    gt = torch.rand(3, H, W, generator=gen)
    bg = torch.tensor([0.1, 0.1, 0.1])
    for m in models:
        for t in m.fields():
            t.requires_grad_(True)
    table = sharing.select_straddlers(models, part.box_low, part.box_up)
    assert table.counts.sum() > 20
    merged = sharing.merge_shared(models, table, reuse_gradients=True)
    frame = pipeline.render_frame(cam.to(DEV), pipeline.submodels_from_shared(merged, part, DEV), rel, bg.to(DEV))
    loss, l1 = l1_ssim_loss(frame["render"], gt.to(DEV), 0.2)
    loss.backward()
    torch.cuda.synchronize()

    # the same on the CPU: checker of every stage, chained
    host = [{n: np32(getattr(m, n)) for n in NAMES} for m in models]
    lent = {(s, d): so.straddler_rows(host[s]["means3D"], host[s]["scales"], part.box_low[s], part.box_up[s],
                                      part.box_low[d], part.box_up[d]) for s in range(K) for d in range(K) if s != d}
    order = sorted((m for m in range(K) if rel[m] >= 0), key=lambda m: rel[m])
    blocks = {d: so.merged_rows([len(h["means3D"]) for h in host], lent, d) for d in order}
    inputs = {d: so.merge_fields(host, blocks[d]) for d in order}
    states, sets = {}, {}
    for d in order:
        sets[d] = oracle_settings(cam, torch.from_numpy(part.box_low[d]), torch.from_numpy(part.box_up[d]), torch.zeros(3))
        states[d] = orc.forward(sets[d], inputs[d]["means3D"], inputs[d]["opacity"], shs=inputs[d]["shs"],
                                scales=inputs[d]["scales"], rotations=inputs[d]["rotations"])
    imgs, deps, alps = ([states[d].color for d in order], [states[d].depth for d in order], [states[d].alpha for d in order])
    image, _, _ = orc.composite_forward(imgs, deps, alps, np32(bg))
    want_loss, want_l1, _, d_image = to.l1_ssim(image, gt.numpy(), 0.2)
    assert abs(float(loss.detach()) - want_loss) < 1e-5 and abs(float(l1) - want_l1) < 1e-5
    assert np.abs(frame["render"].detach().cpu().numpy() - image).mean() < IMAGE_TOL
    d_img, d_dep, d_alp = orc.composite_backward(imgs, deps, alps, np32(bg), d_image.astype(np.float32))
    shapes = [{n: v.shape for n, v in h.items()} for h in host]
    want = [{n: np.zeros(s, np.float32) for n, s in sh.items()} for sh in shapes]
    for k, d in enumerate(order):
        g = orc.backward(sets[d], states[d], d_img[k], d_dep[k], d_alp[k])
        grads = {"means3D": g["means3D"], "means2D": g["means2D"], "opacity": g["opacity"], "scales": g["scales"],
                 "rotations": g["rotations"], "shs": g["sh"]}
        back = so.merge_backward(grads, blocks[d], shapes)
        for s in range(K):
            for n in NAMES:
                want[s][n] += back[s][n]
    for s in range(K):
        for n in NAMES:
            got = getattr(models[s], n).grad.cpu().numpy()
            assert rel_l2(got, want[s][n]) <= GRAD_TOL, (s, n)


@pytest.mark.parametrize("append", [False, True])
def test_the_loss_goes_down(append):
    from retinags_amd.harness import pipeline
    scene, cam, part, rel, models = _setup(spare=0.3 if append else 0.0)
    cam_d = cam.to(DEV)
    bg = torch.zeros(3, device=DEV)
    with torch.no_grad():
        target = pipeline.render_frame(cam_d, pipeline.submodels_from_partition(scene, part, DEV), rel, bg)["render"].clone()
        gen = torch.Generator().manual_seed(3)
        for m in models:                                   # start from disturbed colours and opacities
            m.shs.add_((torch.randn(m.shs.shape, generator=gen) * 0.1).to(DEV))
            m.opacity.mul_(0.8)
    for m in models:
        for t in m.fields():
            t.requires_grad_(True)
    optimisers = pipeline.make_optimisers(models)
    streams = [torch.cuda.current_stream(DEV)] + [torch.cuda.Stream(device=DEV) for _ in range(3)]
    losses = []
    for _ in range(12):
        step = pipeline.training_iteration(models, optimisers, part, cam_d, rel, target, bg, streams=streams, append=append)
        losses.append(float(step["loss"]))
        assert step["lent_rows"] > 0
    assert all(np.isfinite(losses)) and losses[-1] < 0.8 * losses[0], losses
    assert all(opt.state[p]["step"] == 12 for opt in optimisers for g in opt.param_groups for p in g["params"])


@pytest.mark.parametrize("spare", [0.0, 0.3])
def test_the_loss_goes_down_from_stored_parameters(spare):
    """The same loop from the parameters as the reference stores them (log scales, opacity logits, split SH
    coefficients) through the activation kernels; the screen-space gradient reaches the (N,1) placeholder."""
    from retinags_amd.harness import partition, pipeline
    scene, cam, _ = scenes.make_config("C1", shrink=150, resolution_scale=0.25)
    scene["scales"] = scene["scales"] * 2.0
    part = partition.partition_scene(scene["xyz"], scene["scales"], 2)
    rel = partition.relation_vector(part, cam)
    cam_d = cam.to(DEV)
    bg = torch.zeros(3, device=DEV)
    with torch.no_grad():
        target = pipeline.render_frame(cam_d, pipeline.submodels_from_partition(scene, part, DEV), rel, bg)["render"].clone()
    models = pipeline.stored_models_from_partition(scene, part, DEV, spare)
    # stored form and activation are inverse to each other: the untouched models render the target
    with torch.no_grad():
        shown = [m.activated() for m in models]
        from retinags_amd import sharing
        table = sharing.select_straddlers(shown, part.box_low, part.box_up)
        merged = sharing.merge_shared(shown, table, append=spare > 0)
        again = pipeline.render_frame(cam_d, pipeline.submodels_from_shared(merged, part, DEV), rel, bg)["render"]
        assert float((again - target).abs().max()) < 2e-3
        gen = torch.Generator().manual_seed(3)
        for m in models:
            m.features_dc.add_((torch.randn(m.features_dc.shape, generator=gen) * 0.1).to(DEV))
            m.opacity.sub_(0.5)
    for m in models:
        for t in m.parameters():
            t.requires_grad_(True)
    optimisers = pipeline.make_stored_optimisers(models)
    streams = [torch.cuda.current_stream(DEV)] + [torch.cuda.Stream(device=DEV) for _ in range(3)]
    losses, seen_meta_grad = [], False
    for it in range(12):
        if it == 11:      # look at the gradients of the last iteration before the step clears them
            for opt in optimisers:
                opt.zero_grad = lambda set_to_none=True: None
        step = pipeline.stored_training_iteration(models, optimisers, part, cam_d, rel, target, bg, streams=streams)
        losses.append(float(step["loss"]))
    assert all(np.isfinite(losses)) and losses[-1] < 0.8 * losses[0], losses
    for m in models:
        g = m.means2D_meta.grad
        assert g is not None and g.shape == m.means2D_meta.shape and float(g.min()) >= 0.0
        seen_meta_grad = seen_meta_grad or float(g.max()) > 0.0
        assert all(p.grad is not None and torch.isfinite(p.grad).all() for p in m.parameters())
    assert seen_meta_grad


class _Still:
    def step(self):
        pass

    def zero_grad(self, set_to_none=True):
        pass


@pytest.mark.parametrize("depth,spare,grow,unrelated", [(1, 0.0, 2.0, False), (1, 0.3, 2.0, False), (2, 0.0, 2.0, True), (2, 3.0, 100.0, False),
                                                        (1, 0.0, 100.0, False), (3, 4.0, 12.0, True)])
def test_models_shown_together_are_models_shown_one_by_one(depth, spare, grow, unrelated):
    """An iteration's gradients with activation, selection and lending of all models in one launch each and SH rows read as they are
    stored, against activated(), select_straddlers and merge_shared: from a few lent rows to lists longer than the room there is at
    first, with room behind the positions and without, models that the camera does not see, two to eight of them."""
    from retinags_amd.harness import partition, pipeline

    class OneByOne(pipeline.StoredModel):
        def activated(self):
            return super().activated()

    scene, cam, _ = scenes.make_config("C1", shrink=100 if grow > 20 else 150, resolution_scale=0.25)
    scene["scales"] = scene["scales"] * grow
    part = partition.partition_scene(scene["xyz"], scene["scales"], depth)
    rel = partition.relation_vector(part, cam)
    if unrelated:
        rel = np.where(rel == rel.max(), -1.0, rel)
    cam_d, bg = cam.to(DEV), torch.rand(3, device=DEV)
    gt = torch.rand(3, cam.image_height, cam.image_width, device=DEV)
    grads, lent, renders = [], [], []
    for kind in (pipeline.StoredModel, OneByOne):
        models = [kind(**vars(m)) for m in pipeline.stored_models_from_partition(scene, part, DEV, spare)]
        for m in models:
            for t in m.parameters():
                t.requires_grad_(True)
        step = pipeline.stored_training_iteration(models, [_Still() for _ in models], part, cam_d, rel, gt, bg)
        grads.append([[t.grad for t in m.parameters()] for m in models])
        lent.append(step["lent_rows"])
        renders.append(step["frame"]["render"].detach())
    own = [int(m.xyz.shape[0]) for m in models]
    if grow > 20:   # some list is longer than the room for it at first, some model borrows more than there is room for at first
        from retinags_amd.sharing import select_straddlers
        counts = select_straddlers([m.activated() for m in models], part.box_low, part.box_up).counts
        assert any(counts[k].max() > n // 8 + 4096 for k, n in enumerate(own)) and any(counts[:, k].sum() > n // 8 + 4096 for k, n in enumerate(own))
    assert lent[0] == lent[1] > 20 and torch.equal(renders[0], renders[1])
    for a, b in zip(*grads):
        for k, (got, want) in enumerate(zip(a, b)):
            assert got.shape == want.shape
            # (sums of float atomics: equal up to their order)
            assert torch.linalg.norm(got - want) <= 1e-4 * torch.linalg.norm(want), k
    assert any(float(torch.linalg.norm(g[1])) > 0 for g in grads[0])
