"""SH rows in parts (first coefficient, the other fifteen, whole rows of lent Gaussians) against the same rows joined."""
import pytest
import torch

from helpers import scenes

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _frame(sizes, degree, split, seed=1):
    from retinags_amd import GaussianRasterizationSettings, rasterizer
    cam = scenes.look_at_camera((0, 0, 0), (0, 0, 1), (0, -1, 0), 150, 90, 60.0).to(DEV)
    settings, inputs, leaves = [], [], []
    gen = torch.Generator().manual_seed(seed)
    for own, lent in sizes:
        n = own + lent
        scene = scenes.cube_scene(n, seed=n)
        scene["xyz"][::3, 2] *= -1.0   # behind the camera: their gradients are zeros
        rows = torch.randn(n, 16, 3, generator=gen) * 0.4
        leaf = dict(means3D=scene["xyz"], opacities=scene["opacity"], scales=scene["scales"] * 4, rotations=scene["rotations"],
                    shs=rows if not split else rows[:own, :1])
        if split:
            leaf.update(rest=rows[:own, 1:], lent=rows[own:])
        leaf = {k: v.contiguous().to(DEV).requires_grad_(True) for k, v in leaf.items()}
        leaf["means2D"] = torch.zeros(n, 3, device=DEV, requires_grad=True)
        leaves.append(leaf)
        kw = {k: leaf[k] for k in ("means3D", "means2D", "opacities", "scales", "rotations", "shs")}
        if split:
            kw["sh_parts"] = (leaf["rest"], leaf["lent"])
        inputs.append(kw)
        settings.append(GaussianRasterizationSettings(
            image_height=90, image_width=150, tanfovx=cam.tanfovx, tanfovy=cam.tanfovy, bg=torch.zeros(3, device=DEV), scale_modifier=1.0,
            viewmatrix=cam.world_view_transform, projmatrix=cam.full_proj_transform, projmatrix_inv=cam.projection_matrix_inv,
            range_low=torch.full((3,), -99.0, device=DEV), range_up=torch.full((3,), 99.0, device=DEV), sh_degree=degree,
            campos=cam.camera_center, prefiltered=False, debug=False))
    outs = rasterizer._rasterize_layers(settings, inputs)
    upstream = [torch.randn(3, 90, 150, generator=gen).to(DEV) * 1e-2 for _ in outs]
    torch.autograd.backward([o[0] for o in outs], upstream)
    return outs, leaves


@pytest.mark.parametrize("degree", (0, 1, 2, 3))
@pytest.mark.parametrize("sizes", [((1, 0),), ((63, 1), (64, 64)), ((65, 200), (700, 0), (128, 63)), ((500, 333),), ((192, 1), (127, 1))])
def test_rows_in_parts_are_the_joined_rows(sizes, degree):
    whole, w = _frame(sizes, degree, False)
    parts, p = _frame(sizes, degree, True)
    for a, b in zip(whole, parts):
        assert all(torch.equal(x, y) for x, y in zip(a, b))
    for (own, _), a, b in zip(sizes, w, p):
        joined = torch.cat((torch.cat((b["shs"].grad, b["rest"].grad), dim=1), b["lent"].grad))
        for name, want, got in [("shs", a["shs"].grad, joined)] + [(k, a[k].grad, b[k].grad) for k in ("means3D", "means2D", "opacities", "scales", "rotations")]:
            # (sums of float atomics: equal up to their order)
            assert torch.linalg.norm(got - want) <= 1e-5 * torch.linalg.norm(want), name
            assert torch.equal(got == 0, want == 0) or name != "shs"


def test_parts_that_do_not_fit_are_refused():
    from retinags_amd import rasterizer
    _, leaves = _frame(((40, 9),), 3, True)
    settings = None
    leaf = leaves[0]
    cam = scenes.look_at_camera((0, 0, 0), (0, 0, 1), (0, -1, 0), 150, 90, 60.0).to(DEV)
    from retinags_amd import GaussianRasterizationSettings
    settings = GaussianRasterizationSettings(
        image_height=90, image_width=150, tanfovx=cam.tanfovx, tanfovy=cam.tanfovy, bg=torch.zeros(3, device=DEV), scale_modifier=1.0,
        viewmatrix=cam.world_view_transform, projmatrix=cam.full_proj_transform, projmatrix_inv=cam.projection_matrix_inv,
        range_low=torch.full((3,), -99.0, device=DEV), range_up=torch.full((3,), 99.0, device=DEV), sh_degree=3,
        campos=cam.camera_center, prefiltered=False, debug=False)
    kw = {k: leaf[k].detach() for k in ("means3D", "means2D", "opacities", "scales", "rotations", "shs")}
    for rest, lent in ((leaf["rest"][:, :8], leaf["lent"]), (leaf["rest"], leaf["lent"][:-1]), (leaf["rest"][:-1], leaf["lent"])):
        with pytest.raises(RuntimeError, match="SH rows in parts"):
            rasterizer._rasterize_layers([settings], [dict(kw, sh_parts=(rest.detach(), lent.detach()))])
