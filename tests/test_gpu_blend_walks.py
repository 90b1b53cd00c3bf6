"""How the blends deal out strips and walk them, against the checker: images with more strips than a launch has workgroups,
and entries with and without the comparisons that only some need."""
import numpy as np
import pytest
import torch

from helpers import scenes
from test_gpu_rasterizer_parity import _check_backward, _check_forward_stages, _scene_sub

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,height,n,grow", [
    (1808, 1168, 700, 60.0),   # 32 996 strips, nearly all with entries: most workgroups have a second one
    (1808, 1168, 300, 0.5),    # the same, few with entries: the empty ones are dealt out
    (1805, 1149, 300, 60.0),   # 32 544: a workgroup per strip
])
def test_more_strips_than_workgroups(width, height, n, grow):
    scene = scenes.cube_scene(n, seed=33)
    scene["scales"] = scene["scales"] * grow
    cam = scenes.look_at_camera((0.0, 0.0, 0.0), (0.1, -0.05, 4.0), (0.05, -1, 0), width, height, 40.0)
    sub = _scene_sub(scene)
    st = _check_forward_stages(sub, cam, torch.tensor([0.2, 0.1, 0.05]), max_borderline=2e-3)
    assert (np.mean(st.n_contrib > 0) > 0.6) == (grow > 10)
    _check_backward(sub, cam, torch.tensor([0.2, 0.1, 0.05]), seed=3, with_depth_alpha=False)


@pytest.mark.parametrize("width,height", [(1024, 1024), (1040, 1024), (1008, 1025)])   # 16 384, 16 640, 16 380 strips: ordered in one kernel or two
def test_strips_ordered_at_once(width, height):
    scene = scenes.cube_scene(1500, seed=12)
    scene["scales"] = scene["scales"] * 8.0
    cam = scenes.look_at_camera((0.0, 0.0, 0.0), (0.1, -0.05, 4.0), (0.05, -1, 0), width, height, 45.0)
    sub = _scene_sub(scene)
    _check_forward_stages(sub, cam, torch.tensor([0.2, 0.1, 0.05]), max_borderline=2e-3)
    _check_backward(sub, cam, torch.tensor([0.2, 0.1, 0.05]), seed=5, with_depth_alpha=False)


# (up to 4 096 strips, as in most tests of small images, a forward walk is shared by four wavefronts)
@pytest.mark.parametrize("low,up", [((-0.31, -0.27, 3.6), (0.23, 0.19, 4.3)), ((-5.0, 0.05, -1.0), (5.0, 5.0, 9.0)),
                                    ((-5.0, -5.0, 4.95), (5.0, 5.0, 9.0))])
@pytest.mark.parametrize("width,height", [(515, 497), (511, 505)])   # 4 224 and 4 096 strips
def test_box_faces_with_and_without_shared_walks(low, up, width, height):
    scene = scenes.cube_scene(2500, seed=92)
    scene["scales"] = scene["scales"] * 5.0
    cam = scenes.look_at_camera((0.0, 0.0, 0.0), (0.13, -0.07, 4.0), (0.1, -1, 0), width, height, 40.0)
    sub = _scene_sub(scene, low=torch.tensor(low), up=torch.tensor(up))
    _check_forward_stages(sub, cam, torch.tensor([0.2, 0.1, 0.05]), max_borderline=2e-3)
    _check_backward(sub, cam, torch.tensor([0.2, 0.1, 0.05]), seed=17, with_depth_alpha=width == 511)


def test_shared_and_whole_walks_give_the_same_bits():
    """The same view as one job of a launch (4 096 strips: shared walks) and as two (whole ones): transmittances are the
    same products in the same order and the sums add in the same order, so images and last blended entries are equal.
    Some colours are infinite: they reach the pixels that blend them and no others."""
    from retinags_amd import GaussianRasterizationSettings, GaussianRasterizer, rasterizer
    dev = "cuda:0"
    scene = scenes.cube_scene(20_000, seed=93)
    cam = scenes.look_at_camera((0.0, 0.0, 0.0), (0.13, -0.07, 4.0), (0.1, -1, 0), 509, 501, 40.0).to(dev)
    inf = float("inf")
    rasterizers, inputs = [], []
    for low, up in (((-0.4, -9.0, -9.0), (9.0, 9.0, 9.0)), ((-inf,) * 3, (inf,) * 3)):
        rasterizers.append(GaussianRasterizer(GaussianRasterizationSettings(
            image_height=501, image_width=509, tanfovx=cam.tanfovx, tanfovy=cam.tanfovy, bg=torch.zeros(3, device=dev), scale_modifier=1.0,
            viewmatrix=cam.world_view_transform, projmatrix=cam.full_proj_transform, projmatrix_inv=cam.projection_matrix_inv,
            range_low=torch.tensor(low, device=dev), range_up=torch.tensor(up, device=dev), sh_degree=0, campos=cam.camera_center,
            prefiltered=False, debug=False)))
        colours = torch.rand(20_000, 3, generator=torch.Generator().manual_seed(1))
        colours[::200, 1] = inf
        inputs.append(dict(means3D=scene["xyz"].to(dev), means2D=torch.zeros(20_000, 3, device=dev), colors_precomp=colours.to(dev),
                           opacities=scene["opacity"].to(dev), scales=scene["scales"].to(dev) * 2, rotations=scene["rotations"].to(dev)))
    with torch.no_grad():
        together = rasterizer.rasterize_frame(rasterizers, inputs)
        for k, (r, given) in enumerate(zip(rasterizers, inputs)):
            for name, one, both in zip(("colour", "radii", "depth", "alpha"), r(**given), together[k]):
                assert torch.equal(one, both), name
            infinite = torch.isinf(together[k][0][1])
            assert not torch.isnan(together[k][0]).any() and infinite.any() and infinite.float().mean() < 0.9
            assert torch.isfinite(together[k][0][0]).all() and torch.isfinite(together[k][0][2]).all()


@pytest.mark.parametrize("case", ("opaque", "needles", "some of each", "opacity is NaN"))
def test_entries_that_need_every_comparison_of_a_visit(case):
    """Alphas that the 0.99 bound cuts, conics whose exponent may round to above zero at the centre, and both among entries
    that need neither comparison."""
    gen = torch.Generator().manual_seed(5)
    scene = scenes.cube_scene(1500, seed=44)
    scene["scales"] = scene["scales"] * 6.0
    n = scene["xyz"].shape[0]
    some = torch.rand(n, generator=gen) < (0.02 if case == "some of each" else 1.0)
    if case in ("opaque", "some of each"):
        scene["opacity"][some] = 0.98 + 0.02 * torch.rand(int(some.sum()), 1, generator=gen)
    if case in ("needles", "some of each"):
        # (two scales of nothing: the projected covariance is one direction and the low-pass filter's 0.3)
        scene["scales"][some] = torch.tensor([2.0, 1e-5, 1e-5])
    if case == "opacity is NaN":
        scene["opacity"][::97] = float("nan")
    cam = scenes.look_at_camera((0.0, 0.0, 0.0), (0.13, -0.07, 4.0), (0.1, -1, 0), 147, 83, 40.0)
    sub = _scene_sub(scene, low=torch.full((3,), -99.0), up=torch.full((3,), 99.0))
    _check_forward_stages(sub, cam, torch.tensor([0.2, 0.1, 0.05]), max_borderline=5e-3)
    if case == "opaque":   # (a needle's gradients are differences of terms a million times as large, in the checker as here)
        _check_backward(sub, cam, torch.tensor([0.2, 0.1, 0.05]), seed=7, with_depth_alpha=True)


@pytest.mark.parametrize("faces", (False, True))
@pytest.mark.parametrize("n,with_depth_alpha", [(64, False), (65, True), (73, False), (200, True), (257, False), (521, True), (1203, False)])
def test_backward_walks_shared_by_four_wavefronts(n, with_depth_alpha, faces):
    """Strips that blend all of n entries: walks of one chunk by one wavefront, and by four with every number of chunks against the
    buffers they are staged in, the last pass of a chunk full, partly filled or missing for some of the wavefronts."""
    gen = torch.Generator().manual_seed(n)
    scene = scenes.cube_scene(n, seed=71)
    scene["xyz"] = torch.randn(n, 3, generator=gen) * torch.tensor([0.05, 0.05, 0.3]) + torch.tensor([0.0, 0.0, 4.0])
    scene["scales"] = torch.full((n, 3), 0.3) * (0.5 + torch.rand(n, 3, generator=gen))
    scene["opacity"] = 3.0 / n + 2.0 / n * torch.rand(n, 1, generator=gen) + 0.004
    cam = scenes.look_at_camera((0.0, 0.0, 0.0), (0.03, -0.02, 4.0), (0.1, -1, 0), 43, 22, 12.0)
    low, up = ((-0.2, -9.0, -9.0), (9.0, 0.15, 4.3)) if faces else ((-99.0,) * 3, (99.0,) * 3)
    sub = _scene_sub(scene, low=torch.tensor(low), up=torch.tensor(up))
    st = _check_forward_stages(sub, cam, torch.tensor([0.2, 0.1, 0.05]), max_borderline=5e-2)
    assert faces or np.mean(st.n_contrib > 0.9 * n) > 0.5
    _check_backward(sub, cam, torch.tensor([0.2, 0.1, 0.05]), seed=n, with_depth_alpha=with_depth_alpha)


def _slab_along_a_face(n):
    """Opaque Gaussians about a face of the box that the camera sees at 45 degrees: neighbouring pixels enter the box at depths with many
    chunks of entries between them, and what lies behind the box's other faces is blended by no pixel."""
    gen = torch.Generator().manual_seed(n)
    scene = scenes.cube_scene(n, seed=n)
    z = 2.0 + 0.3 * torch.rand(n, generator=gen) - 0.15
    z[::5] = 2.0 + 3.0 * torch.rand(z[::5].shape, generator=gen)
    side = z * (0.8 + 0.4 * torch.rand(n, generator=gen))
    scene["xyz"] = torch.stack([side, (torch.rand(n, generator=gen) - 0.5) * 0.4 * (side + z), z], 1)
    scene["scales"] = torch.full((n, 3), 0.012)
    scene["opacity"] = torch.full((n, 1), 0.97)
    return scene, (-9.0, -9.0, 2.0), (9.0, 0.4, 2.6)


def test_chunks_that_no_pixel_can_blend_are_passed_over():
    """Whole walks, which pass over chunks that the box clips for every unfinished pixel, against walks shared by four wavefronts, which
    stage every chunk (the same view as two jobs of a launch and as one): equal images and last blended entries."""
    from retinags_amd import GaussianRasterizationSettings, GaussianRasterizer, _capi, rasterizer
    dev, n = "cuda:0", 250_000
    scene, low, up = _slab_along_a_face(n)
    cam = scenes.look_at_camera((0.0, 0.0, 0.0), (1.0, 0.0, 1.0), (0.0, -1, 0), 509, 501, 40.0).to(dev)
    r = GaussianRasterizer(GaussianRasterizationSettings(
        image_height=501, image_width=509, tanfovx=cam.tanfovx, tanfovy=cam.tanfovy, bg=torch.zeros(3, device=dev), scale_modifier=1.0,
        viewmatrix=cam.world_view_transform, projmatrix=cam.full_proj_transform, projmatrix_inv=cam.projection_matrix_inv,
        range_low=torch.tensor(low, device=dev), range_up=torch.tensor(up, device=dev), sh_degree=0, campos=cam.camera_center,
        prefiltered=False, debug=False))
    given = dict(means3D=scene["xyz"].to(dev), means2D=torch.zeros(n, 3, device=dev), opacities=scene["opacity"].to(dev),
                 colors_precomp=torch.rand(n, 3, generator=torch.Generator().manual_seed(1)).to(dev), scales=scene["scales"].to(dev),
                 rotations=scene["rotations"].to(dev))
    im = _capi.image_layout(509, 501)
    read = lambda img, key, count: img[im[key]:im[key] + 4 * count].view(torch.int32)
    alone, both = [], []
    with torch.no_grad():
        one = rasterizer.rasterize_frame([r], [given], workspaces=alone)[0]
        two = rasterizer.rasterize_frame([r, r], [given, given], workspaces=both)
    totals, walked = (read(alone[0][3], key, 4096).long() for key in ("strip_total", "strip_filed"))
    # some lists go on for more chunks than are looked at together behind the last entry that is blended
    assert int((totals - walked).max()) > 64 * 16 and int(walked.max()) > 64 * 5
    for k in range(2):
        for name, a, b in zip(("colour", "radii", "depth", "alpha"), one, two[k]):
            assert torch.equal(a, b), name
        for key, count in (("strip_filed", 4096), ("n_contrib", 509 * 501)):
            assert torch.equal(read(alone[0][3], key, count), read(both[k][3], key, count)), key


def test_chunks_passed_over_against_the_checker():
    scene, low, up = _slab_along_a_face(60_000)
    cam = scenes.look_at_camera((0.0, 0.0, 0.0), (1.0, 0.0, 1.0), (0.0, -1, 0), 515, 497, 40.0)
    _check_forward_stages(_scene_sub(scene, low=torch.tensor(low), up=torch.tensor(up)), cam, torch.tensor([0.2, 0.1, 0.05]), max_borderline=2e-3)
