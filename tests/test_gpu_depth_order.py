"""The depth order's small kernels at the sizes where they change their way."""
import numpy as np
import pytest
import torch

from helpers import orc, scenes
from test_gpu_rasterizer_parity import test_sorts_at_the_sizes_where_their_tiles_change as check_sorts

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("totals", (8191, 8192, 8193, 32767, 32768, 32769))   # of 256 each: from memory, through LDS, from memory again
def test_scan_of_block_totals(totals):
    from retinags_amd import _capi
    n = 256 * totals - 3
    x = np.random.default_rng(totals).integers(0, 50, size=n, dtype=np.uint32)
    xi = torch.from_numpy(x.view(np.int32).copy()).to(DEV)
    out = torch.empty_like(xi)
    temp = torch.empty(_capi.lib.rgs_scan_temp_bytes(n), dtype=torch.uint8, device=DEV)
    _capi.check(_capi.lib.rgs_inclusive_sum(_capi.ptr(xi), _capi.ptr(out), n, _capi.ptr(temp),
                                            torch.cuda.current_stream(torch.device(DEV)).cuda_stream))
    assert np.array_equal(out.cpu().numpy().view(np.uint32), orc.inclusive_sum(x))


def _view(width, height):
    from retinags_amd import GaussianRasterizationSettings, GaussianRasterizer
    cam = scenes.look_at_camera((0, 0, 0), (0, 0, 1), (0, -1, 0), width, height, 60.0).to(DEV)
    return GaussianRasterizer(GaussianRasterizationSettings(
        image_height=height, image_width=width, tanfovx=cam.tanfovx, tanfovy=cam.tanfovy, bg=torch.zeros(3, device=DEV), scale_modifier=1.0,
        viewmatrix=cam.world_view_transform, projmatrix=cam.full_proj_transform, projmatrix_inv=cam.projection_matrix_inv,
        range_low=torch.full((3,), -99.0, device=DEV), range_up=torch.full((3,), 99.0, device=DEV), sh_degree=0,
        campos=cam.camera_center, prefiltered=False, debug=False))


def test_copies_of_the_digit_counts():
    """The counts a sort starts from lie in memory once for up to 128 workgroups of the kernel that makes them and several times
    for more: Gaussians behind the camera take the depth order from one to the other (131 072 and 131 073 of them), bounds for
    the instances the key duplication (32 768 and 32 769 positions).  The images stay the same, bit for bit."""
    rasterizer = _view(320, 200)
    scene = scenes.cube_scene(6000, seed=4)
    scene["xyz"][3000:] = scene["xyz"][:3000]
    colors = torch.rand(6000, 3, generator=torch.Generator().manual_seed(2))
    kw = {k: v.to(DEV) for k, v in dict(means3D=scene["xyz"], opacities=scene["opacity"], colors_precomp=colors,
                                        scales=scene["scales"], rotations=scene["rotations"]).items()}

    def run(n, bound):
        padded = {k: torch.cat((v, torch.ones(n - 6000, *v.shape[1:], device=DEV))) for k, v in kw.items()}
        padded["means3D"][6000:, 2] = -5.0
        with torch.no_grad():
            stage = rasterizer.enqueue_geometry(**padded, **({} if bound is None else {"instance_bound": bound}))
            out = rasterizer(means2D=torch.zeros_like(padded["means3D"]), geometry=stage, **padded)
            again = rasterizer(means2D=torch.zeros_like(padded["means3D"]), **padded)
        assert all(torch.equal(a, b) for a, b in zip(out, again))
        return stage.instances(), out

    instances, want = run(6000, None)
    assert 5000 < instances <= 32767 and want[0].max() > 0
    for n, bound in ((131072, None), (131073, None), (6000, 32768), (6000, 32769), (131073, 32767), (131072, 100000), (400001, 3000001)):
        count, got = run(n, bound)
        assert count == instances and torch.equal(got[1][:6000], want[1])
        assert all(torch.equal(got[k], want[k]) for k in (0, 2, 3)), (n, bound)


@pytest.mark.parametrize("n", (8 * 2**20, 8 * 2**20 + 1025))   # 8 192 groups of 1 024 Gaussians: the most of which all are looked at; more
@pytest.mark.parametrize("spread", (1, 700, 2500))             # neighbours in memory, a few per group, one in some groups
def test_groups_without_listed_gaussians(n, spread):
    """3 000 Gaussians of a view among millions behind the camera, `spread` places apart, the last one at the very end: the same
    images, bit for bit, as those 3 000 alone (ties in depth keep their order)."""
    rasterizer = _view(160, 120)
    scene = scenes.cube_scene(3000, seed=8)
    scene["xyz"][1500:] = scene["xyz"][:1500]
    few = dict(means3D=scene["xyz"], opacities=scene["opacity"], colors_precomp=torch.rand(3000, 3, generator=torch.Generator().manual_seed(2)),
               scales=scene["scales"] * 3, rotations=scene["rotations"])
    few = {k: v.to(DEV) for k, v in few.items()}
    at = n - 1 - spread * torch.arange(2999, -1, -1, device=DEV)
    many = {k: torch.ones(n, *v.shape[1:], device=DEV) for k, v in few.items()}
    many["means3D"][:, 2] = -5.0
    for k, v in few.items():
        many[k][at] = v
    with torch.no_grad():
        want = rasterizer(means2D=torch.zeros_like(few["means3D"]), **few)
        got = rasterizer(means2D=torch.zeros_like(many["means3D"]), **many)
    assert (want[1] > 0).sum() > 2000 and torch.equal(want[1], got[1][at]) and int((got[1] > 0).sum()) == int((want[1] > 0).sum())
    for k in (0, 2, 3):
        assert torch.equal(want[k], got[k])


def test_sorts_in_the_largest_tiles():
    """2^26 Gaussians and some more, 2^25 instances and more under 17 tile bits: both sorts take tiles of 16 384 pairs."""
    check_sorts((1 << 26) + 5, 4112, 4096)


@pytest.mark.parametrize("width,height", ((16, 16), (256, 128), (192, 176), (256, 256), (272, 256), (512, 256), (384, 352), (512, 512), (656, 400),
                                          (1024, 512), (832, 640)))
def test_tile_digits_of_every_width(width, height):
    """1, 128, 132, 256, 272, 512, 528, 1 024, 1 025, 2 048 and 2 080 tiles: on both sides of every width of the instance sort's digit, up to one
    pass of 11 bits (two digit values per thread) and the first two passes beyond."""
    check_sorts(70_001, width, height)


@pytest.mark.parametrize("n", ((1 << 20) + 4097, 34_000_003))   # sort tiles of 8 192 and of 16 384 pairs
@pytest.mark.parametrize("width,height", ((512, 512), (1024, 512)))
def test_wide_tile_digits_in_larger_tiles(n, width, height):
    check_sorts(n, width, height)


@pytest.mark.parametrize("n", (8, 1023, 1024, 1025, 1026, 1027, 4096 + 6))
def test_totals_of_ragged_groups(n):
    """All in view: the sums of 1 024 tile counts where the last group is whole, short of a quad or a few counts beyond."""
    check_sorts(n, 400, 300)


@pytest.mark.parametrize("n", (9, 65, 4095, 4096, 4097, 8191, 8192, 8193, 8192 + 1027))
def test_order_of_few_gaussians_by_one_workgroup(n):
    """Up to 8 192 Gaussians are ordered out of LDS, four or eight per thread; one more by the general path."""
    check_sorts(n, 400, 300)


@pytest.mark.parametrize("n", (900, 4096, 8000, 9000))
def test_depths_that_need_the_fourth_pass(n):
    """Gaussians at depths below and beyond 8 192, equal depths among them and a third behind the camera, on both sides of the bound up to which one
    workgroup orders them: depth order and offsets against a stable argsort, the images against the checker."""
    from test_gpu_rasterizer_parity import _check_forward_stages, _scene_sub
    scene = scenes.cube_scene(n, seed=n)
    scene["xyz"][1::2] = scene["xyz"][::2][:scene["xyz"][1::2].shape[0]]
    far, behind = torch.arange(n) % 4 >= 2, torch.arange(n) % 3 == 0
    scene["xyz"][far] *= 4000.0
    scene["scales"][far] *= 4000.0
    scene["xyz"][behind, 2] *= -1.0
    cam = scenes.look_at_camera((0, 0, 0), (0, 0, 1), (0, -1, 0), 160, 100, 60.0)
    st = _check_forward_stages(_scene_sub(scene), cam, torch.tensor([0.1, 0.2, 0.3]), max_borderline=2e-3)
    listed = st.depths[st.radii > 0]
    assert listed.max() > 8192 and listed.min() < 8 and 0.3 * n < len(listed) < 0.8 * n
