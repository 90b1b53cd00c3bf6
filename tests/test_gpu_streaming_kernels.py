"""Kernels that move rows between layouts 16 bytes at a time: sizes around a workgroup's share, and arrays that do not start at
a multiple of 16 bytes."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _tensor(shape, gen, offset):
    """Normal values in memory that starts `offset` floats behind a multiple of 16 bytes."""
    room = torch.empty(int(np.prod(shape)) + offset, device=DEV)
    t = room[offset:].view(shape)
    return t.copy_(torch.randn(*shape, generator=gen, device=DEV))


@pytest.mark.parametrize("rest", (1, 2, 3, 8, 14, 15, 16))
@pytest.mark.parametrize("offset", (0, 1))
def test_sh_rows_are_joined_and_split_bit_for_bit(rest, offset):
    from retinags_amd import _host
    gen = torch.Generator(device=DEV).manual_seed(rest)
    for n in (1, 2, 127, 128, 129, 1021):
        dc, more = _tensor((n, 1, 3), gen, offset), _tensor((n, rest, 3), gen, offset)
        small = [torch.randn(n, k, generator=gen, device=DEV) for k in (3, 4, 1)]
        leaves = [t.requires_grad_(True) for t in (dc, more, *small)]
        shs = _host.activate(*leaves, 0)[0]
        assert torch.equal(shs.detach(), torch.cat((dc, more), dim=1).detach())
        upstream = torch.randn(n, 1 + rest, 3, generator=gen, device=DEV)
        d_dc, d_more = torch.autograd.grad([shs], leaves[:2], [upstream])
        assert torch.equal(d_dc, upstream[:, :1]) and torch.equal(d_more, upstream[:, 1:])


@pytest.mark.parametrize("n", (1, 1023, 1024, 1025, 4097))
def test_activated_values_at_the_edges_of_a_workgroup(n):
    """Every row against torch's expressions in 64 bits: a library exp, division and square root differ by a few units in
    the last place (2^-23 each), so 1e-6 relative leaves room for eight of them."""
    from retinags_amd import _host
    gen = torch.Generator(device=DEV).manual_seed(n)
    features = torch.randn(n, 1, 3, generator=gen, device=DEV), torch.randn(n, 15, 3, generator=gen, device=DEV)
    small = [torch.randn(n, k, generator=gen, device=DEV) for k in (3, 4, 1)]
    leaves = [t.requires_grad_(True) for t in (*features, *small)]
    outs = _host.activate(*leaves, 0)[1:]
    upstream = [torch.randn_like(o) for o in outs]
    grads = torch.autograd.grad(outs, leaves[2:], upstream)
    wide = [t.detach().double().requires_grad_(True) for t in small]
    want = [torch.exp(wide[0]), torch.nn.functional.normalize(wide[1]), torch.sigmoid(wide[2])]
    want_grads = torch.autograd.grad(want, wide, [u.double() for u in upstream])
    for got, ref in zip(outs, want):
        assert torch.allclose(got.double(), ref, rtol=1e-6, atol=0)
    for got, ref in zip(grads, want_grads):
        # (the quaternion's gradient is a difference of terms as large as the upstream gradient)
        assert float((got.double() - ref).norm() / ref.norm()) < 2e-6


@pytest.mark.parametrize("n", (1, 63, 64, 65, 127, 128, 129, 777))
def test_gradient_rows_leave_alike_on_and_off_a_16_byte_boundary(n, monkeypatch):
    """Rows of whole wavefronts go out 16 bytes per lane, those of the last and of arrays off a 16-byte boundary one float at a
    time; every row is written either way.  Two runs differ by the order of the atomic additions alone (1e-4, as between
    repeats)."""
    from helpers import rel_l2
    from retinags_amd import GaussianRasterizationSettings, GaussianRasterizer, rasterizer
    from retinags_amd.harness import scenes
    gen = torch.Generator().manual_seed(n)
    cam = scenes.look_at_camera((0, 0, 0), (0, 0, 1), (0, -1, 0), 96, 64, 60.0).to(DEV)
    given = dict(means3D=torch.cat((torch.rand(n, 2, generator=gen) * 4 - 2, torch.rand(n, 1, generator=gen) * 6 - 1), 1),
                 opacities=torch.rand(n, 1, generator=gen), shs=torch.randn(n, 16, 3, generator=gen) * 0.2,
                 scales=torch.rand(n, 3, generator=gen) * 0.2, rotations=torch.nn.functional.normalize(torch.randn(n, 4, generator=gen)))
    given = {k: v.to(DEV).requires_grad_(True) for k, v in given.items()}
    given["means2D"] = torch.zeros(n, 3, device=DEV, requires_grad=True)
    settings = GaussianRasterizationSettings(
        image_height=64, image_width=96, tanfovx=cam.tanfovx, tanfovy=cam.tanfovy, bg=torch.zeros(3, device=DEV), scale_modifier=1.0,
        viewmatrix=cam.world_view_transform, projmatrix=cam.full_proj_transform, projmatrix_inv=cam.projection_matrix_inv,
        range_low=torch.full((3,), -99.0, device=DEV), range_up=torch.full((3,), 99.0, device=DEV), sh_degree=3,
        campos=cam.camera_center, prefiltered=False, debug=False)
    upstream = torch.randn(3, 64, 96, generator=gen).to(DEV)
    make, made = rasterizer._gradient_outputs, []

    def run(offset):
        def arrays(*args, **kwargs):
            out = make(*args, **kwargs)
            for name, t in out.items():
                if t is not None and name != "sums":
                    if offset and t.dim() == 2 and t.shape[1] in (3, 6):
                        out[name] = torch.empty(t.numel() + offset, device=DEV)[offset:].view(t.shape)
                    out[name].fill_(float("nan"))
            made.append(out)
            return out
        monkeypatch.setattr(rasterizer, "_gradient_outputs", arrays)
        color, radii = GaussianRasterizer(settings)(**given)[:2]
        torch.autograd.grad([color], list(given.values()), [upstream])
        return radii, {k: v for k, v in made[-1].items() if v is not None and k != "sums"}

    radii, even = run(0)
    for offset in (1, 2):
        odd = run(offset)[1]
        for name, t in even.items():
            assert not torch.isnan(t).any() and not torch.isnan(odd[name]).any(), name
            assert rel_l2(odd[name].cpu().numpy(), t.cpu().numpy()) <= 1e-4, name
            assert (t[radii <= 0] == 0).all() and (odd[name][radii <= 0] == 0).all(), name


@pytest.mark.parametrize("n", (2**20 - 1, 2**20, 2**20 + 1))
def test_geometry_is_the_same_with_and_without_streaming_stores(n):
    """Up to 2^20 - 1 Gaussians the forward's geometry is stored one way and beyond the other; radii and images of a scene whose
    further Gaussians lie behind the camera do not depend on how many those are."""
    from retinags_amd import GaussianRasterizationSettings, GaussianRasterizer
    from retinags_amd.harness import scenes
    cam = scenes.look_at_camera((0, 0, 0), (0, 0, 1), (0, -1, 0), 160, 120, 60.0).to(DEV)
    settings = GaussianRasterizationSettings(
        image_height=120, image_width=160, tanfovx=cam.tanfovx, tanfovy=cam.tanfovy, bg=torch.zeros(3, device=DEV), scale_modifier=1.0,
        viewmatrix=cam.world_view_transform, projmatrix=cam.full_proj_transform, projmatrix_inv=cam.projection_matrix_inv,
        range_low=torch.full((3,), -99.0, device=DEV), range_up=torch.full((3,), 99.0, device=DEV), sh_degree=3,
        campos=cam.camera_center, prefiltered=False, debug=False)
    scene = scenes.cube_scene(3000, seed=8)
    few = dict(means3D=scene["xyz"], opacities=scene["opacity"], shs=scene["shs"], scales=scene["scales"] * 3, rotations=scene["rotations"])
    few = {k: v.to(DEV) for k, v in few.items()}
    many = {k: torch.cat((torch.ones(n - 3000, *v.shape[1:], device=DEV), v)) for k, v in few.items()}
    many["means3D"][:n - 3000, 2] = -5.0
    with torch.no_grad():
        color, radii, depth, alpha = GaussianRasterizer(settings)(means2D=torch.zeros_like(few["means3D"]), **few)
        color_m, radii_m, depth_m, alpha_m = GaussianRasterizer(settings)(means2D=torch.zeros_like(many["means3D"]), **many)
    assert (radii > 0).sum() > 2000 and torch.equal(radii, radii_m[n - 3000:]) and (radii_m[:n - 3000] == 0).all()
    assert torch.equal(color, color_m) and torch.equal(depth, depth_m) and torch.equal(alpha, alpha_m)
