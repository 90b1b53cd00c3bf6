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
