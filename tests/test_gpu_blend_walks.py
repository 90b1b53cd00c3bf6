"""How the blends deal out strips and walk them, against the checker."""
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
