"""The kernel that writes the (tile, Gaussian) instances, at the sizes where its runs of 256 positions and its tables end."""
import pytest
import torch

from helpers import scenes
from test_gpu_rasterizer_parity import _check_forward_stages, _scene_sub

pytestmark = pytest.mark.gpu


# one instance per Gaussian or hardly more (255 Gaussians and more begin inside a run), a run's worth of a Gaussian and more, and
# more tile columns than the table of their coordinates has room for
@pytest.mark.parametrize("n,width,height,size", [(255, 96, 80, 0.05), (256, 96, 80, 0.05), (257, 96, 80, 0.05), (1500, 640, 480, 0.05),
                                                 (1500, 640, 480, 3.0), (70, 330, 290, 60.0), (300, 131200, 16, 1.0)])
def test_runs_of_positions(n, width, height, size):
    scene = scenes.cube_scene(n, seed=n)
    scene["scales"] = scene["scales"] * size
    cam = scenes.look_at_camera((0.0, 0.0, 0.0), (0.0, 0.0, 4.0), (0, -1, 0), width, height, 60.0)
    st = _check_forward_stages(_scene_sub(scene), cam, torch.tensor([0.2, 0.1, 0.05]))
    assert st.R > 0
