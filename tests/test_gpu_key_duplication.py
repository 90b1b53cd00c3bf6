"""The kernel that writes the (tile, Gaussian) instances, at the sizes where its runs of 256 positions and its tables end, and those
that find the tiles' ranges in them and file them for strips."""
import numpy as np
import pytest
import torch

from helpers import scenes, view_ws
from test_gpu_rasterizer_parity import _check_forward_stages, _run_gpu_forward, _scene_sub

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


# 8 192 groups of 1 024 instances: up to there a workgroup each, beyond that a workgroup takes several
@pytest.mark.parametrize("n", (4_800_000, 5_000_000))
def test_ranges_and_strip_lists_of_many_groups(n):
    from retinags_amd import _capi
    width, height = 700, 520
    gen = torch.Generator(device="cuda:0").manual_seed(n)
    xyz = torch.rand(n, 3, generator=gen, device="cuda:0") * 1.6 - 0.8
    xyz[:, 2] += 4.0
    q = torch.zeros(n, 4, device="cuda:0")
    q[:, 0] = 1.0
    sub = dict(xyz=xyz, opacity=torch.full((n, 1), 0.5, device="cuda:0"), scales=torch.full((n, 3), 0.003, device="cuda:0"), rotations=q,
               shs=torch.zeros(n, 1, 3, device="cuda:0"), low=torch.full((3,), -9.0), up=torch.full((3,), 9.0))
    cam = scenes.look_at_camera((0.0, 0.0, 0.0), (0.0, 0.0, 1.0), (0, -1, 0), width, height, 60.0)
    R, _, _, _, _, _, binning, img = _run_gpu_forward(sub, cam, torch.zeros(3), torch.device("cuda:0"), sh_degree=0)
    torch.cuda.synchronize()
    assert (R > 8192 * 1024) == (n > 4_900_000)
    b, im, tiles = _capi.binning_layout(R, width, height), _capi.image_layout(width, height), ((width + 15) // 16) * ((height + 15) // 16)
    keys = view_ws(binning, b["keys_sorted"], R, np.uint32)
    tile = keys & np.uint32(0xFFFFFF)
    ranges = view_ws(img, im["ranges"], 2 * tiles, np.uint32).reshape(tiles, 2).astype(np.int64)
    begin, end = np.searchsorted(tile, np.arange(tiles)), np.searchsorted(tile, np.arange(tiles), side="right")
    some = end > begin
    assert np.array_equal(ranges[some], np.stack([begin, end], 1)[some]) and (ranges[~some] == 0).all()
    # every strip's list: the positions in the tile of the entries filed for it, in their order
    lists = view_ws(binning, b["strip_lists"], 4 * R, np.uint32)
    for t in np.flatnonzero(some)[::37]:
        x, y = ranges[t]
        for s in range(4):
            filed = np.flatnonzero((keys[x:y] >> (24 + s)) & 1)
            at = 4 * x + s * (y - x)
            assert np.array_equal(lists[at:at + len(filed)] & np.uint32(0x7FFFFFFF), filed)
