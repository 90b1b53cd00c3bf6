"""Where the geometry stage's instance count lands: pinned words are written by the kernel that adds the counts up, other memory by a copy."""
import ctypes

import numpy as np
import pytest
import torch

from helpers import scenes

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


class _Geometry:
    def __init__(self, n):
        from retinags_amd import _capi
        self.capi, self.n = _capi, n
        scene = scenes.cube_scene(n, seed=n)
        cam = scenes.look_at_camera((0, 0, 0), (0, 0, 1), (0, -1, 0), 160, 120, 60.0)
        self.tan = cam.tanfovx, cam.tanfovy
        self.colors = torch.rand(n, 3, device=DEV)
        self.t = [scene[k].to(DEV).contiguous() for k in ("xyz", "opacity", "scales", "rotations")]
        self.cam = [t.to(DEV).contiguous() for t in (cam.world_view_transform, cam.full_proj_transform, cam.camera_center)]
        self.radii = torch.zeros(n, dtype=torch.int32, device=DEV)
        self.bytes = _capi.lib.rgs_geom_bytes(n)
        self.ws = torch.zeros(self.bytes, dtype=torch.uint8, device=DEV)

    def run(self, entry, word, *tail):
        p, (xyz, opacity, scales, rotations), (view, proj, campos) = self.capi.ptr, self.t, self.cam
        stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        self.capi.check(entry(self.n, 0, 0, 160, 120, p(xyz), None, p(self.colors), p(opacity), p(scales), 1.0, p(rotations), None, p(view), p(proj),
                              p(campos), *self.tan, 0, p(self.radii), p(self.ws), self.bytes, ctypes.c_void_p(word), *tail, stream, 0))

    def expected(self):
        torch.cuda.synchronize()
        from helpers import view_ws
        return int(view_ws(self.ws, self.capi.geom_layout(self.n)["tiles_touched"], self.n, np.uint32).sum())


@pytest.mark.parametrize("n", (1, 300, 9000))
@pytest.mark.parametrize("memory", ("pageable", "pinned", "pinned, further in"))
def test_the_count_lands_in_any_host_memory(n, memory):
    g = _Geometry(n)
    words = torch.full((64,), -7, dtype=torch.int32, pin_memory=memory != "pageable")
    at = 5 if memory == "pinned, further in" else 0
    for _ in range(2):
        words.fill_(-7)
        g.run(g.capi.lib.rgs_forward_geom, words.data_ptr() + 4 * at)
        assert int(words[at]) == g.expected() and int((words != -7).sum()) == 1
        words.fill_(-7)
        g.run(g.capi.lib.rgs_forward_geom_enqueue, words.data_ptr() + 4 * at, None)
        torch.cuda.synchronize()
        assert int(words[at]) == g.expected() and int((words != -7).sum()) == 1


def test_the_count_of_every_replay():
    """A captured geometry stage writes its pinned word again on every replay, from the Gaussians of that time."""
    g = _Geometry(5000)
    word = torch.zeros(1, dtype=torch.int32, pin_memory=True)
    g.run(g.capi.lib.rgs_forward_geom_enqueue, word.data_ptr(), None)
    first = g.expected()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        g.run(g.capi.lib.rgs_forward_geom_enqueue, word.data_ptr(), None)
    seen = []
    for keep in (5000, 2500, 5000, 1000):
        g.t[0][:, 2] = g.t[0][:, 2].abs()
        g.t[0][keep:, 2] *= -1.0
        word.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        want = g.expected()
        assert int(word[0]) == want
        seen.append(want)
    assert seen[0] == seen[2] == first and seen[0] > seen[1] > seen[3] > 0
