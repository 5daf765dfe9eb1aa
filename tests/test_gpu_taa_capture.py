"""The temporal accumulation recorded into a graph after one ordinary call of its
size (of any shape with as many pixels, with or without motion): plain, and with
an output over its light, which goes through scratch. Every replay equals the
eager, non-overlapping call."""
import numpy as np
import pytest
import torch

from test_gpu_taa_tiles import _inputs
from voxelengine_amd import configs, views

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("overlap", [False, True])
def test_recorded_after_an_ordinary_call(overlap):
    from voxelengine_amd import api
    W, H = 200, 90
    light, last, motion, depth, n, mat = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in _inputs(W, H, 3))
    pal = torch.from_numpy(configs.make_palette()).cuda()
    view = lambda w, h: views.make_view((0.0, 2.0, 0.0), (1.0, 0.0, 1.0), w, h, frame=1)
    ref, buf = (torch.zeros((W * H, 4), dtype=torch.float32, device="cuda") for _ in range(2))
    over = buf.view(-1)[:W * H * 3].view(W * H, 3) if overlap else light
    side = torch.cuda.Stream()
    c = api.Context(0)
    try:
        # the first call: another shape of as many pixels, no motion, no overlap
        api.light_taa(c, view(H, W), light, last, ref, depth, n, mat, pal)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            api.light_taa(c, view(W, H), over, last, buf, depth, n, mat, pal, motion=motion, stream=side.cuda_stream)
        torch.cuda.synchronize()
        for _ in range(3):
            api.light_taa(c, view(W, H), light, last, ref, depth, n, mat, pal, motion=motion)
            buf.fill_(-1.0)
            if overlap:
                over.copy_(light)
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(buf.view(torch.int32), ref.view(torch.int32))
    finally:
        c.close()
