"""vx_trace_noalloc records no kernel timing: with vx_ctx_profile on, small and
large views, eagerly and under graph capture, leave the launch count at what
vx_trace alone made it, and the collection can still be read."""
import ctypes as C

import pytest
import torch

from helpers import device_scene

pytestmark = pytest.mark.gpu


# one kernel for the whole view, and (above 16384 tiles x rays) the ray-parallel one
@pytest.mark.parametrize("W,H", [(61, 43), (640, 400)])
def test_noalloc_trace_is_not_timed(ctx, W, H):
    from voxelengine_amd import _lib, api, configs, views
    L = _lib.lib()
    model, occ, vol = device_scene(api, ctx, 64, seed=9, nboxes=20)
    pal = torch.from_numpy(configs.make_palette()).cuda()
    params = configs.trace_params(n_ao=16, ao_maxt=32.0, n_spec=1, march="dda")
    tp = api.trace_params(params)
    vd = views.scene_view((64, 64, 64), W, H)
    g = api.GBuffer(W, H)
    api.primary(ctx, model, vd, g)
    vis = api.Visibility(W, H)
    v, gs, o = api.view_struct(vd), g.struct(), vis.struct()

    def noalloc(stream):
        assert L.vx_trace_noalloc(ctx.h, occ.h, C.byref(v), C.byref(gs), api._ptr(pal), C.byref(tp), C.byref(o),
                                  stream.cuda_stream) == 0, L.vx_last_error()

    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    ctx.profile(True)
    try:
        for _ in range(2):
            noalloc(side)
        torch.cuda.synchronize()
        assert ctx.profile_read() == (0.0, 0)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            noalloc(side)
        for _ in range(2):
            graph.replay()
        torch.cuda.synchronize()
        assert ctx.profile_read() == (0.0, 0)
        api.trace(ctx, occ, vd, g, pal, params, vis)
        ms, n = ctx.profile_read()
        assert n == 1 and ms > 0.0
    finally:
        ctx.profile(False)
