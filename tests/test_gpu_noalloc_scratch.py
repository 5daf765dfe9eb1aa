"""vx_trace_noalloc over its shared scratch on views that auto would trace with
the scratch-free kernel: the ray-parallel kernel is named (kernel 2), so the
queue counters, the tile ranges, the listed rays and the resolve run on what
earlier and larger calls left there, eagerly and in replays of a recorded call.
The reference is the per-pixel kernel (kernel 1)."""
import ctypes as C

import pytest
import torch

from helpers import device_scene

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def scene(ctx):
    from voxelengine_amd import api
    return device_scene(api, ctx, 96, seed=21, nboxes=40)


def _setup(ctx, scene, W, H, ao, fetches):
    from voxelengine_amd import _lib, api, configs, views
    L = _lib.lib()
    model, occ, vol = scene
    pal = torch.from_numpy(configs.make_palette()).cuda()
    params = configs.trace_params(n_ao=ao, ao_maxt=32.0, n_spec=1, march="dda")
    tp = api.trace_params(params)
    vd = views.scene_view((96, 96, 96), W, H)
    g = api.GBuffer(W, H)
    api.primary(ctx, model, vd, g)
    ref, out = api.Visibility(W, H, fetches=fetches), api.Visibility(W, H, fetches=fetches)
    ctx.set_tuning(kernel=1)
    api.trace(ctx, occ, vd, g, pal, params, ref)
    ctx.set_tuning(kernel=2)
    v, gs, o = api.view_struct(vd), g.struct(), out.struct()

    def call(stream):
        assert L.vx_trace_noalloc(ctx.h, occ.h, C.byref(v), C.byref(gs), api._ptr(pal), C.byref(tp), C.byref(o),
                                  stream.cuda_stream) == 0, L.vx_last_error()

    def same():
        torch.cuda.synchronize()
        for f in ("shadow", "ao", "spec") + (("fetches",) if fetches else ()):
            assert torch.equal(getattr(out, f).view(torch.uint8), getattr(ref, f).view(torch.uint8)), f

    def spoil():
        out.shadow.fill_(7)
        out.ao.fill_(-1.0)
        out.spec.fill_(-1.0)

    assert int((g.material > 0).sum().item()) > 0.3 * W * H
    call.inputs = g, pal    # (the structs hold their addresses)
    return call, same, spoil


@pytest.mark.parametrize("ao", [16, 64])
@pytest.mark.parametrize("fetches", [False, True])
def test_calls_over_each_others_scratch(ctx, scene, ao, fetches):
    try:
        # (at 64 AO rays the first view spans several tile ranges)
        for W, H in ((400, 300), (123, 77), (61, 43), (400, 300)):
            call, same, spoil = _setup(ctx, scene, W, H, ao, fetches)
            spoil()
            call(torch.cuda.current_stream())
            same()
    finally:
        ctx.reset_tuning()


def test_replays_over_each_others_scratch(ctx, scene):
    side = torch.cuda.Stream()
    try:
        recorded = []
        for W, H, ao in ((160, 96, 8), (400, 300, 64)):
            call, same, spoil = _setup(ctx, scene, W, H, ao, False)
            torch.cuda.synchronize()
            call(side)
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=side):
                call(side)
            recorded.append((graph, same, spoil, call))
        for k in range(3):
            for graph, same, spoil, call in recorded:
                spoil()
                _ = torch.randn(4096, device="cuda").sum().item()    # eager work between replays
                graph.replay()
                same()
                spoil()
                call(torch.cuda.current_stream())
                same()
    finally:
        ctx.reset_tuning()
