"""The adjoint's accumulator across calls that fail: a call whose finishing
launch is left out (the injected failure of the check between the two launches)
or whose checks fail at all leaves nothing in the gradients of the next call,
of a batched one, of a call recorded before or after it, or of one on another
stream. Integer sums: every repetition gives the same bits."""
import pytest
import torch

from helpers import device_scene

pytestmark = pytest.mark.gpu


@pytest.fixture
def case(ctx):
    from voxelengine_amd import api, configs, views
    W, H = 160, 90
    model, occ, vol = device_scene(api, ctx, 64, seed=21, nboxes=10)
    vd = views.scene_view(model.dims, W, H, variant=3)
    g = api.GBuffer(W, H)
    api.primary(ctx, model, vd, g)
    pal = torch.from_numpy(configs.make_palette()).cuda()
    vis = api.Visibility(W, H)
    api.trace(ctx, occ, vd, g, pal, configs.trace_params(n_ao=8, ao_maxt=32.0, n_spec=0), vis)
    dl = torch.randn((W * H, 3), device="cuda", generator=torch.Generator("cuda").manual_seed(4))
    light = configs.default_light()
    out = torch.empty((256, 6), device="cuda"), torch.empty(6, device="cuda")

    def single(stream=None, ctx=ctx):
        api.shade_backward(ctx, vd, g, vis, pal, light, dl, *out, stream=stream)

    def batch(stream=None):
        api.shade_backward_batch(ctx, [(vd, g, vis, dl, None)], pal, light, *out, stream=stream)

    def result(call, **kw):
        for o in out:
            o.fill_(7.0)
        torch.cuda.synchronize()
        call(**kw)
        torch.cuda.synchronize()
        return [o.clone() for o in out]

    yield dict(single=single, batch=batch, result=result, api=api)
    api.inject_failure(api.FAIL_LAUNCH, -1)


def _same(a, b):
    return all(torch.equal(x.view(torch.int32), y.view(torch.int32)) for x, y in zip(a, b))


@pytest.mark.parametrize("form", ["single", "batch"])
@pytest.mark.parametrize("check", [0, 1])
def test_next_call_after_a_failed_one(case, form, check):
    from voxelengine_amd import _lib
    api, result = case["api"], case["result"]
    ref = result(case["single"])
    assert float(ref[0].abs().sum()) > 0 and _same(result(case["batch"]), ref)
    api.inject_failure(api.FAIL_LAUNCH, check)
    with pytest.raises(_lib.VXError) as e:
        case[form]()
    assert e.value.code == _lib.VX_ERR_DEVICE
    # the failed call's clean-up, and again once it is settled
    for call in (case["single"], case["batch"], case["single"]):
        assert _same(result(call), ref)
    # a failure of the clearing launch of the call after a failed one
    api.inject_failure(api.FAIL_LAUNCH, 0)
    with pytest.raises(_lib.VXError):
        case[form]()
    api.inject_failure(api.FAIL_LAUNCH, 0)
    with pytest.raises(_lib.VXError):
        case[form]()
    assert _same(result(case["single"]), ref) and _same(result(case["batch"]), ref)


def test_recorded_calls_around_a_failed_one(case):
    from voxelengine_amd import _lib
    api, result = case["api"], case["result"]
    ref = result(case["single"])
    side = torch.cuda.Stream()

    def record():
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            case["single"](stream=side.cuda_stream)
        torch.cuda.synchronize()
        return graph

    before = record()
    api.inject_failure(api.FAIL_LAUNCH, 0)
    with pytest.raises(_lib.VXError):
        case["single"]()
    after = record()
    # (the recorded calls have not run: the accumulator is as the failed call left it)
    assert _same(result(before.replay), ref)
    for _ in range(2):
        assert _same(result(after.replay), ref)
        assert _same(result(case["single"]), ref)
        assert _same(result(before.replay), ref)


def test_first_call_of_a_context_on_another_stream(case):
    api, result = case["api"], case["result"]
    ref = result(case["single"])
    side = torch.cuda.Stream()
    for _ in range(4):
        # the context's allocation holds what a freed one left there
        junk = torch.full((1 << 20,), 3, dtype=torch.int64, device="cuda")
        torch.cuda.synchronize()
        del junk
        torch.cuda.empty_cache()
        c = api.Context(0)
        try:
            case["single"](stream=side.cuda_stream, ctx=c)
            torch.cuda.synchronize()
            assert _same(result(case["single"], ctx=c), ref)
            assert _same(result(case["single"], stream=side.cuda_stream, ctx=c), ref)
        finally:
            c.close()
