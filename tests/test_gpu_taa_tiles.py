"""The tiled temporal accumulation against the oracle, bit for bit: images smaller than a tile, ragged ones on both
tile sizes, spiral samples past the staged neighbourhood (variance above 1), tiles of sky only, values that a zero
weight does not cancel, and an output that overlaps an input."""
import numpy as np
import pytest

from helpers import assert_bitwise
from voxelengine_amd import configs, views

pytestmark = pytest.mark.gpu


def _inputs(W, H, seed):
    """Surfaces in patches, so that neighbours share material and normal, with edges between them."""
    rng = np.random.default_rng(seed)
    npx = W * H
    y, x = np.divmod(np.arange(npx), W)
    patch = (x // 11) * 7919 + (y // 7) * 104729
    mat = (1 + patch % 5).astype(np.uint8)
    n = rng.normal(size=(64, 3))[patch % 64]
    n = (n / np.linalg.norm(n, axis=1, keepdims=True)).astype(np.float32)
    depth = (0.002 + 1e-6 * (patch % 50)).astype(np.float32)
    sky = (y < H // 4) | (patch % 13 == 0)
    mat[sky], depth[sky], n[sky] = 0, 1.0, 0.0
    motion = (rng.normal(size=(npx, 2)) * 0.003).astype(np.float32)
    motion[patch % 17 == 1] += np.float32(0.3)          # another object: far motion, some of it off the image
    motion[sky] = 0.0
    light = rng.random((npx, 3)).astype(np.float32)
    last = rng.random((npx, 4)).astype(np.float32)
    last[patch % 3 == 2, 3] *= 4.0                      # samples past the tile's neighbourhood
    return light, last, motion, depth, n, mat


def _run(ctx, oracle, W, H, arrays, motion=True, seed=4):
    import torch
    from voxelengine_amd import api
    light, last, mo, depth, n, mat = arrays
    pal = configs.make_palette()
    vd = views.make_view((0.0, 2.0, 0.0), (1.0, 0.0, 1.0), W, H, frame=2)
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    out = torch.zeros((W * H, 4), dtype=torch.float32, device="cuda")
    api.light_taa(ctx, vd, d(light), d(last), out, d(depth), d(n), d(mat), d(pal), motion=d(mo) if motion else None, seed=seed)
    torch.cuda.synchronize()
    ref = oracle.light_taa(W, H, 2, seed, light, last, mo if motion else np.zeros_like(mo), depth, n, mat, pal)
    assert_bitwise(out.cpu().numpy(), ref, f"{W}x{H}")


@pytest.mark.parametrize("size", [(1, 1), (3, 50), (16, 16), (33, 31), (97, 45), (737, 737), (1024, 520)])
def test_taa_tiles_match_oracle(ctx, oracle, size):
    _run(ctx, oracle, *size, _inputs(*size, seed=sum(size)), motion=size != (97, 45))


def test_taa_uncancelled_values_match_oracle(ctx, oracle):
    W, H = 80, 48
    light, last, motion, depth, n, mat = _inputs(W, H, 8)
    rng = np.random.default_rng(1)
    light[rng.random(W * H) < 0.01, 1] = np.inf
    n[(rng.random(W * H) < 0.01) & (mat > 0)] = [1e30, 0.0, 0.0]
    import torch
    from voxelengine_amd import api
    pal = configs.make_palette()
    vd = views.make_view((0.0, 2.0, 0.0), (1.0, 0.0, 1.0), W, H, frame=2)
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    out = torch.zeros((W * H, 4), dtype=torch.float32, device="cuda")
    api.light_taa(ctx, vd, d(light), d(last), out, d(depth), d(n), d(mat), d(pal), motion=d(motion), seed=4)
    got = out.cpu().numpy()
    ref = oracle.light_taa(W, H, 2, 4, light, last, motion, depth, n, mat, pal)
    nan = np.isnan(ref)          # the default NaN's sign differs between the GPU and x86
    assert nan.any()
    np.testing.assert_array_equal(np.isnan(got), nan)
    assert_bitwise(np.where(nan, np.float32(0), got), np.where(nan, np.float32(0), ref), "uncancelled")


def test_taa_output_over_its_light(ctx):
    import torch
    from voxelengine_amd import api
    W, H = 200, 90
    light, last, motion, depth, n, mat = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in _inputs(W, H, 3))
    pal = torch.from_numpy(configs.make_palette()).cuda()
    vd = views.make_view((0.0, 2.0, 0.0), (1.0, 0.0, 1.0), W, H, frame=1)
    ref = torch.zeros((W * H, 4), dtype=torch.float32, device="cuda")
    api.light_taa(ctx, vd, light, last, ref, depth, n, mat, pal, motion=motion)
    buf = torch.zeros((W * H, 4), dtype=torch.float32, device="cuda")
    over = buf.view(-1)[:W * H * 3].view(W * H, 3)
    over.copy_(light)
    api.light_taa(ctx, vd, over, last, buf, depth, n, mat, pal, motion=motion)
    assert torch.equal(buf.view(torch.int32), ref.view(torch.int32))
