"""The batched march's step pairs (no counts asked for) against its single steps (fetch counts asked for), bit for bit:
rays that end at the 256-step limit before a wall and rays that reach one just inside it, short and long limits, empty,
sparse and dense scenes, every steps-per-block setting."""
import numpy as np
import pytest
import torch

from helpers import assert_bitwise

pytestmark = pytest.mark.gpu


def _items(api, ctx):
    """Volumes of uneven size with G-buffers of random surface points and normals."""
    rng = np.random.default_rng(21)
    items = []
    for k, (dims, fill, wall) in enumerate([((130, 40, 40), 0.0, 127), ((40, 140, 33), 0.0005, 128), ((64, 64, 64), 0.01, None),
                                            ((20, 24, 150), 0.2, 100), ((150, 30, 30), 0.0, 129)]):
        shape = dims[::-1]
        host = ((rng.random(shape) < fill) * rng.integers(1, 256, shape)).astype(np.uint8)
        axis = int(np.argmax(dims))
        if wall is not None:
            at = [slice(None)] * 3
            at[2 - axis] = wall
            host[tuple(at)] = 255
        occ = api.Volume(ctx, *dims, nlevels=0)
        occ.upload_region(host, [(0, 0, 0, *dims)])
        from voxelengine_amd import views
        w, h = 70 + 13 * k, 50 - 3 * k
        vd = views.make_view((0.0, 4.0, 0.0), (1.0, 0.0, 1.0), w, h, frame=k)
        g = api.GBuffer(w, h)
        pos = rng.uniform(0.0, 1.0, (w * h, 3)) * 2.0 * np.array(dims)
        pos[:, axis] *= 0.04
        n = rng.normal(size=(w * h, 3)) * 0.05
        n[:, axis] += 1.0                      # rays down the long axis
        n /= np.linalg.norm(n, axis=1, keepdims=True)
        g.pos.copy_(torch.from_numpy(pos.astype(np.float32)))
        g.normal.copy_(torch.from_numpy(n.astype(np.float32)))
        g.material.copy_(torch.from_numpy(rng.integers(0, 4, w * h).astype(np.uint8)))
        items.append((occ, vd, g, axis))
    return items


@pytest.mark.parametrize("steps", [2, 4, 8, 16])
@pytest.mark.parametrize("maxt", [(1e4, 1e4), (20.0, 3.0)])
def test_pairs_match_single_steps(ctx, steps, maxt):
    from voxelengine_amd import api, configs
    items = _items(api, ctx)
    pal = torch.from_numpy(configs.make_palette()).cuda()
    try:
        ctx.set_tuning(steps=steps)
        for seed in (1, 2):
            p = configs.trace_params(n_shadow=1, n_ao=5, n_spec=1, ao_maxt=maxt[1], shadow_maxt=maxt[0], spec_maxt=maxt[0], seed=seed)
            res = []
            for counted in (False, True):
                outs = [api.Visibility(vd["width"], vd["height"], fetches=counted) for _, vd, _, _ in items]
                b = api.Batch(ctx, [(occ, vd, g, o) for (occ, vd, g, _), o in zip(items, outs)], pal, p)
                b.launch()
                torch.cuda.synchronize()
                res.append(outs)
            limited = 0
            for k, (x, y) in enumerate(zip(*res)):
                for f in ("shadow", "ao", "spec"):
                    assert_bitwise(getattr(x, f).cpu().numpy(), getattr(y, f).cpu().numpy(), f"item {k} {f}")
                limited += int((y.fetches >= 4 * 256).sum())   # a ray of 256 free steps counts 1024
            if maxt[0] > 256.0:
                assert limited > 100
    finally:
        ctx.reset_tuning()
