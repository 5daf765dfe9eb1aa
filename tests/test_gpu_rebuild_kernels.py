"""The volume's write kernels bit for bit against the oracle where their forms
meet: axis-keeping transforms (whole 64-bit cell masks, shifted, split over
cells, outside the volume, rounding at integers) and rotated ones, models whose
rows are no whole dwords or start at any byte, instances that have not moved,
more dirty regions than one launch takes, both mips in one pass, and the empty
volume's march grid."""
import math

import numpy as np
import pytest
import torch

from helpers import IDENTITY, assert_bitwise

pytestmark = pytest.mark.gpu


def _mat(scale=(1.0, 1.0, 1.0), at=(0.0, 0.0, 0.0), turn=0.0, tilt=0.0):
    c, s, ct, st = math.cos(turn), math.sin(turn), math.cos(tilt), math.sin(tilt)
    r = np.array([[c, 0, s], [0, 1, 0], [-s, 0, c]]) @ np.array([[1, 0, 0], [0, ct, -st], [0, st, ct]])
    m = np.eye(4)
    m[:3, :3] = r * np.array(scale)
    m[:3, 3] = at
    return np.ascontiguousarray(m.T.reshape(16), np.float32)


MATS = {
    "identity": _mat(), "cells": _mat(at=(0.8, 1.6, 0.4)), "shifted": _mat(at=(0.5, 0.3, 0.7)),
    "fraction": _mat(at=(0.537, 1.2999, 0.8001)), "negative": _mat(at=(-0.7, -1.3, -0.2)),
    "far faces": _mat(at=(3.1, 2.2, 2.9)), "outside": _mat(at=(100.0, 0.0, 0.0)), "huge": _mat(at=(3e9, 0.0, 0.0)),
    "flipped": _mat(scale=(-1.0, 1.0, -1.0), at=(3.0, 0.2, 3.0)), "double": _mat(scale=(2.0, 2.0, 2.0), at=(0.3, 0.0, 0.1)),
    "half": _mat(scale=(0.5, 0.5, 0.5), at=(0.25, 0.1, 0.0)), "stretched": _mat(scale=(1.0, 3.0, 1.0)),
    "quarter turn": _mat(turn=math.pi / 2, at=(1.0, 0.5, 3.0)), "turned": _mat(turn=0.7, tilt=0.2, at=(1.0, 0.6, 1.2)),
}


def _models(dims, seed, shift=0):
    """The same voxels in host memory and on the device, `shift` bytes off alignment."""
    sx, sy, sz = dims
    h = np.random.default_rng(seed).integers(0, 256, (sz, sy, sx)).astype(np.uint8)
    h[np.random.default_rng(seed + 1).random(h.shape) < 0.4] = 0
    dev = torch.zeros(h.size + 16, dtype=torch.uint8, device="cuda")
    dev[shift:shift + h.size] = torch.from_numpy(h.reshape(-1)).cuda()
    return h, dev


def _both(ctx, oracle, vdims, items, thr=16, prefill=True):
    """items: (host model, device tensor, shift, prev, cur, pivot, flags)."""
    from voxelengine_amd import api
    occ = api.Volume(ctx, *vdims, nlevels=3)
    occ.clear()
    ref = np.zeros(vdims[::-1], np.uint8)
    if prefill:
        ref[:] = np.random.default_rng(5).integers(0, 256, ref.shape)
        occ.upload_region(ref, [(0, 0, 0, *vdims)])
    gi = [api.make_instance(d.data_ptr() + s, h.shape[::-1], p, c, pv, fl) for h, d, s, p, c, pv, fl in items]
    regs = occ.rebuild(gi, threshold=thr)
    rr = oracle.rebuild(ref, [oracle.make_instance(h, p, c, pv, fl) for h, d, s, p, c, pv, fl in items], thr)
    assert [tuple(r) for r in rr.tolist()] == [tuple(r) for r in regs]
    assert_bitwise(occ.download(), ref, "occupancy")
    return occ, regs


@pytest.mark.parametrize("dims,shift", [((20, 24, 28), 0), ((20, 24, 28), 1), ((1, 1, 1), 0), ((3, 5, 7), 0), ((66, 9, 4), 2)])
@pytest.mark.parametrize("prev,cur", [("identity", "identity"), ("shifted", "shifted"), ("cells", "shifted"), ("fraction", "negative"),
                                      ("far faces", "outside"), ("huge", "far faces"), ("flipped", "double"),
                                      ("half", "stretched"), ("quarter turn", "turned"), ("turned", "fraction")])
def test_footprints(ctx, oracle, dims, shift, prev, cur):
    h, d = _models(dims, 3, shift)
    _both(ctx, oracle, (23, 18, 21), [(h, d, shift, MATS[prev], MATS[cur], (0.0, 0.0, 0.0), 1)])


@pytest.mark.parametrize("thr", [0, 1, 16, 255, 256])
def test_thresholds(ctx, oracle, thr):
    h, d = _models((12, 8, 16), 4)
    for a, b in (("identity", "cells"), ("turned", "shifted"), ("shifted", "shifted")):
        _both(ctx, oracle, (23, 18, 21), [(h, d, 0, MATS[a], MATS[b], (0.0, 0.0, 0.0), 1)], thr=thr)


def test_unmoved_instances_among_others(ctx, oracle):
    """Overlapping instances in order: one that has not moved re-sets what it covers."""
    ms = [_models((16, 12, 20), k) for k in range(4)]
    order = ["shifted", "turned", "cells", "identity", "fraction", "shifted"]
    items = [(*ms[k % 4], 0, MATS[a], MATS[a if k % 2 == 0 else "turned"], (0.1 * k, 0.0, 0.2), 1) for k, a in enumerate(order)]
    items.insert(3, (*ms[1], 0, MATS["cells"], MATS["cells"], (0.0, 0.0, 0.0), 2))
    _both(ctx, oracle, (23, 18, 21), items)


def test_levels_of_many_regions(ctx, oracle):
    rng = np.random.default_rng(9)
    h, d = _models((4, 4, 4), 8)
    items = []
    for _ in range(300):
        at = rng.uniform(0.0, 20.0, 3)
        items.append((h, d, 0, _mat(at=at), _mat(at=at + rng.uniform(-0.5, 0.5, 3)), (0.0, 0.0, 0.0), 1))
    occ, regs = _both(ctx, oracle, (110, 108, 107), items, prefill=False)
    assert len(regs) > 256
    occ.build_levels(regs)
    part = [occ.download_level(l) for l in (1, 2, 3)]
    occ.build_levels()
    for l in (1, 2, 3):
        assert_bitwise(part[l - 1], occ.download_level(l), f"level {l}")


@pytest.mark.parametrize("dims", [(4, 4, 4), (8, 4, 12), (68, 20, 36), (132, 8, 4)])
def test_mips(ctx, oracle, dims):
    from voxelengine_amd import api
    h, _ = _models(dims, 12)
    h[np.random.default_rng(2).random(h.shape) < 0.7] = 0
    m = api.Model(ctx, *dims)
    m.upload(h)
    m.build_mips()
    for k, ref in enumerate(oracle.build_mips(h)):
        assert_bitwise(m.download(k), ref, f"mip {k}")


@pytest.mark.parametrize("vdims", [(1, 1, 1), (23, 18, 21), (64, 32, 16)])
def test_cleared_volume_traces_as_empty(ctx, oracle, vdims):
    """clear() leaves cells, levels and march grid as a new volume has them."""
    from voxelengine_amd import api, configs, views
    occ = api.Volume(ctx, *vdims, nlevels=3)
    occ.upload_region(np.full(vdims[::-1], 255, np.uint8), [(0, 0, 0, *vdims)])
    occ.build_levels()
    occ.clear()
    assert not occ.download().any()
    assert not any(occ.download_level(l).any() for l in (1, 2, 3))
    m = api.Model(ctx, 48, 40, 44)
    m.generate(seed=3, terrain_fill=0.3)
    m.build_mips()
    vd = views.scene_view(m.dims, 40, 30)
    g = api.GBuffer(40, 30)
    api.primary(ctx, m, vd, g)
    pal = torch.from_numpy(configs.make_palette()).cuda()
    out = []
    for v in (occ, api.Volume(ctx, *vdims, nlevels=3)):
        vis = api.Visibility(40, 30, fetches=True)
        api.trace(ctx, v, vd, g, pal, configs.trace_params(n_ao=4), vis)
        out.append([t.cpu().numpy() for t in (vis.shadow, vis.ao, vis.spec, vis.fetches)])
    for a, b in zip(*out):
        assert_bitwise(a, b, "cleared against new")
