"""The primary pass's march bit for bit against the oracle where its two forms
and its limits meet: rays along an axis (a zero component: the general form),
starts outside, on the faces of and inside the box, passes that leave a level
through every face, the 512-step limit with and without a wall past it, glass,
coarse hits far away, and models from one coarse cell up."""
import numpy as np
import pytest

from helpers import assert_bitwise

pytestmark = pytest.mark.gpu


def _check(ctx, oracle, h, vd, what):
    from voxelengine_amd import api
    sz, sy, sx = h.shape
    m = api.Model(ctx, sx, sy, sz)
    m.upload(h)
    m.build_mips()
    w, hh = vd["width"], vd["height"]
    g = api.GBuffer(w, hh)
    api.primary(ctx, m, vd, g)
    mips = oracle.build_mips(h)
    pos, nrm, mat = oracle.primary(mips, vd)
    assert_bitwise(g.material.cpu().numpy(), mat, f"{what} material")
    assert_bitwise(g.pos.cpu().numpy(), pos, f"{what} position")
    assert_bitwise(g.normal.cpu().numpy(), nrm, f"{what} normal")
    # the instance pass marches the same model from its own rays
    ext = api.GBufferExt(w, hh)
    api.primary_instances(ctx, [api.make_vox_cmd(m, api.IDENTITY, volume_rid=1, palette=3)], vd, g, ext)
    ref = oracle.primary_instances([dict(mips=mips, world=api.IDENTITY, rid=1, palette=3)], vd)
    for name, a in (("pos", g.pos), ("nrm", g.normal), ("mat", g.material), ("depth", ext.depth)):
        assert_bitwise(a.cpu().numpy(), ref[name], f"{what} instance {name}")
    return mat


def _view(pos, at, w, h, frame=0):
    from voxelengine_amd import views
    return views.make_view(np.asarray(pos, np.float64) / 10.0, np.asarray(at, np.float64) / 10.0, w, h, frame=frame)


@pytest.mark.parametrize("dims", [(4, 4, 4), (8, 4, 12), (36, 20, 28)])
def test_every_side_of_the_box(ctx, oracle, dims):
    rng = np.random.default_rng(3)
    h = rng.integers(0, 256, dims[::-1]).astype(np.uint8)
    h[rng.random(h.shape) < 0.9] = 0
    c = np.array(dims) / 2.0
    for k, off in enumerate([(90, 1, 2), (-90, 3, 1), (2, 80, 3), (1, -80, 2), (2, 1, 90), (3, 2, -90), (40, 35, 30), (0.3, 0.2, 0.1)]):
        _check(ctx, oracle, h, _view(c + off, c, 47, 33, frame=k), f"{dims} from {off}")
    # on a face and on a corner of the box, and well outside the range of the fast form
    _check(ctx, oracle, h, _view((0.0, 1.0, 1.0), c + (9.0, 0.3, 0.1), 31, 21), "on a face")
    _check(ctx, oracle, h, _view((0.0, 0.0, 0.0), c, 31, 21), "on a corner")
    _check(ctx, oracle, h, _view(c + (6e6, 3.0, 5.0), c, 15, 9), "far away")


@pytest.mark.parametrize("axis", [0, 2])
@pytest.mark.parametrize("sign", [1, -1])
def test_rays_along_an_axis(ctx, oracle, axis, sign):
    """An odd view straight along an axis: its middle row and column hold zero components."""
    rng = np.random.default_rng(4)
    h = rng.integers(0, 256, (24, 20, 28)).astype(np.uint8)
    h[rng.random(h.shape) < 0.95] = 0
    c = np.array([14.0, 10.0, 12.0])
    off = np.zeros(3)
    off[axis] = 60.0 * sign
    for at in (c, c + 0.5, np.floor(c) + 0.25):
        _check(ctx, oracle, h, _view(at + off, at, 33, 25), f"along {axis}")


@pytest.mark.parametrize("wall", [300, 500, 530, 620])
def test_step_limit(ctx, oracle, wall):
    """Rays that a coarse cell stops but no voxel does march on at mip 0, 512 steps at most."""
    h = np.zeros((8, 8, 640), np.uint8)
    h[1, 1, 4] = 200            # stops mips 2 and 1 at the start of the model
    h[:, :, wall] = 77
    for y in (0.5, 2.5, 3.5, 5.0):
        mat = _check(ctx, oracle, h, _view((-20.0, y, y), (640.0, 0.6, 0.7), 41, 29), f"wall {wall} from {y}")
        # the middle ray enters the voxel's cells of mips 2 and 1 and misses the voxel
        if y == 0.5:
            assert mat.reshape(29, 41)[14, 20] == (77 if wall < 512 else 0)


def test_glass_and_coarse_hits(ctx, oracle):
    rng = np.random.default_rng(5)
    h = rng.integers(0, 40, (64, 64, 64)).astype(np.uint8)
    h[rng.random(h.shape) < 0.8] = 0
    for frame in (0, 1, 2):
        _check(ctx, oracle, h, _view((150.0, 90.0, 120.0), (32.0, 30.0, 31.0), 64, 48, frame=frame), f"glass frame {frame}")
    # past 1000 and 2000 voxels a hit of mip 1 and of mip 2 is accepted
    for dist in (900.0, 1500.0, 2600.0):
        _check(ctx, oracle, h, _view((32.0 + dist, 40.0, 35.0), (32.0, 32.0, 32.0), 64, 48), f"from {dist}")
