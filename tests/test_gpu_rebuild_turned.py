"""Turned operations of the rebuild, whose voxels meet in a window of cells per 16^3 of the model, against the oracle:
models below, at and past a block's 16, windows inside, across and outside the volume, transforms that scale past what a
window holds, flip, flatten, or are not finite."""
import numpy as np
import pytest

from test_gpu_rebuild_kernels import _both, _mat, _models

pytestmark = pytest.mark.gpu


def _nan():
    m = _mat(turn=0.4, at=(1.0, 1.0, 1.0))
    m[5] = np.nan
    return m


TURNED = {
    "inside": _mat(turn=0.6, tilt=0.3, at=(1.5, 1.0, 2.0)), "corner": _mat(turn=2.1, tilt=-0.4, at=(0.2, 0.1, 0.3)),
    "far corner": _mat(turn=-0.9, tilt=0.5, at=(6.0, 5.0, 6.5)), "outside": _mat(turn=0.5, at=(-50.0, 3.0, 2.0)),
    "far away": _mat(turn=0.5, tilt=0.1, at=(3e9, 0.0, 0.0)), "scaled": _mat(scale=(6.0, 7.0, 5.0), turn=0.5, tilt=0.2, at=(0.5, 0.4, 1.0)),
    "small": _mat(scale=(0.3, 0.2, 0.3), turn=0.5, tilt=0.2, at=(2.0, 2.0, 2.0)),
    "flat": _mat(scale=(1.0, 0.0, 1.0), turn=0.7, tilt=0.3, at=(2.0, 2.0, 2.0)),
    "mirrored": _mat(scale=(-1.0, 1.0, -1.0), turn=0.7, tilt=0.3, at=(4.0, 1.0, 4.0)), "not finite": _nan(),
}


@pytest.mark.parametrize("dims,shift", [((5, 3, 7), 0), ((16, 16, 16), 0), ((17, 33, 20), 1), ((40, 15, 48), 0)])
@pytest.mark.parametrize("prev,cur", [("inside", "corner"), ("corner", "far corner"), ("outside", "inside"), ("far away", "mirrored"),
                                      ("scaled", "small"), ("mirrored", "scaled"), ("flat", "inside"), ("inside", "not finite"),
                                      ("not finite", "flat")])
def test_turned_footprints(ctx, oracle, dims, shift, prev, cur):
    h, d = _models(dims, 4, shift)
    _both(ctx, oracle, (40, 33, 37), [(h, d, shift, TURNED[prev], TURNED[cur], (0.2, 0.1, 0.0), 1)])


def test_many_turned_objects(ctx, oracle):
    items = []
    for k in range(9):
        h, d = _models((12 + 5 * k, 20, 9 + 4 * k), 10 + k)
        a = _mat(turn=0.4 * k, tilt=0.1 * k - 0.3, at=(0.5 * k, 0.8, 0.4 * k))
        b = _mat(turn=0.4 * k + 0.1, tilt=0.1 * k - 0.3, at=(0.5 * k + 0.3, 0.8, 0.4 * k + 0.1))
        items.append((h, d, 0, a, b, (0.3, 0.0, 0.2), 1))
    _both(ctx, oracle, (60, 40, 60), items)
