"""The primary march's two kernels (a launch whose waves are all resident, and a larger one) on either side of the line
between them, against the oracle: voxels in a box seen from outside and inside, the 512-step limit, glass."""
import numpy as np
import pytest

from test_gpu_primary_march import _check, _view

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(1024, 512), (1025, 512)])     # 2048 and 2080 tiles
def test_either_side_of_the_line(ctx, oracle, size):
    rng = np.random.default_rng(9)
    h = rng.integers(0, 64, (28, 20, 36)).astype(np.uint8)
    h[rng.random(h.shape) < 0.85] = 0
    for k, at in enumerate([(-40.0, 18.0, 9.0), (17.3, 60.0, 14.2), (18.2, 9.9, 13.7)]):
        _check(ctx, oracle, h, _view(at, (18.0, 10.0, 14.0), *size, frame=k), f"{size} from {at}")
    wall = np.zeros((8, 8, 640), np.uint8)
    wall[1, 1, 4] = 200
    wall[:, :, 530] = 77
    _check(ctx, oracle, wall, _view((-20.0, 0.5, 0.5), (640.0, 0.6, 0.7), *size), f"{size} step limit")
