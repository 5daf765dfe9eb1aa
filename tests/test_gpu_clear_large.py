"""vx_volume_clear on a volume whose arrays together take more blocks than one
launch may hold: voxels in the first and the last of its slices are set by a
rebuild, found by all marchers, and gone from the cells, the march grid and the
texel words after the clear."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_clear_of_a_volume_beyond_one_launch(ctx):
    from voxelengine_amd import _lib, api
    dims = (4096, 4096, 1400)
    need = 53 << 30          # cells, march grid (23.6 GB each), texel words, levels
    if torch.cuda.mem_get_info()[0] < need + (8 << 30):
        pytest.skip("device memory")
    model = api.Model(ctx, 16, 16, 16)
    model.upload(np.full((16, 16, 16), 40, np.uint8))
    occ = api.Volume(ctx, *dims, nlevels=3)
    try:
        # objects of 16^3 voxels (a voxel is 0.1 units) in the corners and between
        at = [(0, 0, 0), (8176, 8176, 2784), (4096, 4096, 1400), (8176, 0, 2700), (0, 8176, 96)]
        inst = []
        for x, y, z in at:
            m = np.eye(4, dtype=np.float32)
            m[3, :3] = np.array([x, y, z], np.float64) * 0.1 + 0.01
            inst.append(api.make_instance(model.mip_ptr(0), model.dims, m.reshape(16), m.reshape(16)))
        # along x from the inner side, 6 voxels off (the sparse marches' fine phase, which
        # reads the march grid) and 60 off (their coarse phase, which reads the texel words)
        rays = []
        for x, y, z in at:
            for off in (6, 60):
                s = -1.0 if x > 4000 else 1.0
                o = x - off if s < 0 else x + 15 + off
                rays.append([o + 0.3, y + 8.4, z + 8.4, -s, 1e-4, 1e-4, 150.0])
        rays = torch.tensor(rays, dtype=torch.float32, device="cuda")

        def hits():
            return [api.trace_rays(ctx, occ, rays, m)["hit"] for m in
                    (_lib.MARCH_DDA, _lib.MARCH_SPARSE, _lib.MARCH_SUPERSPARSE)]

        for _ in range(2):
            occ.rebuild(inst)
            occ.build_levels()
            assert all(h.all() for h in hits())
            occ.clear()
            assert not any(h.any() for h in hits())
            for level in (1, 2, 3):
                assert not occ.download_level(level).any()
    finally:
        occ.close()
        model.close()
