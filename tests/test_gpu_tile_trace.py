"""The trace of small launches (k_trace_tile: waves of a block take a tile's
rays, marches read ahead) bit for bit against the oracle and against the
launch with fetch counts, which takes the other kernels: ragged views, ray
counts below, at and above the waves of a block, every mix of marchers, rays
outside the fast path, volumes that rays leave through every face and start
outside of, and both sides of the size at which a launch changes kernels."""
import numpy as np
import pytest
import torch

from helpers import IDENTITY, assert_bitwise

pytestmark = pytest.mark.gpu

DDA, SPARSE, SUPER = 0, 1, 2


@pytest.fixture(scope="module", params=[(45, 37, 43), (48, 40, 44), (17, 50, 9)])
def scene(request, ctx, oracle):
    from voxelengine_amd import api
    m = api.Model(ctx, 96, 80, 88)
    m.generate(seed=11, terrain_fill=0.25, nboxes=30, box_min=2, box_max=12)
    m.build_mips()
    occ = api.Volume(ctx, *request.param, nlevels=1)
    occ.clear()
    occ.rebuild([api.make_instance(m.mip_ptr(0), m.dims, IDENTITY, IDENTITY)])
    occ.build_levels()
    return m, occ, occ.download()


def _check(ctx, oracle, scene, w, h, params, variant=0):
    from voxelengine_amd import api, configs, views
    m, occ, occ_h = scene
    vd = views.scene_view(m.dims, w, h, frame=variant, variant=variant)
    g = api.GBuffer(w, h)
    api.primary(ctx, m, vd, g)
    pal = configs.make_palette()
    pal_d = torch.from_numpy(pal).cuda()
    ref = oracle.trace(occ_h, vd, params, g.pos.cpu().numpy(), g.normal.cpu().numpy(), g.material.cpu().numpy(), pal)
    for fetches in (False, True):
        vis = api.Visibility(w, h, fetches=fetches)
        for t in (vis.shadow, vis.ao, vis.spec):
            t.fill_(7)
        api.trace(ctx, occ, vd, g, pal_d, params, vis)
        for name, a, b in zip(("shadow", "ao", "spec"), (vis.shadow, vis.ao, vis.spec), ref):
            assert_bitwise(a.cpu().numpy(), b, f"{w}x{h} {name} fetches={fetches}")


@pytest.mark.parametrize("w,h", [(1, 1), (7, 9), (61, 43)])
@pytest.mark.parametrize("rays", [(0, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 4, 1), (1, 15, 0), (1, 16, 1), (1, 64, 1)])
@pytest.mark.parametrize("march", [(DDA, DDA, DDA), (SPARSE, SUPER, SPARSE), (SPARSE, DDA, SUPER)])
def test_small_views(ctx, oracle, scene, w, h, rays, march):
    from voxelengine_amd import configs
    p = configs.trace_params(n_shadow=rays[0], n_ao=rays[1], n_spec=rays[2], ao_maxt=30.0, march="dda")
    p["shadow_march"], p["ao_march"], p["spec_march"] = march
    _check(ctx, oracle, scene, w, h, p, variant=1)


@pytest.mark.parametrize("light", [(0.0, 1.0, 0.0), (1.0, 0.0, 0.0), (0.0, -1.0, 1e-38)])
def test_rays_outside_the_fast_path(ctx, oracle, scene, light):
    from voxelengine_amd import configs
    p = configs.trace_params(n_ao=2, ao_maxt=30.0, march="dda")
    p["light_dir"], p["jitter_shadow"] = light, 0
    _check(ctx, oracle, scene, 40, 33, p)


# 8x8 tiles x rays around 16384 waves (DDA), tiles around 4096 (sparse)
@pytest.mark.parametrize("w,h,n_ao,march", [(511, 256, 7, "dda"), (513, 256, 7, "dda"), (511, 512, 1, "reference"),
                                            (513, 512, 1, "reference")])
def test_both_sides_of_the_kernel_rule(ctx, oracle, scene, w, h, n_ao, march):
    from voxelengine_amd import configs
    _check(ctx, oracle, scene, w, h, configs.trace_params(n_ao=n_ao, n_spec=0, ao_maxt=16.0, march=march), variant=2)
