"""The work that a program has this framework do, as cases that can be timed.

Each case is one pass through the public entry points (voxelengine_amd.api over the C ABI) with its
scene, view and buffers resident on the GPU, as a renderer keeps them. listed() names fixed sizes,
draw() gives others of the same ranges, prepare() makes a case's inputs from a seed, run() is the pass,
work() what it cannot do without and exact() its result in 64 bits where it has one (a traversal has
none: which voxel a ray meets is defined by its fp32 steps).
"""
from __future__ import annotations

import math

import numpy as np
import torch

from voxelengine_amd import api, configs, views


def listed():
    return [
        # The smallest call: a probe or thumbnail view of a small scene, all launches and latency.
        dict(name="trace_small", kind="trace", nx=64, ny=64, nz=64, fill=0.3, boxes=20, width=61, height=43,
             n_shadow=1, n_ao=4, n_spec=1, ao_maxt=16.0, march="dda"),
        # The shipped marchers (Sparse shadow, SuperSparse AO) at a preview size.
        dict(name="trace_reference", kind="trace", nx=256, ny=256, nz=256, fill=0.3, boxes=0, width=640, height=360,
             n_shadow=1, n_ao=4, n_spec=0, ao_maxt=16.0, march="reference"),
        # The headline frame: exact marching of every ray class at 1080p.
        dict(name="trace_1080p", kind="trace", nx=512, ny=512, nz=512, fill=0.3, boxes=2000, width=1920, height=1080,
             n_shadow=1, n_ao=16, n_spec=1, ao_maxt=32.0, march="dda"),
        # Many scenes and views of uneven size in one captured launch (an offline or training renderer).
        dict(name="batch_uneven", kind="batch", scenes=64, layout=7, max_edge=512, max_width=1920, max_height=1080, n_ao=8,
             ao_maxt=32.0),
        # The largest: four 4K views of a city, forward and the adjoint accumulated over the views.
        dict(name="city_views", kind="city", edge=1024, boxes=20000, views=4, width=3840, height=2160, n_ao=32, n_spec=1),
        # The geometry pass of a world model with its depth attachment and screen-space occlusion.
        dict(name="primary_1080p", kind="primary", nx=512, ny=512, nz=512, fill=0.3, boxes=2000, width=1920, height=1080),
        # A game frame with moving objects: volume update, draws of every object, shipped marchers.
        dict(name="moving_frame", kind="moving", draws=67, edge=40, nx=1048, ny=376, nz=1048, width=1920, height=1080),
        # The first frame after a world was loaded or edited: mips, occupancy, coarse levels, a preview view.
        dict(name="world_load", kind="world", nx=512, ny=512, nz=512, fill=0.3, boxes=2000, width=640, height=360),
        # The light passes: sun and ambient, then every point and spot light with its shadow ray.
        dict(name="lights_1080p", kind="lights", nx=512, ny=512, nz=512, fill=0.3, boxes=2000, width=1920, height=1080,
             points=64, spots=64),
        # The reflection pass with the shipped marcher.
        dict(name="reflection_1080p", kind="reflection", nx=512, ny=512, nz=512, fill=0.3, boxes=2000, width=1920,
             height=1080, sky=0),
        # Temporal accumulation under a moving camera.
        dict(name="taa_1080p", kind="taa", nx=512, ny=512, nz=512, fill=0.3, boxes=2000, width=1920, height=1080,
             move=0.4),
        # One step of fitting materials and light to an image: forward, loss gradient, adjoint.
        dict(name="shade_720p", kind="shade", nx=256, ny=256, nz=256, fill=0.3, width=1280, height=720, n_ao=8, ssao=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _edge(rng, lo=64, hi=512):
    return 4 * max(1, _log(rng, lo, hi) // 4)   # models round their edges up to multiples of 4


def draw(rng):
    kind = rng.choice(["trace", "trace", "batch", "city", "primary", "moving", "world", "lights", "reflection", "taa", "shade"])
    scene = dict(nx=_edge(rng), ny=_edge(rng), nz=_edge(rng), fill=round(rng.uniform(0.05, 0.4), 3), boxes=_log(rng, 1, 2000) - 1)
    view = dict(width=_log(rng, 48, 1920), height=_log(rng, 32, 1080))
    if kind == "trace":
        march = rng.choice(["dda", "reference"])
        return dict(kind=kind, **scene, **view, n_shadow=1, n_ao=rng.choice([1, 2, 4, 8, 16]), n_spec=rng.choice([0, 1]),
                    ao_maxt=rng.choice([16.0, 32.0, 128.0] if march == "reference" else [16.0, 32.0]), march=march)
    if kind == "batch":
        return dict(kind=kind, scenes=_log(rng, 2, 64), layout=rng.randrange(1000), max_edge=8 * rng.randint(12, 64),
                    max_width=rng.randint(300, 1920), max_height=rng.randint(300, 1080), n_ao=rng.choice([1, 4, 8]), ao_maxt=rng.choice([16.0, 32.0]))
    if kind == "city":
        return dict(kind=kind, edge=8 * rng.randint(24, 96), boxes=_log(rng, 200, 10000), views=rng.randint(1, 4),
                    width=_log(rng, 320, 2560), height=_log(rng, 200, 1440), n_ao=rng.choice([4, 8, 16]), n_spec=rng.choice([0, 1]))
    if kind == "moving":
        return dict(kind=kind, draws=_log(rng, 1, 200), edge=4 * rng.randint(2, 16), nx=_edge(rng, 128, 1048),
                    ny=_edge(rng, 64, 376), nz=_edge(rng, 128, 1048), **view)
    if kind == "lights":
        return dict(kind=kind, **scene, **view, points=rng.randint(0, 64), spots=rng.randint(1, 64))
    if kind == "reflection":
        return dict(kind=kind, **scene, **view, sky=rng.choice([0, 0, 64, 333]))
    if kind == "taa":
        return dict(kind=kind, **scene, **view, move=round(rng.uniform(0.0, 1.0), 3))
    if kind == "shade":
        scene.pop("boxes")
        return dict(kind=kind, **scene, **view, n_ao=rng.choice([1, 4, 8]), ssao=rng.choice([False, True]))
    return dict(kind=kind, **scene, **view)


# ---------------------------------------------------------------- inputs

class State:
    """What a program holds between passes of one case."""


def _palette(seed):
    return torch.from_numpy(configs.make_palette(seed=seed)).cuda()


def _scene(ctx, dims, seed, fill, boxes, box=(2, 32), grounded=False, levels=2):
    """A generated world model and its rebuilt occupancy volume."""
    m = api.Model(ctx, *dims)
    m.generate(seed=seed, terrain_fill=fill, nboxes=boxes, box_min=box[0], box_max=box[1], grounded=grounded)
    m.build_mips()
    d = m.dims
    occ = api.Volume(ctx, d[0] // 2, d[1] // 2, d[2] // 2, nlevels=levels)
    inst = [api.make_instance(m.mip_ptr(0), d, api.IDENTITY, api.IDENTITY)]
    occ.rebuild(inst)
    occ.build_levels()
    return m, occ, inst


def _world_case(case, seed):
    """Context, scene, view and G-buffer of a case over one generated world."""
    s = State()
    s.ctx = api.Context(0)
    s.model, s.occ, s.inst = _scene(s.ctx, (case["nx"], case["ny"], case["nz"]), seed, case["fill"], case.get("boxes", 0))
    s.vd = views.scene_view(s.model.dims, case["width"], case["height"], frame=seed % 64, variant=seed)
    s.g = api.GBuffer(case["width"], case["height"])
    api.primary(s.ctx, s.model, s.vd, s.g)
    s.pal = _palette(seed)
    s.vis = api.Visibility(case["width"], case["height"])
    return s


def _lights(case, seed, dims):
    """Point and spot lights over the scene, the shipped per-type limit of 64 at most."""
    rng = np.random.default_rng(seed)
    ext = np.array(dims, np.float64) * 0.1
    n = case["points"] + case["spots"]
    L = np.zeros(n, api.LIGHT_DTYPE)
    L["type"][case["points"]:] = 1
    L["position"] = rng.uniform([0.0, 0.3, 0.0], [1.0, 0.7, 1.0], (n, 3)) * ext
    L["range"] = rng.uniform(0.1, 0.3, n) * ext.max()
    L["color"] = rng.uniform(0.2, 4.0, (n, 3))
    L["attenuation"] = rng.uniform(0.5, 2.0, n)
    d = rng.normal(size=(n, 3))
    d[:, 1] = -np.abs(d[:, 1])
    L["direction"] = d / np.linalg.norm(d, axis=1, keepdims=True)
    L["angle"] = rng.uniform(0.2, 0.9, n)
    L["angle_attenuation"] = rng.uniform(0.5, 3.0, n)
    return L


def _pose(angle, tilt, t):
    """Column-major world matrix: a turn about y, a tilt about x, a translation."""
    c, s, ct, st = math.cos(angle), math.sin(angle), math.cos(tilt), math.sin(tilt)
    r = np.array([[c, 0, s], [0, 1, 0], [-s, 0, c]]) @ np.array([[1, 0, 0], [0, ct, -st], [0, st, ct]])
    m = np.eye(4)
    m[:3, :3] = r
    m[:3, 3] = t
    return np.ascontiguousarray(m.T.reshape(16), np.float32)


def _moving(case, seed):
    s = State()
    s.ctx = api.Context(0)
    rng = np.random.default_rng(seed)
    # object models of uneven size (shared by the draws, as props are) on a ground plate
    s.models = []
    for k in range(min(case["draws"], 24)):
        dims = [4 * int(rng.integers(max(1, case["edge"] // 8), case["edge"] // 2 + 1)) for _ in range(3)]
        m = api.Model(s.ctx, *dims)
        m.generate(seed=seed + k, terrain_fill=0.55, nboxes=6, box_min=2, box_max=max(2, min(dims) // 2))
        m.build_mips()
        s.models.append(m)
    ground = api.Model(s.ctx, case["nx"], 8, case["nz"])
    ground.generate(seed=seed + 99, terrain_fill=0.5)
    ground.build_mips()
    ext = np.array([case["nx"], case["ny"], case["nz"]]) * 0.1
    s.instances, s.cmds = [], [api.make_vox_cmd(ground, api.IDENTITY, volume_rid=1, palette=1)]
    s.occ = api.Volume(s.ctx, case["nx"] // 2, case["ny"] // 2, case["nz"] // 2, nlevels=2)
    placed = [api.make_instance(ground.mip_ptr(0), ground.dims, api.IDENTITY, api.IDENTITY)]
    for k in range(case["draws"]):
        m = s.models[k % len(s.models)]
        # a third of the objects stand upright along the axes, the others are turned and tilted
        turn, tilt = (0.0, 0.0) if k % 3 == 0 else (rng.uniform(0, 2 * math.pi), rng.uniform(-0.3, 0.3))
        at = rng.uniform([0.1, 0.03, 0.1], [0.9, 0.25, 0.9]) * ext
        prev = _pose(turn, tilt, at)
        cur = _pose(turn if k % 3 == 0 else turn + rng.uniform(-0.1, 0.1), tilt, at + rng.uniform(-0.5, 0.5, 3))
        pivot = np.array([m.dims[0] * 0.05, 0.0, m.dims[2] * 0.05])
        placed.append(api.make_instance(m.mip_ptr(0), m.dims, prev, prev, pivot))
        s.instances.append(api.make_instance(m.mip_ptr(0), m.dims, prev, cur, pivot))
        shift = np.eye(4, dtype=np.float64)
        shift[3, :3] = -pivot
        s.cmds.append(api.make_vox_cmd(m, (shift @ cur.reshape(4, 4)).reshape(16), (shift @ prev.reshape(4, 4)).reshape(16),
                                       volume_rid=k + 2, palette=k % 7))
    s.models.append(ground)
    s.occ.rebuild(placed)
    s.occ.build_levels()
    s.vd = views.make_view(ext * [0.08, 0.42, 0.06], ext * [0.4, 0.0, 0.4], case["width"], case["height"], frame=seed % 64)
    s.g, s.ext = api.GBuffer(case["width"], case["height"]), api.GBufferExt(case["width"], case["height"])
    s.pal = _palette(seed)
    s.vis = api.Visibility(case["width"], case["height"])
    # the shipped settings: one Sparse shadow ray, one SuperSparse AO ray to 128
    s.params = configs.trace_params(n_shadow=1, n_ao=1, ao_maxt=128.0, n_spec=0, march="reference", seed=seed)
    return s


def _batch_items(s, items, npx):
    """Visibility buffers of the items as slices of one allocation per channel."""
    s.shadow = torch.zeros(npx, dtype=torch.uint8, device="cuda")
    s.ao = torch.zeros(npx, dtype=torch.float32, device="cuda")
    s.spec = torch.zeros(npx, dtype=torch.float32, device="cuda")
    out, at = [], 0
    for occ, vd, g in items:
        n = vd["width"] * vd["height"]
        vis = api.Visibility(1, 1)
        vis.shadow, vis.ao, vis.spec = s.shadow[at:at + n], s.ao[at:at + n], s.spec[at:at + n]
        out.append((occ, vd, g, vis))
        at += n
    return out


def _batch(case, seed):
    s = State()
    s.ctx = api.Context(0)
    rng = np.random.default_rng(case["layout"])     # the sizes are the case's, the contents the seed's
    items, npx = [], 0
    s.models = []
    for k in range(case["scenes"]):
        dims = tuple(int(8 * rng.integers(8, case["max_edge"] // 8 + 1)) for _ in range(3))
        m, occ, _ = _scene(s.ctx, dims, seed + 31 * k, float(rng.uniform(0.05, 0.40)), int(rng.integers(0, 200)), box=(2, 16))
        w, h = int(rng.integers(256, case["max_width"] + 1)), int(rng.integers(256, case["max_height"] + 1))
        vd = views.scene_view(dims, w, h, variant=k)
        g = api.GBuffer(w, h)
        api.primary(s.ctx, m, vd, g)
        s.models.append(m)
        items.append((occ, vd, g))
        npx += w * h
    s.items = _batch_items(s, items, npx)
    s.pal = _palette(seed)
    s.batch = api.Batch(s.ctx, s.items, s.pal, configs.trace_params(n_shadow=1, n_ao=case["n_ao"], ao_maxt=case["ao_maxt"],
                                                                    n_spec=0, march="dda", seed=seed))
    return s


def _city(case, seed):
    s = State()
    s.ctx = api.Context(0)
    e, w, h = case["edge"], case["width"], case["height"]
    s.model, occ, _ = _scene(s.ctx, (e, e, e), seed, 0.0, case["boxes"], box=(8, 56), grounded=True, levels=3)
    items = []
    for k in range(case["views"]):
        vd = views.city_view((e, e, e), w, h, variant=k)
        g = api.GBuffer(w, h)
        api.primary(s.ctx, s.model, vd, g)
        items.append((occ, vd, g))
    s.items = _batch_items(s, items, w * h * case["views"])
    s.pal, s.light = _palette(seed), configs.default_light()
    s.batch = api.Batch(s.ctx, s.items, s.pal, configs.trace_params(n_shadow=1, n_ao=case["n_ao"], ao_maxt=32.0,
                                                                    n_spec=case["n_spec"], march="dda", seed=seed))
    gen = torch.Generator(device="cuda").manual_seed(seed)
    s.shade = [(vd, g, vis, torch.randn((w * h, 3), generator=gen, device="cuda"), None) for _, vd, g, vis in s.items]
    s.dpal = torch.zeros((256, 6), dtype=torch.float32, device="cuda")
    s.dlight = torch.zeros(6, dtype=torch.float32, device="cuda")
    return s


def _taa(case, seed):
    s = _world_case(case, seed)
    w, h = case["width"], case["height"]
    npx = w * h
    # the camera moved since the last frame: motion of every hit pixel, as the geometry pass writes it
    nx, ny, nz = s.model.dims
    before = views.make_view(np.asarray(s.vd["cam_pos"], np.float64) + case["move"] * np.array([0.5, 0.2, -0.3]),
                             np.array([0.5 * nx, 0.15 * ny, 0.5 * nz]) / 10.0, w, h)
    pos = torch.cat([s.g.pos * 0.1, torch.ones((npx, 1), device="cuda")], 1)

    def clip(vd):
        v, p = (torch.from_numpy(vd[k].reshape(4, 4)).cuda() for k in ("view", "proj"))
        c = (pos @ v) @ p
        return c[:, :2] / c[:, 3:]
    mo = (clip(s.vd) - clip(before)) * torch.tensor([-0.5, 0.5], device="cuda")
    s.motion = torch.where((s.g.material > 0)[:, None], mo, torch.zeros_like(mo)).contiguous()
    s.depth = torch.zeros(npx, dtype=torch.float32, device="cuda")
    api.gbuf_depth(s.ctx, s.vd, s.g, s.depth, volume_rid=1)
    api.trace(s.ctx, s.occ, s.vd, s.g, s.pal, configs.trace_params(n_ao=1, n_spec=0, ao_maxt=128.0, march="reference", seed=seed),
              s.vis)
    s.rgb = torch.zeros((npx, 3), dtype=torch.float32, device="cuda")
    api.shade_forward(s.ctx, s.vd, s.g, s.vis, s.pal, configs.default_light(), s.rgb)
    # two accumulated frames are the history of the timed one
    s.last, s.out = (torch.zeros((npx, 4), dtype=torch.float32, device="cuda") for _ in range(2))
    for k in range(2):
        api.light_taa(s.ctx, s.vd, s.rgb, s.last, s.out, s.depth, s.g.normal, s.g.material, s.pal, motion=s.motion, seed=seed + k)
        s.last, s.out = s.out, s.last
    s.seed = seed
    return s


def _shade(case, seed):
    s = _world_case(case, seed)
    w, h = case["width"], case["height"]
    api.trace(s.ctx, s.occ, s.vd, s.g, s.pal, configs.trace_params(n_ao=case["n_ao"], n_spec=0, march="dda", seed=seed), s.vis)
    s.light = configs.default_light()
    s.ssao = None
    if case["ssao"]:
        depth = torch.zeros(w * h, dtype=torch.float32, device="cuda")
        s.ssao = torch.zeros(w * h, dtype=torch.float32, device="cuda")
        api.gbuf_depth(s.ctx, s.vd, s.g, depth, volume_rid=1)
        api.ssao(s.ctx, s.vd, s.g, depth, s.ssao, seed=seed)
    # the image to fit: the same frame under perturbed materials
    near = torch.from_numpy(configs.perturbed_palette(s.pal.cpu().numpy(), seed=seed + 1)).cuda()
    s.target, s.rgb = (torch.zeros((w * h, 3), dtype=torch.float32, device="cuda") for _ in range(2))
    api.shade_forward(s.ctx, s.vd, s.g, s.vis, near, s.light, s.target, ssao=s.ssao)
    s.dpal = torch.zeros((256, 6), dtype=torch.float32, device="cuda")
    s.dlight = torch.zeros(6, dtype=torch.float32, device="cuda")
    return s


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        s = _batch(case, seed)
    elif kind == "city":
        s = _city(case, seed)
    elif kind == "moving":
        s = _moving(case, seed)
    elif kind == "taa":
        s = _taa(case, seed)
    elif kind == "shade":
        s = _shade(case, seed)
    else:
        s = _world_case(case, seed)
        npx = case["width"] * case["height"]
        if kind == "trace":
            s.params = configs.trace_params(n_shadow=case["n_shadow"], n_ao=case["n_ao"], ao_maxt=case["ao_maxt"],
                                            n_spec=case["n_spec"], march=case["march"], seed=seed)
        elif kind == "world":
            s.params = configs.trace_params(n_shadow=1, n_ao=4, ao_maxt=16.0, n_spec=0, march="dda", seed=seed)
        elif kind == "primary":
            s.depth, s.ssao = (torch.zeros(npx, dtype=torch.float32, device="cuda") for _ in range(2))
        elif kind == "lights":
            s.lights = api.lights_to_device(_lights(case, seed, s.model.dims))
            api.trace(s.ctx, s.occ, s.vd, s.g, s.pal, configs.trace_params(n_ao=1, n_spec=0, ao_maxt=128.0, march="reference"),
                      s.vis)
            s.light = configs.default_light()
            s.rgb = torch.zeros((npx, 3), dtype=torch.float32, device="cuda")
        elif kind == "reflection":
            s.depth = torch.zeros(npx, dtype=torch.float32, device="cuda")
            api.gbuf_depth(s.ctx, s.vd, s.g, s.depth, volume_rid=1)
            gen = torch.Generator(device="cuda").manual_seed(seed)
            s.light = torch.rand((npx, 4), dtype=torch.float32, device="cuda", generator=gen)
            n = case["sky"]
            s.sky = torch.rand((6, n, n, 4), dtype=torch.float32, device="cuda", generator=gen) if n else None
            s.out = torch.zeros((npx, 4), dtype=torch.float32, device="cuda")
            s.t = torch.zeros(npx, dtype=torch.float32, device="cuda")
    s.kind, s.seed = kind, seed
    s.npoint = case.get("points", 0) + case.get("spots", 0)
    return s


# ---------------------------------------------------------------- the pass

def _gbuffer(s):
    return {"pos": s.g.pos, "normal": s.g.normal, "material": s.g.material}


def run(s):
    if s.kind == "trace":
        api.trace(s.ctx, s.occ, s.vd, s.g, s.pal, s.params, s.vis)
        return {"shadow": s.vis.shadow, "ao": s.vis.ao, "spec": s.vis.spec}
    if s.kind == "batch":
        s.batch.launch()
        return {"shadow": s.shadow, "ao": s.ao, "spec": s.spec}
    if s.kind == "city":
        s.batch.launch()
        api.shade_backward_batch(s.ctx, s.shade, s.pal, s.light, s.dpal, s.dlight)
        return {"shadow": s.shadow, "ao": s.ao, "spec": s.spec, "dpalette": s.dpal, "dlight": s.dlight}
    if s.kind == "primary":
        api.primary(s.ctx, s.model, s.vd, s.g)
        api.gbuf_depth(s.ctx, s.vd, s.g, s.depth, volume_rid=1)
        api.ssao(s.ctx, s.vd, s.g, s.depth, s.ssao, seed=s.seed)
        return dict(_gbuffer(s), depth=s.depth, ssao=s.ssao)
    if s.kind == "moving":
        regions = s.occ.rebuild(s.instances)
        s.occ.build_levels(regions)
        api.primary_instances(s.ctx, s.cmds, s.vd, s.g, s.ext)
        api.trace(s.ctx, s.occ, s.vd, s.g, s.pal, s.params, s.vis)
        return dict(_gbuffer(s), motion=s.ext.motion, depth=s.ext.depth, palette=s.ext.palette, shadow=s.vis.shadow,
                    ao=s.vis.ao, spec=s.vis.spec, regions=np.array(regions, np.int64))
    if s.kind == "world":
        s.model.build_mips()
        s.occ.clear()
        regions = s.occ.rebuild(s.inst)
        s.occ.build_levels()
        api.primary(s.ctx, s.model, s.vd, s.g)
        api.trace(s.ctx, s.occ, s.vd, s.g, s.pal, s.params, s.vis)
        return dict(_gbuffer(s), shadow=s.vis.shadow, ao=s.vis.ao, spec=s.vis.spec, regions=np.array(regions, np.int64))
    if s.kind == "lights":
        api.shade_forward(s.ctx, s.vd, s.g, s.vis, s.pal, s.light, s.rgb)
        api.light_pass(s.ctx, s.occ, s.vd, s.g, s.pal, s.lights, s.npoint, s.rgb, seed=s.seed)
        return {"rgb": s.rgb}
    if s.kind == "reflection":
        api.reflection(s.ctx, s.occ, s.vd, s.g, s.pal, s.light, s.depth, s.out, t=s.t, sky=s.sky, seed=s.seed)
        # pixels without a ray hold NaN in t: their bits are compared
        return {"out": s.out, "t": s.t.view(torch.int32)}
    if s.kind == "taa":
        api.light_taa(s.ctx, s.vd, s.rgb, s.last, s.out, s.depth, s.g.normal, s.g.material, s.pal, motion=s.motion, seed=s.seed)
        return {"out": s.out}
    if s.kind == "shade":
        api.shade_forward(s.ctx, s.vd, s.g, s.vis, s.pal, s.light, s.rgb, ssao=s.ssao)
        dl = torch.sub(s.rgb, s.target).mul_(2.0)
        api.shade_backward(s.ctx, s.vd, s.g, s.vis, s.pal, s.light, dl, s.dpal, s.dlight, ssao=s.ssao)
        return {"rgb": s.rgb, "dpalette": s.dpal, "dlight": s.dlight}
    raise ValueError(s.kind)


# ---------------------------------------------------------------- floors

def work(case):
    """Inputs read once and outputs written once. A traversal's inputs are its G-buffer and the scene (a bit per
    voxel for the occupancy, a byte for the materials); its operations are counted as 60 to set a ray up and 24 a
    voxel step over 8 steps, the least a ray takes in these scenes."""
    kind = case["kind"]
    ray = 60 + 24 * 8
    if kind == "batch":
        px = case["scenes"] * (256 + case["max_width"]) / 2 * (256 + case["max_height"]) / 2
        vox = case["scenes"] * ((64 + case["max_edge"]) / 2) ** 3
        return {"bytes": px * (25 + 9) + vox / 8, "flops": px * 0.7 * (1 + case["n_ao"]) * ray}
    if kind == "city":
        px = case["views"] * case["width"] * case["height"]
        return {"bytes": px * (25 + 9 + 30 + 12) + case["edge"] ** 3 / 8, "flops": px * ((1 + case["n_ao"] + case["n_spec"]) * ray + 200)}
    px = case["width"] * case["height"]
    vox = case["nx"] * case["ny"] * case["nz"]
    if kind == "trace":
        rays = case["n_shadow"] + case["n_ao"] + case["n_spec"]
        return {"bytes": px * (25 + 9) + vox / 8, "flops": px * 0.7 * rays * ray}
    if kind == "primary":
        return {"bytes": px * (25 + 4 + 4) + vox / 8, "flops": px * (ray + 400)}
    if kind == "moving":
        model = case["draws"] * (case["edge"] * 0.75) ** 3 + 8 * case["nx"] * case["nz"]
        return {"bytes": 2 * model + px * (25 + 14 + 9), "flops": 2 * model * 12 + px * 4 * ray}
    if kind == "world":
        return {"bytes": vox * (1 + 1 / 8 + 1 / 64 + 2 / 8) + px * (25 + 9), "flops": vox * 12 + px * 0.7 * 6 * ray}
    if kind == "lights":
        return {"bytes": px * (25 + 5 + 12) + vox / 8, "flops": px * 0.7 * (100 + 0.03 * (case["points"] + case["spots"]) * ray)}
    if kind == "reflection":
        return {"bytes": px * (25 + 4 + 16 + 16 + 4) + vox / 8, "flops": px * 0.7 * 3 * ray}
    if kind == "taa":
        return {"bytes": px * (12 + 16 + 8 + 4 + 12 + 1 + 16), "flops": px * 12 * 200}
    return {"bytes": px * (25 + 5 + 12 + 25 + 5 + 12 + 12), "flops": px * (60 + 200)}   # shade


# ---------------------------------------------------------------- results in 64 bits

def _shade_exact(s):
    """The shaded image and the L2 loss gradient's palette and light gradients, by autograd in float64."""
    f = lambda t: t.double()
    mat = s.g.material.long()
    hit = mat > 0
    pal = f(s.pal).requires_grad_(True)
    light = torch.from_numpy(np.asarray(s.light, np.float64)).cuda().requires_grad_(True)
    e = pal[mat[hit]]
    n, pos = f(s.g.normal[hit]), f(s.g.pos[hit])
    cam = torch.from_numpy(np.asarray(s.vd["cam_pos"], np.float64)).cuda() * 10.0
    v = torch.nn.functional.normalize(cam - pos, dim=1)
    s5 = (1.0 - (n * v).sum(1).clamp(min=0.0)).clamp(min=0.0) ** 5
    ndl = (n @ (light[:3] / light[:3].norm())).clamp(min=0.0)
    vis = f(s.vis.shadow[hit])
    amb = f(s.vis.ao[hit]) * 0.05 * (f(s.ssao[hit]) if s.ssao is not None else 1.0)
    rough, metal, emit = e[:, 3], e[:, 4], e[:, 5]
    f0 = 0.04 * (1.0 - metal) + metal
    kd = (1.0 - (f0 + (1.0 - f0) * s5)) * (1.0 - metal)
    sky = 1.0 - 0.2 * 0.8
    irr = torch.tensor([sky * sky * 1.1, sky * 1.1, (0.6 + sky * 0.4) * 1.1], dtype=torch.float64, device="cuda")
    f0a = 0.04 * (1.0 - metal[:, None]) + e[:, :3] * metal[:, None]
    fr = f0a + (torch.maximum(1.0 - rough[:, None], f0a) - f0a) * s5[:, None]
    direct = (kd * ndl * vis)[:, None] * e[:, :3] / math.pi * light[3:]
    col = irr * e[:, :3] * (emit[:, None] * 10.0 + (1.0 - fr) * amb[:, None]) + direct
    rgb = torch.zeros(s.g.pos.shape, dtype=torch.float64, device="cuda").masked_scatter(hit[:, None].expand(-1, 3), col)
    ((rgb - f(s.target)) ** 2).sum().backward()
    return {"rgb": rgb.detach(), "dpalette": pal.grad, "dlight": light.grad}


def _hash32(x):
    x = x & 0xffffffff
    x = ((x ^ (x >> 16)) * 0x7feb352d) & 0xffffffff
    x = ((x ^ (x >> 15)) * 0x846ca68b) & 0xffffffff
    return x ^ (x >> 16)


def _taa_exact(case, s):
    """The accumulated frame in float64, with the sampler's 8-bit weights as they are defined."""
    w, h = case["width"], case["height"]
    npx = w * h
    f = lambda t: t.double()
    mat = s.g.material.long()
    e = torch.where((mat > 0)[:, None], f(s.pal)[mat], torch.zeros((), dtype=torch.float64, device="cuda"))
    one = lambda x: x[:, None]
    # per pixel: light 0:3, its alpha 3, colour 4:7, material 7:10, border flag 10, normal 11:14, motion 14:16, depth 16
    rec = torch.cat([f(s.rgb), one(f(mat == 0)), e, torch.zeros((npx, 1), dtype=torch.float64, device="cuda"), f(s.g.normal),
                     f(s.motion), one(f(s.depth))], 1)
    edge = torch.zeros((1, 17), dtype=torch.float64, device="cuda")
    edge[0, 3] = edge[0, 10] = 1.0
    rec = torch.cat([rec, edge])
    last = torch.cat([f(s.last), torch.tensor([[0.0, 0.0, 0.0, 1.0]], dtype=torch.float64, device="cuda")])

    def sample(img, u, v):
        def axis(x, size):
            x = x.clamp(-2.0, size + 1.0)
            fl = x.floor()
            fr = ((x - fl) * 256.0 + 0.5).floor() / 256.0
            return (fl + (fr >= 1.0)).long(), torch.where(fr >= 1.0, torch.zeros_like(fr), fr)
        (x0, fx), (y0, fy) = axis(u * w - 0.5, w), axis(v * h - 0.5, h)
        acc = 0.0
        for dx, dy in ((0, 0), (1, 0), (0, 1), (1, 1)):
            x, y = x0 + dx, y0 + dy
            at = torch.where((x >= 0) & (y >= 0) & (x < w) & (y < h), y * w + x, npx)
            acc = acc + img[at] * one((fx if dx else 1.0 - fx) * (fy if dy else 1.0 - fy))
        return acc

    def surface(c, n):
        k = (0.8 <= 1.0 - (c[:, 7:11] - n[:, 7:11]).norm(dim=1)).double()
        k = k * (c[:, 11:14] * n[:, 11:14]).sum(1).clamp(min=0.0) * (1.0 - ((c[:, 16] - n[:, 16]).abs() * 4096.0).clamp(0.0, 1.0))
        return torch.where((c[:, 14:16] - n[:, 14:16]).norm(dim=1) > 0.1, torch.zeros_like(k), k)

    i = torch.arange(npx, device="cuda")
    u, v = (f(i % w) + 0.5) / w, (f(i // w) + 0.5) / h
    c = sample(rec, u, v)
    out = c[:, :4].clone()                                   # sky pixels keep this frame's light
    ou, ov = u + c[:, 14], v + c[:, 15]
    off = (ou < 0.0) | (ou > 1.0) | (ov < 0.0) | (ov > 1.0)
    hit = c[:, 16] != 1.0
    at = torch.nonzero(hit & off).reshape(-1)                # history outside the image: a 19x19 neighbourhood
    if at.numel():
        cc, acc, cnt = c[at], 0.0, 0.0
        for x in range(-9, 10):
            for y in range(-9, 10):
                n = sample(rec, (u[at] + x / w).clamp(0.001, 0.999), (v[at] + y / h).clamp(0.001, 0.999))
                k = surface(cc, n) * (1.0 - (cc[:, 4:7] - n[:, 4:7]).norm(dim=1).clamp(0.0, 1.0))
                acc, cnt = acc + one(k) * n[:, :3], cnt + k
        out[at] = torch.cat([acc / one(cnt), torch.ones_like(one(cnt))], 1)
    at = torch.nonzero(hit & ~off).reshape(-1)
    if at.numel():
        cc, hist = c[at], sample(last, ou[at], ov[at])
        frame = _hash32(torch.tensor(s.vd["frame"] + 0x9e3779b9, device="cuda"))
        pk = _hash32(_hash32((s.seed ^ 0x85ebca6b) ^ frame) ^ _hash32(at))
        angle = f(_hash32(pk) >> 8) / 16777216.0 * 3.1415 * 2.118033988749895
        lvar, scale = hist[:, 3], torch.minimum(torch.full_like(angle, 0.5), 1.0 / cc[:, 16])
        lo, hi = torch.full_like(cc[:, :3], 10000.0), torch.zeros_like(cc[:, :3])
        acc, cnt, diff = 0.0, 0.0, 1.0
        for r in range(2, 14):
            rr = r * (lvar + 1.0) * scale
            n = sample(rec, (u[at] + angle.cos() / w * rr).clamp(0.001, 0.999), (v[at] + angle.sin() / h * rr).clamp(0.001, 0.999))
            k = (1.212 - r / 12.0) * surface(cc, n) * (1.0 - ((cc[:, 4:7] - n[:, 4:7]).norm(dim=1) * 10000.0).clamp(0.0, 1.0))
            lo, hi = torch.minimum(lo, n[:, :3]), torch.maximum(hi, n[:, :3])
            acc, cnt = acc + one(k) * n[:, :3], cnt + k
            diff = diff + (n[:, :3] - cc[:, :3]).norm(dim=1) * k
            angle = angle + 2.39
        cur = (cc[:, :3] + acc) / one(cnt + 1.0)
        old = torch.minimum(torch.maximum(hist[:, :3], lo), hi)
        var = ((cur - old).abs() @ torch.tensor([0.2125, 0.7154, 0.0721], dtype=torch.float64, device="cuda") * 5.5).clamp(0.0, 1.0)
        lvar = lvar + var - diff / 13.0 * 0.08 + cc[:, 14:16].norm(dim=1) * 20.0
        t = one((1.0 - lvar).clamp(0.3, 0.9))
        out[at] = torch.cat([cur * (1.0 - t) + old * t, one((lvar * 0.7).clamp(0.0, 1.0))], 1)
    return {"out": out}


def exact(case, seed):
    if case["kind"] == "shade":
        return _shade_exact(prepare(case, seed))
    if case["kind"] == "taa":
        return _taa_exact(case, prepare(case, seed))
    # What a ray meets, and with it the shadow, occlusion, light and reflection values, is defined by fp32 steps and
    # comparisons.
    return None
