"""The forms that view dicts and region lists may take: the structures filled as
bytes equal those filled element by element through ctypes, and what ctypes
refuses stays refused (host only)."""
import ctypes as C

import numpy as np
import pytest
import torch

from voxelengine_amd import _lib as L
from voxelengine_amd import api, views

BASE = views.scene_view((64, 64, 64), 61, 43, frame=3)
MAT = np.asarray(BASE["view"], np.float32).reshape(16)


def _view_by_elements(vd):
    v = L.View()
    for k in ("last_view", "view", "inv_view", "proj", "inv_proj"):
        setattr(v, k, L.f16(*np.asarray(vd[k], np.float32).reshape(16)))
    for k, n in (("res", 2), ("ires", 2), ("cam_pos", 3), ("jitter", 2)):
        setattr(v, k, (C.c_float * n)(*[float(x) for x in vd[k]]))
    v.frame, v.width, v.height = vd["frame"], vd["width"], vd["height"]
    return v


VIEWS = {
    "as made": {}, "short": dict(res=(61.0,), jitter=(), cam_pos=[1, 2]), "text": dict(res=("61", "4.5e1")),
    "tensors": dict(res=tuple(torch.tensor([61.0, 43.0])), cam_pos=torch.tensor([1.0, 2.0, 3.0])),
    "beyond fp32": dict(cam_pos=(1e300, -1e300, 1e-300)), "nan": dict(cam_pos=(float("nan"), float("inf"), -0.0)),
    "whole": dict(cam_pos=(10 ** 30, 2, -3), ires=np.array([1, 2])), "widths": dict(cam_pos=(np.float16(1.1), np.float32(2.2), np.longdouble(3.3))),
    "bytes": dict(res=b"=+"), "4x4": dict(view=MAT.reshape(4, 4)), "column order": dict(view=np.asfortranarray(MAT.reshape(4, 4))),
    "float64": dict(view=MAT.astype(np.float64), proj=MAT.tolist()), "other byte order": dict(view=MAT.astype(">f4")),
    "strided": dict(view=np.repeat(MAT, 2)[::2], last_view=torch.from_numpy(MAT.copy())),
}


@pytest.mark.parametrize("name", VIEWS)
def test_views(name):
    vd = dict(BASE, **VIEWS[name])
    assert bytes(api.view_struct(vd)) == bytes(_view_by_elements(vd))


def test_view_elements_from_an_iterator():
    want = bytes(_view_by_elements(dict(BASE, cam_pos=("1", 2, 3))))
    assert bytes(api.view_struct(dict(BASE, cam_pos=(x for x in ("1", 2, 3))))) == want


@pytest.mark.parametrize("bad", [dict(res=(1.0, 2.0, 3.0)), dict(cam_pos=(None, 0, 0)), dict(cam_pos=(1j, 0, 0)), dict(res=("a", "b")),
                                 dict(cam_pos=[[1, 2], [3, 4], [5, 6]]), dict(view=np.zeros(15, np.float32)), dict(jitter=None)])
def test_refused_views(bad):
    vd = dict(BASE, **bad)
    with pytest.raises(Exception) as by_elements:
        _view_by_elements(vd)
    with pytest.raises(by_elements.type):
        api.view_struct(vd)


REGIONS = {
    "tuples": lambda: [(1, 2, 3, 4, 5, 6), (7, 8, 9, 1, 2, 3)], "iterators": lambda: [iter((1, 2, 3, 4, 5, 6)), map(int, "123456")],
    "short": lambda: [(1, 2, 3), (1, 2, 3, 4, 5, 6)], "lists": lambda: [[1, 2, 3, 4, 5, 6]], "arrays": lambda: [np.arange(6), np.arange(6, dtype=np.int8)],
    "truth values": lambda: [(True,) * 6], "negative": lambda: [(-1, -2, -3, 4, 5, 6)], "wide": lambda: [(2 ** 40 + 1, 2, 3, 4, 5, 2 ** 32 - 1)],
    "wider": lambda: [(2 ** 70 + 1, 2, 3, 4, 5, 6)], "unsigned": lambda: [(np.uint64(2 ** 63 + 3), -2, 3, 4, 5, 6), (np.uint64(3), 2, 3, 4, 5, 6)],
    "tensors": lambda: [torch.arange(6), tuple(torch.arange(6))],
    # refused
    "seven": lambda: [(1, 2, 3, 4, 5, 6, 7)], "floats": lambda: [(1.0, 2, 3, 4, 5, 6)], "texts": lambda: ["123456", ("1", "2", "3", "4", "5", "6")],
    "nested": lambda: [(np.array([1]),) * 6], "nothing": lambda: [(None,) * 6], "structures": lambda: [L.Region(1, 2, 3, 4, 5, 6)],
}


@pytest.mark.parametrize("name", REGIONS)
def test_regions(name):
    try:
        want = bytes((L.Region * len(REGIONS[name]()))(*[L.Region(*r) for r in REGIONS[name]()]))
    except Exception as e:
        with pytest.raises(type(e)):
            api._regions(REGIONS[name]())
    else:
        assert bytes(api._regions(REGIONS[name]())) == want
