"""Large results of which some go to pinned memory and the others to pageable memory, in every order: the same bytes as
with all of them pageable."""
import ctypes as C

import numpy as np
import pytest
import torch

import clovers_amd
from clovers_amd import abi, synth

pytestmark = pytest.mark.gpu


def _pinned(n):
    t = torch.empty(n, dtype=torch.float32, pin_memory=True)
    return t, t.numpy()


@pytest.mark.parametrize("pinned", [(True, False), (False, True), (True, True)])
def test_image_and_second_moments(pinned):
    w, h = 1921, 1080
    keep, res = [], []
    with clovers_amd.Renderer(0) as r:
        sid = r.upload(synth.cornell())
        o = abi.render_opts(w, h, 1, 2, seed=3)
        want = [a.reshape(-1) for a in r.render(sid, o, want_sq=True)]
        for p in pinned:
            t, a = _pinned(3 * w * h) if p else (None, np.empty(3 * w * h, np.float32))
            keep.append(t)
            res.append(a)
        for _ in range(4):
            for a in res:
                a.fill(-1.0)
            r._check(r.lib.clv_render(r.h, sid, C.byref(o), res[0].ctypes.data, res[1].ctypes.data))
            for a, b in zip(res, want):
                assert np.array_equal(a, b, equal_nan=True)


@pytest.mark.parametrize("ids_pinned", [True, False])
def test_hits(ids_pinned):
    w, h = 3001, 2003
    with clovers_amd.Renderer(0) as r:
        sid = r.upload(synth.spheres(seed=3))
        o = abi.render_opts(w, h, 1, 1, seed=5)
        want = r.primary_hits(sid, o)
        t, pin = _pinned(w * h)
        page = np.empty(w * h, np.float32)
        for _ in range(4):
            pin.fill(-1.0)
            page.fill(-1.0)
            a, b = (pin, page) if ids_pinned else (page, pin)
            r._check(r.lib.clv_primary_hits(r.h, sid, C.byref(o), a.ctypes.data, b.ctypes.data))
            assert np.array_equal(a.view(np.uint32), want[0].reshape(-1)) and np.array_equal(b, want[1].reshape(-1))
