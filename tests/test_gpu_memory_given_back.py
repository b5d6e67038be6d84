"""A context keeps the buffers of its largest passes.  A later call that finds no memory gets theirs: uploads, larger
images, probes and other renders work after a large render as they do before it."""
import numpy as np
import pytest
import torch

import clovers_amd
from clovers_amd import abi, synth

pytestmark = pytest.mark.gpu

MB = 1 << 20


@pytest.fixture(scope="module")
def most():
    """all memory but 12 GB, held once: taking it takes seconds"""
    torch.zeros(1, device="cuda")
    kept = [torch.empty(torch.cuda.mem_get_info()[0] - (12 << 30), dtype=torch.uint8, device="cuda")]
    yield  # not the tensor: a fixture's value outlives its end
    kept.clear()
    torch.cuda.empty_cache()


@pytest.fixture(autouse=True)
def nothing_cached():
    yield
    torch.cuda.empty_cache()


def _leave(left):
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    return torch.empty(torch.cuda.mem_get_info()[0] - left, dtype=torch.uint8, device="cuda")


def _large(r, guiding):
    """a render whose passes take 1.6 GB (plain) or 9 GB (guided)"""
    sid = r.upload(synth.prism())
    r.set_tuning(guide_photons=1 << 14, guide_pre_rounds=1)
    r.render(sid, abi.render_opts(1024, 1024, 128 if guiding == abi.GUIDE_OFF else 96, 2, seed=3, guiding=guiding))
    return sid


@pytest.mark.parametrize("guiding", [abi.GUIDE_OFF, abi.GUIDE_ON])
@pytest.mark.parametrize("builder", ["host", "device"])
def test_upload(most, guiding, builder):
    mesh, o = synth.mesh(freq=224), abi.render_opts(64, 48, 2, 4, seed=1)
    with clovers_amd.Renderer(0) as r:
        want = r.render(r.upload(mesh, builder=builder), o)[0]
    with clovers_amd.Renderer(0) as r:
        first = _large(r, guiding)
        held = _leave(96 * MB)  # the scene takes 110 MB, its build more
        sid = r.upload(mesh, builder=builder)
        assert np.array_equal(r.render(sid, o)[0], want)
        assert r.render(first, o)[0].shape == (48, 64, 3)
        del held


@pytest.mark.parametrize("what,guiding", [("hits", abi.GUIDE_OFF), ("debug", abi.GUIDE_OFF), ("image", abi.GUIDE_OFF),
                                          ("image", abi.GUIDE_ON), ("network", abi.GUIDE_ON)])
def test_other_calls(most, what, guiding):
    """calls that take 1.2 to 1.6 GB where 768 MB are left"""
    def call(r, sid):
        if what == "hits":
            return r.primary_hits(sid, abi.render_opts(3000, 2000, 1, 2, seed=1))[1]
        if what == "debug":
            return r.render_debug(sid, abi.render_opts(3000, 2000, 1, 2, seed=1), abi.MODE_NORMAL_MAP)
        if what == "network":
            return r.guide_eval(np.zeros((7 << 19, 7), np.float32))[0]
        return r.render(sid, abi.render_opts(5000, 3000, 1, 2, seed=1))[0]
    with clovers_amd.Renderer(0) as r:
        sid = r.upload(synth.prism())
        r.guide_reset(5)
        want = call(r, sid)
    with clovers_amd.Renderer(0) as r:
        sid = _large(r, guiding)
        r.guide_reset(5)
        held = _leave(768 * MB)
        assert np.array_equal(call(r, sid), want, equal_nan=True)
        del held


def test_a_tuned_size(most):
    """passes of a size that was asked for, while larger ones are held"""
    with clovers_amd.Renderer(0) as r:
        sid = _large(r, abi.GUIDE_OFF)
        held = _leave(64 * MB)
        r.set_tuning(target_paths=1 << 21, trace_kernel=abi.TRACE_SIMPLE)
        o = abi.render_opts(1024, 1024, 4, 4, seed=2)
        got = r.render(sid, o)[0]
        del held
        torch.cuda.empty_cache()
        with clovers_amd.Renderer(0) as q:
            assert np.array_equal(q.render(q.upload(synth.prism()), o)[0], got)
