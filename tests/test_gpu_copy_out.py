"""Results on their way to the caller: pageable memory is reached through pinned windows, a flag behind
every 64 KB and helper threads; memory that the runtime knows (pinned) is copied to directly.  Both give the
same bytes, whatever the size and the destination's alignment, and nothing beside them is written."""
import ctypes as C
import threading

import numpy as np
import pytest
import torch

import clovers_amd
from clovers_amd import abi, synth

pytestmark = pytest.mark.gpu

# ids and ts: 4 bytes a pixel.  Less than a chunk, one chunk and its neighbours, one window (8 MB) and its
# neighbours, and more windows than the two that alternate.
SIZES = [(1, 1), (127, 43), (128, 128), (16385, 1), (2048, 1024), (2099, 1000), (1920, 1080), (3001, 2003)]


@pytest.fixture(scope="module")
def scene():
    r = clovers_amd.Renderer(0)
    sid = r.upload(synth.spheres(seed=3))
    for _ in range(3):  # a context's first small copies are the runtime's
        r.primary_hits(sid, abi.render_opts(3001, 2003, 1, 1, seed=5))
    return r, sid


def _buffers(words, shift):
    """the same room in pageable and in pinned memory, `shift` words into an array with canaries around it"""
    page = np.full(words + 64, 0xC0FFEE, np.uint32)
    pin = torch.empty(words, dtype=torch.int32, pin_memory=True)
    return page, page[16 + shift:16 + shift + words], pin, pin.numpy().view(np.uint32)


def _canaries(page, words, shift):
    assert (page[:16 + shift] == 0xC0FFEE).all() and (page[16 + shift + words:] == 0xC0FFEE).all()


@pytest.mark.parametrize("w,h", SIZES)
@pytest.mark.parametrize("shift", [0, 1])
def test_hits(scene, w, h, shift):
    r, sid = scene
    o = abi.render_opts(w, h, 1, 1, seed=5)
    a, b = _buffers(w * h, shift), _buffers(w * h, 3 * shift)
    r._check(r.lib.clv_primary_hits(r.h, sid, C.byref(o), a[1].ctypes.data, b[1].ctypes.data))
    r._check(r.lib.clv_primary_hits(r.h, sid, C.byref(o), a[3].ctypes.data, b[3].ctypes.data))
    for got, k in ((a, shift), (b, 3 * shift)):
        assert np.array_equal(got[1], got[3])
        _canaries(got[0], w * h, k)


@pytest.mark.parametrize("w,h", SIZES)
def test_normals(scene, w, h):
    r, sid = scene
    o = abi.render_opts(w, h, 1, 1, seed=5)
    page, got, _pin, want = _buffers(3 * w * h, 1)
    for dst in (got, want):
        r._check(r.lib.clv_render_debug(r.h, sid, C.byref(o), abi.MODE_NORMAL_MAP, dst.ctypes.data))
    assert np.array_equal(got, want)
    _canaries(page, 3 * w * h, 1)


def _batch(r, sid, sizes, bufs, sqs):
    arr = (abi.Job * len(sizes))()
    for k, (w, h) in enumerate(sizes):
        arr[k].scene_id = sid
        arr[k].opts = abi.render_opts(w, h, 1, 2, seed=7 + k)
        arr[k].xyz_out = bufs[k].ctypes.data
        arr[k].xyz_sq_out = sqs[k].ctypes.data if sqs[k] is not None else None
    r._check(r.lib.clv_render_batch(r.h, arr, len(sizes)))


def test_batch(scene):
    """images of odd sizes whose borders lie anywhere in the windows, one destination pinned, second moments
    of some"""
    r, sid = scene
    sizes = [(33, 21), (1001, 701), (17, 1), (1280, 719), (640, 333)]
    words = [3 * w * h for w, h in sizes]
    img, sq = [_buffers(n, k) for k, n in enumerate(words)], [_buffers(n, 1) for n in words]
    some = [k != 1 for k in range(len(sizes))]
    _batch(r, sid, sizes, [b[3] for b in img], [b[3] if s else None for b, s in zip(sq, some)])
    _batch(r, sid, sizes, [b[3 if k == 2 else 1] for k, b in enumerate(img)],
           [b[1] if s else None for b, s in zip(sq, some)])
    for k, n in enumerate(words):
        if k != 2:
            assert np.array_equal(img[k][1], img[k][3])
        _canaries(img[k][0], n, k)
        if some[k]:
            assert np.array_equal(sq[k][1], sq[k][3])
        else:
            assert (sq[k][0] == 0xC0FFEE).all()


def test_same_destination(scene):
    """two jobs that write the same array: the later one's image is what is left"""
    r, sid = scene
    w, h = 1025, 800
    both, last = np.empty(3 * w * h, np.float32), np.empty(3 * w * h, np.float32)
    other = np.empty_like(last)
    _batch(r, sid, [(w, h), (w, h)], [other, last], [None, None])
    _batch(r, sid, [(w, h), (w, h)], [both, both], [None, None])
    assert np.array_equal(both, last) and not np.array_equal(other, last)


def test_contexts_beside_each_other(scene):
    """a context's windows, flags and helpers are its own"""
    r, sid = scene
    w, h = 1920, 1080
    want = r.primary_hits(sid, abi.render_opts(w, h, 1, 1, seed=1))
    bad = []

    def program(k):
        q = clovers_amd.Renderer(0)
        s = q.upload(synth.spheres(seed=3))
        for _ in range(8):
            got = q.primary_hits(s, abi.render_opts(w, h, 1, 1, seed=1))
            if not all(np.array_equal(a, b) for a, b in zip(got, want)):
                bad.append(k)

    threads = [threading.Thread(target=program, args=(k,)) for k in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
