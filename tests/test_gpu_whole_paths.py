"""Renders whose passes run whole paths in one launch (k_paths, the LDS-cached
kernel without guided jobs) against the bounce-by-bounce wavefront: the same
bytes, second moments and ray counts.  The sizes are where its bookkeeping can
go wrong: fewer samples than a wave, a block or the grid, one more or less
than each, samples split over passes, jobs of one batch in one pass and in
several."""
import numpy as np
import pytest

import clovers_amd
from clovers_amd import abi, synth

pytestmark = pytest.mark.gpu


def both(r, jobs, **tuning):
    """the batch by whole paths and by the wavefront: (images and second moments) and rays of each"""
    out = []
    for kernel in (abi.TRACE_LDS_CACHED, abi.TRACE_SIMPLE):
        r.set_tuning(trace_kernel=kernel, **tuning)
        res = r.render_batch(jobs, want_sq=True)
        out.append(([a for pair in res for a in pair], r.counters()["rays"]))
    return out


def same(a, b):
    assert a[1] == b[1]
    for x, y in zip(a[0], b[0]):
        assert np.array_equal(x, y, equal_nan=True)


@pytest.mark.parametrize("name", ["cornell", "spheres", "motion", "prism", "features", "media", "mesh"])
@pytest.mark.parametrize("size", [(1, 1, 1), (63, 1, 1), (65, 1, 1), (13, 59, 1), (8, 96, 1), (769, 1, 1),
                                  (127, 33, 96), (641, 617, 1), (129, 1, 1), (511, 1, 1), (513, 1, 1)])
def test_whole_paths_equal_the_wavefront(name, size):
    make = {"cornell": synth.cornell, "spheres": synth.spheres, "motion": lambda: synth.spheres(moving=True),
            "prism": synth.prism, "features": synth.features, "media": synth.media,
            "mesh": lambda: synth.mesh(freq=24)}[name]
    w, h, spp = size
    with clovers_amd.Renderer(0) as r:
        sid = r.upload(make())
        same(*both(r, [(sid, abi.render_opts(w, h, spp, 9, seed=w + h))]))


@pytest.mark.parametrize("target", [1 << 16, 1 << 22])
def test_batches_of_scenes_and_passes(target):
    """jobs of several scenes (one of them in LDS), sizes, depths and accumulator types; at the
    small pass size most jobs are split over passes"""
    with clovers_amd.Renderer(0) as r:
        a, b, c = r.upload(synth.cornell()), r.upload(synth.spheres()), r.upload(synth.mesh(freq=16))
        jobs = [(a, abi.render_opts(97, 61, 33, 8, seed=1)), (b, abi.render_opts(160, 90, 12, 16, seed=2, fp64_accum=1)),
                (c, abi.render_opts(64, 64, 17, 12, seed=3)), (a, abi.render_opts(31, 7, 1, 0, seed=4)),
                (b, abi.render_opts(128, 130, 5, 3, seed=5, sample_offset=1000))]
        x, y = both(r, jobs, target_paths=target)
        assert (r.counters()["passes"] > 5) == (target == 1 << 16)
        same(x, y)
        r.set_tuning(trace_kernel=abi.TRACE_LDS_CACHED)
        for k, (sid, o) in enumerate(jobs):  # and each job alone
            img, sq = r.render(sid, o, want_sq=True)
            assert np.array_equal(img, x[0][2 * k]) and np.array_equal(sq, x[0][2 * k + 1])


def test_scenes_that_share_a_batch_are_read_from_memory():
    """a batch of several scenes is not in LDS: instance chains, checkers, a cone light, moving
    spheres and media through the kernel that reads nodes and records from memory, and a scene
    that fits in LDS but not in the tuned share of it"""
    with clovers_amd.Renderer(0) as r:
        a, b, c = r.upload(synth.features()), r.upload(synth.media()), r.upload(synth.spheres(moving=True))
        o = abi.render_opts(90, 70, 7, 11, seed=8)
        for jobs in ([(a, o), (c, o)], [(a, o), (b, o), (c, o)]):
            x, y = both(r, jobs)
            same(x, y)
            r.set_tuning(trace_kernel=abi.TRACE_LDS_CACHED)
            for k, (sid, _) in enumerate(jobs):
                assert np.array_equal(r.render(sid, o)[0], x[0][2 * k])
        want = r.render(c, o)[0]
        r.set_tuning(lds_bytes=16384)
        assert np.array_equal(r.render(c, o)[0], want)
