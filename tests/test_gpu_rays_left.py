"""Rays of scenes in memory that a wave leaves on their way (k_paths): a ray that is gone on with later, with its
stack in LDS or beyond it, ends at the hit that it finds in one go.  Against the bounce-by-bounce wavefront: the same
bytes, second moments and ray counts, for scenes whose rays differ in length (a deep tree beside a plane, instances,
media, moving spheres) and for so few rays that none is left."""
import numpy as np
import pytest

import clovers_amd
from clovers_amd import abi, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(3, 1, 1), (64, 2, 1), (131, 97, 2), (320, 180, 8)])
@pytest.mark.parametrize("names", [("mesh",), ("mesh", "features"), ("features", "media"), ("mesh", "motion", "media")])
def test_rays_left_on_their_way(names, size):
    make = {"mesh": lambda: synth.mesh(freq=90), "features": synth.features, "media": synth.media,
            "motion": lambda: synth.spheres(moving=True)}
    w, h, spp = size
    with clovers_amd.Renderer(0) as r:
        jobs = [(r.upload(make[k]()), abi.render_opts(w, h, spp, 14, seed=w + i)) for i, k in enumerate(names)]
        got = r.render_batch(jobs, want_sq=True)
        rays = r.counters()["rays"]
        r.set_tuning(trace_kernel=abi.TRACE_SIMPLE)
        want = r.render_batch(jobs, want_sq=True)
        assert rays == r.counters()["rays"]
        for a, b in zip(got, want):
            for x, y in zip(a, b):
                assert np.array_equal(x, y, equal_nan=True)
