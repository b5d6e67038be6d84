"""Guided renders of scenes that LDS does not hold trace by majority (a wave takes turns of nodes or of primitives):
the same images, second moments, ray counts and trained network as with the other traversal kernels, for one large
scene, a small one, and scenes that share a batch (instances and moving spheres among them)."""
import numpy as np
import pytest

import clovers_amd
from clovers_amd import abi, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("names", [("mesh",), ("small",), ("mesh", "prism"), ("features", "motion", "mesh")])
@pytest.mark.parametrize("w,h,spp", [(7, 3, 40), (161, 97, 37)])
def test_majority_traces_the_same_hits(names, w, h, spp):
    make = {"mesh": lambda: synth.mesh(freq=40), "small": lambda: synth.mesh(freq=8), "prism": synth.prism,
            "features": synth.features, "motion": lambda: synth.spheres(moving=True)}
    res = []
    with clovers_amd.Renderer(0) as r:
        jobs = [(r.upload(make[k]()), abi.render_opts(w, h, spp, 8, seed=w + i, guiding=abi.GUIDE_ON))
                for i, k in enumerate(names)]
        r.set_tuning(guide_rounds=2, guide_pre_rounds=1, guide_photons=1 << 14)
        for kernel in (abi.TRACE_LDS_CACHED, abi.TRACE_SIMPLE, abi.TRACE_WW):
            r.set_tuning(trace_kernel=kernel)
            out = r.render_batch(jobs, want_sq=True)
            res.append([a for pair in out for a in pair] + [r.guide_params(), np.array([r.counters()["rays"]])])
    for other in res[1:]:
        for x, y in zip(res[0], other):
            assert np.array_equal(x, y, equal_nan=True)
