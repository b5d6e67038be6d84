"""Wavefront passes behind the last training round are joined into larger ones
in a context with the default pass size: the same bytes as with the passes
planned one by one (a pass size next to the default), for a guided job alone,
beside an unguided job that starts in the training passes, and with a frozen
network."""
import numpy as np
import pytest

import clovers_amd
from clovers_amd import abi, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("frozen", [False, True])
@pytest.mark.parametrize("other", [None, (96, 64, 500), (700, 500, 20)])
def test_joined_passes_give_the_same_bytes(other, frozen):
    with clovers_amd.Renderer(0) as r:
        p, a = r.upload(synth.prism()), r.upload(synth.cornell())
        flags = abi.FLAG_GUIDE_FROZEN if frozen else 0
        jobs = [(p, abi.render_opts(320, 256, 160, 12, seed=4, guiding=abi.GUIDE_ON, flags=flags))]
        if other:
            jobs.append((a, abi.render_opts(other[0], other[1], other[2], 6, seed=9)))
        r.set_tuning(guide_rounds=2, guide_pre_rounds=2, guide_photons=1 << 16)
        got = r.render_batch(jobs, want_sq=True)
        passes = r.counters()["passes"]
        r.set_tuning(target_paths=(1 << 22) + 1)
        want = r.render_batch(jobs, want_sq=True)
        assert passes < r.counters()["passes"]
        for (x, xs), (y, ys) in zip(got, want):
            assert np.array_equal(x, y, equal_nan=True) and np.array_equal(xs, ys, equal_nan=True)
