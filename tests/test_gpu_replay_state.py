"""The replay of a captured render leaves the guiding network's state alone: parameters loaded after the capture are
still the trained network of the next guided render that keeps it."""
import numpy as np
import pytest

import clovers_amd
from clovers_amd import abi, synth
from oracle import guide_ref as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("replays", [0, 1, 3])
def test_loaded_parameters_survive_replays(replays):
    plain = abi.render_opts(64, 64, 4, 6, seed=2)
    keep = abi.render_opts(64, 64, 8, 6, seed=3, guiding=abi.GUIDE_ON, flags=abi.FLAG_GUIDE_KEEP)
    P = G.init_params(5).astype(np.float32)
    with clovers_amd.Renderer(0) as r:
        sid = r.upload(synth.prism())
        r.set_tuning(guide_rounds=0, guide_photons=0)
        r.guide_grad(G.random_samples(64, seed=1).astype(np.float32))  # the network exists, untrained
        images = [r.render(sid, plain)[0] for _ in range(3)]  # eager, captured, replayed
        r.guide_set_params(P)
        images += [r.render(sid, plain)[0] for _ in range(replays)]
        got = r.render(sid, keep)[0]
        assert r.counters()["guide_queries"] > 0
        assert np.array_equal(r.guide_params(), P)
    assert all(np.array_equal(images[0], i) for i in images)
    with clovers_amd.Renderer(0) as r:
        sid = r.upload(synth.prism())
        r.set_tuning(guide_rounds=0, guide_photons=0)
        r.guide_set_params(P)
        assert np.array_equal(r.render(sid, keep)[0], got)
