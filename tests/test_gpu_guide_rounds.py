"""The training round's kernels at the edges of their groups: the gradient of
1 to 17 x 64 + 1 records (64 to a group, 16 groups to a chunk of the sum, 16
records to a wave's tile) against the float64 oracle with fp16 operands
emulated, and the copies of the gate's record counts across batches of other
sizes."""
import numpy as np
import pytest

import clovers_amd
from clovers_amd import abi, synth
from oracle import guide_ref as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 1023, 1024, 1025, 1089])
def test_gradient_at_group_edges(n):
    """tolerance: an fp16 operand is off by up to 2^-11 of itself and a gradient passes through 8 rounded
    layers (4 forward, 4 back), so 8 x 2^-11 = 3.9e-3 of a layer's norm if every rounding fell the same way"""
    P = G.init_params(5).astype(np.float32)
    s = G.random_samples(n, seed=n).astype(np.float32)
    with clovers_amd.Renderer(0) as r:
        r.guide_set_params(P)
        g = r.guide_grad(s)
        again = r.guide_grad(s)
    assert np.array_equal(g, again)
    ref = G.grad(P.astype(np.float64), s.astype(np.float64), fp16=True)
    for a, b in [(G.W1, G.B1), (G.B1, G.W2), (G.W2, G.B2), (G.B2, G.W3), (G.W3, G.B3), (G.B3, G.W4), (G.W4, G.B4),
                 (G.B4, G.NPARAM)]:
        assert np.linalg.norm(g[a:b] - ref[a:b]) < 4e-3 * np.linalg.norm(ref[a:b]), (n, a)


@pytest.mark.parametrize("photons", [1, 63, 65, 100003])
def test_record_counts_do_not_leak_between_batches(photons):
    """a guided render gives the same bytes and evaluations before and after guided batches of 2 and of 17
    jobs, whose counts lie in other copies of the same buffer"""
    with clovers_amd.Renderer(0) as r:
        sid = r.upload(synth.prism())
        r.set_tuning(guide_photons=photons, guide_pre_rounds=2)
        one = (sid, abi.render_opts(96, 80, 12, 12, seed=5, guiding=abi.GUIDE_ON))
        first, _ = r.render(*one)
        q = r.counters()["guide_queries"]
        for n in (2, 17):
            r.render_batch([(sid, abi.render_opts(24, 24, 6, 8, seed=k, guiding=abi.GUIDE_ON)) for k in range(n)])
            again, _ = r.render(*one)
            assert np.array_equal(first, again) and r.counters()["guide_queries"] == q
