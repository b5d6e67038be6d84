"""The autotuner tries only what makes a difference: a batch whose fastest shape runs whole paths in one launch keeps
the tail setting it had, and its pass size stays automatic unless a smaller one is faster."""
import pytest

import clovers_amd
from clovers_amd import abi, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tail", [0, 5])
def test_whole_paths_have_no_tail_to_tune(tail):
    with clovers_amd.Renderer(0) as r:
        sid = r.upload(synth.spheres())
        for w, h, spp in ((64, 48, 4), (128, 128, 8), (320, 180, 16), (320, 180, 64)):
            r.set_tuning(tail_depth=tail, trace_kernel=abi.TRACE_LDS_CACHED, target_paths=1 << 22)
            best = r.autotune([(sid, abi.render_opts(w, h, spp, 12, seed=1))])
            if best["trace_kernel"] == abi.TRACE_LDS_CACHED:
                assert best["tail_depth"] == tail
            assert r.tuning() == best
        assert best["trace_kernel"] == abi.TRACE_LDS_CACHED  # twice as fast on this scene


@pytest.mark.parametrize("spp", [3, 15, 32])
def test_a_size_that_gives_the_same_passes_is_not_chosen(spp):
    """the trial in one pass is the automatic size's; a set size that holds the trial too is kept to in renders of
    more samples, so it is no candidate"""
    with clovers_amd.Renderer(0) as r:
        sid = r.upload(synth.spheres())
        n = 1920 * 1080 * spp
        best = r.autotune([(sid, abi.render_opts(1920, 1080, spp, 12, seed=1))])
        assert best["trace_kernel"] == abi.TRACE_LDS_CACHED  # twice as fast on this scene
        assert best["target_paths"] == 1 << 22 or best["target_paths"] < n
