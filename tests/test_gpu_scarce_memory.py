"""An untuned context runs larger passes than the default size where memory allows; where it does not, renders run
with passes of that size and give the same bytes."""
import numpy as np
import pytest
import torch

import clovers_amd
from clovers_amd import abi, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("guiding,left", [(abi.GUIDE_ON, 3 << 30), (abi.GUIDE_OFF, 3 << 28)])
def test_passes_of_the_default_size_when_memory_is_scarce(guiding, left):
    with clovers_amd.Renderer(0) as r:
        opts = abi.render_opts(1024, 1024, 96, 3, seed=3, guiding=guiding)
        r.set_tuning(guide_photons=1 << 14, guide_pre_rounds=1)
        sid = r.upload(synth.prism())
        free, _ = torch.cuda.mem_get_info()
        held = torch.empty(free - left, dtype=torch.uint8, device="cuda")
        try:
            few = r.render(sid, opts)[0]
            passes = r.counters()["passes"]
        finally:
            del held
            torch.cuda.empty_cache()
    with clovers_amd.Renderer(0) as r:
        r.set_tuning(guide_photons=1 << 14, guide_pre_rounds=1)
        sid = r.upload(synth.prism())
        assert np.array_equal(r.render(sid, opts)[0], few)
        assert r.counters()["passes"] < passes
