"""A call that finds no memory fails by itself: it leaves no error of the runtime behind for this context's next call
or for another library in the process."""
import numpy as np
import pytest
import torch

import clovers_amd
from clovers_amd import abi, synth

pytestmark = pytest.mark.gpu


def test_a_failed_call_leaves_no_error_behind():
    with clovers_amd.Renderer(0) as r:
        sid = r.upload(synth.cornell())
        o = abi.render_opts(64, 64, 2, 4, seed=2)
        want = r.render(sid, o)[0]
        one = torch.ones(1, device="cuda")
        held = torch.empty(torch.cuda.mem_get_info()[0] - (64 << 20), dtype=torch.uint8, device="cuda")
        for _ in range(2):
            with pytest.raises(clovers_amd.ClvError) as e:
                r.primary_hits(sid, abi.render_opts(4096, 4096, 1, 1, seed=1))
            assert e.value.status == abi.ENOMEM
        assert float((one + one).item()) == 2.0
        del held
        torch.cuda.empty_cache()
        for _ in range(2):
            assert np.array_equal(r.render(sid, o)[0], want)
