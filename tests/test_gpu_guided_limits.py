"""A guided render whose large passes just fit: the network's and the gate's memory belong to what has to fit beside
them, so the render falls back to passes of the default size instead of failing."""
import numpy as np
import pytest
import torch

import clovers_amd
from clovers_amd import abi, synth

pytestmark = pytest.mark.gpu


def test_network_and_gate_have_room():
    o = abi.render_opts(1024, 1024, 96, 3, seed=3, guiding=abi.GUIDE_ON)

    def free_bytes():
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        return torch.cuda.mem_get_info()[0]

    def render(left=None):
        with clovers_amd.Renderer(0) as r:
            r.set_tuning(guide_photons=1 << 14, guide_pre_rounds=1)
            sid = r.upload(synth.prism())
            r.primary_hits(sid, abi.render_opts(16, 16, 1, 1, seed=1))
            held = torch.empty(free_bytes() - left, dtype=torch.uint8, device="cuda") if left else None
            before = free_bytes()
            try:
                img = r.render(sid, o)[0]
                used = before - free_bytes()
            finally:
                del held
            return img, r.counters()["passes"], used

    render()  # what the runtime allocates once per process
    want, few, used = render()
    most = torch.empty(free_bytes() - used - (512 << 20), dtype=torch.uint8, device="cuda")

    def fits(spare):
        img, n, _ = render(used + spare)
        assert np.array_equal(img, want), spare
        return n == few
    spare = 160 << 20
    assert fits(spare)
    while fits(spare - (16 << 20)):
        spare -= 16 << 20
    for k in range(1, 7):  # through the 18 MB of the gate's buffers
        fits(spare - k * (4 << 20))
    del most
    torch.cuda.empty_cache()
