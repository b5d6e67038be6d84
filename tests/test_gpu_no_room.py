"""A context that found no memory for large passes does not look for it again in every call: a call takes about what it
takes with passes that were asked for at the default size, and large passes come back once there is memory."""
import time

import numpy as np
import pytest
import torch

import clovers_amd
from clovers_amd import abi, synth

pytestmark = pytest.mark.gpu


def test_no_room_is_remembered_until_there_is_some():
    o = abi.render_opts(512, 512, 64, 3, seed=3, guiding=abi.GUIDE_ON)
    with clovers_amd.Renderer(0) as r:
        r.set_tuning(guide_photons=1 << 14, guide_pre_rounds=1)
        sid = r.upload(synth.prism())

        def call():
            t = time.perf_counter()
            img = r.render(sid, o)[0]
            return (time.perf_counter() - t) * 1e3, r.counters()["passes"], img
        torch.zeros(1, device="cuda")
        held = [torch.empty(torch.cuda.mem_get_info()[0] - (3 << 30), dtype=torch.uint8, device="cuda")]
        scarce = [call() for _ in range(6)]
        r.set_tuning(target_paths=(1 << 22) - 1)
        asked = [call() for _ in range(6)]
        r.set_tuning(target_paths=1 << 22)
        scarce += [call() for _ in range(2)]
        held.clear()
        torch.cuda.empty_cache()
        roomy = [call() for _ in range(2)]
    med = lambda rows: sorted(t for t, _, _ in rows)[len(rows) // 2]  # noqa: E731
    # trying again took 90 to 120 ms a call beside renders of 7
    assert med(scarce[1:]) < 3 * med(asked[1:]), (scarce, asked)
    assert all(np.array_equal(img, scarce[0][2]) for _, _, img in scarce + asked + roomy)
    assert {n for _, n, _ in roomy} == {min(n for _, n, _ in roomy)} and roomy[0][1] < scarce[0][1], (roomy, scarce)
