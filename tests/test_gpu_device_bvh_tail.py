"""The end of the GPU tree builder's clustering runs in one block, from 1,024 clusters down.  Trees of as many
primitives as lead there, at once or after some iterations over the whole device, spread out and all at one place
(every union ties): the hits and images of the host-built tree."""
import numpy as np
import pytest

import clovers_amd
from clovers_amd import abi
from test_gpu_device_bvh import both, lamp_scene, sphere

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 3, 63, 64, 65, 1022, 1023, 1024, 1025, 2049, 3000])
@pytest.mark.parametrize("spread", [True, False])
def test_hits_do_not_depend_on_the_tree(n, spread):
    rng = np.random.Generator(np.random.PCG64(n))
    objs = [sphere((0, 0, 0), 0.5, "lamp", priority=True)]
    for _ in range(n - 1):
        c = rng.uniform(-2, 2, 3) if spread else np.array([0.25, 0.1, 0.2])
        objs.append(sphere([float(x) for x in c], float(rng.uniform(0.02, 0.1)) if spread else 0.3))
    o = abi.render_opts(48, 48, 4, 4, seed=7)
    with clovers_amd.Renderer(0) as r:
        scene = lamp_scene(objs)
        a, b = both(r, scene, lambda sid: (r.primary_hits(sid, o)[1], r.render(sid, o)[0], r.counters()["rays"]))
        assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1]) and a[2] == b[2]
