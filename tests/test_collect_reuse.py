"""collect after populations of changing size on one simulator: its packing
buffer is kept, grown or given back."""
import numpy as np
import pytest

import mercury_amd as mh
from mercury_amd.robots import Element

pytestmark = pytest.mark.gpu


def test_collect_after_populations_of_changing_size():
    print("collect reuse", flush=True)
    rng = np.random.default_rng(0)
    sim = mh.Simulator(mh.workload_materials(), mh.SimConfig(time_step=1e-4))
    for masses, copies in ((3, 1), (700, 9), (701, 9), (400, 9), (300, 3), (2, 1), (1000, 40)):
        pos, vel = rng.normal(size=(2, masses, 3)).astype(np.float32)
        el = Element(pos, np.ones(masses, np.uint8), np.array([[0, 1]], np.uint16), np.ones(1, np.float32),
                     np.ones(1, np.uint8), vel=vel)
        sim.SetElements([el] * copies)
        for _ in range(2):
            p, v, _ = sim.collect_arrays()
            assert np.array_equal(p, np.tile(pos, (copies, 1))) and np.array_equal(v, np.tile(vel, (copies, 1)))
