"""collect: positions and velocities packed on the device, at mass counts
around the packing kernel's blocks, and the stress buffer, which is read as
zero until a tracked step or set_stress may have written it."""
import numpy as np
import pytest

import mercury_amd as mh
from mercury_amd.robots import Element

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("masses", [2, 85, 86, 256, 1000])
def test_collect_returns_what_was_uploaded(masses):
    print("collect", masses, flush=True)
    rng = np.random.default_rng(masses)
    pos, vel = rng.normal(size=(2, masses, 3)).astype(np.float32)
    el = Element(pos, np.ones(masses, np.uint8), np.array([[0, 1]], np.uint16), np.ones(1, np.float32),
                 np.ones(1, np.uint8), vel=vel)
    sim = mh.Simulator(mh.workload_materials(), mh.SimConfig(time_step=1e-4))
    sim.SetElements([el, el])
    for _ in range(2):
        p, v, st = sim.collect_arrays()
        assert np.array_equal(p, np.concatenate([pos, pos])) and np.array_equal(v, np.concatenate([vel, vel]))
        assert not st.any()


def test_stress_after_each_kind_of_write():
    print("collect stress", flush=True)
    ms = mh.workload_materials()
    robots = mh.voxel_population(ms, 2, voxels_per_axis=3, seed=4, mass=0.001)
    active = np.concatenate([r.spring_material != 0 for r in robots])
    sim = mh.Simulator(ms, mh.SimConfig(solver=mh.MH_SOLVER_XPBD_REF, time_step=1e-4))
    sim.SetElements(robots)
    sim.Step(200)
    assert not sim.collect_arrays()[2].any()
    sim.Step(50, trackStresses=True)
    st = sim.collect_arrays()[2]
    assert st[active].any() and not st[~active].any()
    sim.Step(20)  # untracked: kept
    assert np.array_equal(sim.collect_arrays()[2], st)
    sim.SetElements(robots)
    assert not sim.collect_arrays()[2].any()
    sim.set_stress(st + 1)
    assert np.array_equal(sim.collect_arrays()[2], st + 1)
