"""Both sides of the lines where the mass-parallel kernels change form, exact
against the FP32 mirror, with the plan each parameter is meant to have: XPBD
packs of at most 512 masses (at most 256 where every mass starts at most one
spring), and the force step's launches of at most one workgroup per CU."""
import numpy as np
import pytest
import torch

import mercury_amd as mh
from helpers import LAND, Case, bits, gpu_sim, mirror, workload_case
from test_pair_order import ring

pytestmark = pytest.mark.gpu
XPBD = mh.MH_SOLVER_XPBD_REF


@pytest.mark.parametrize("stress", [False, True])
@pytest.mark.parametrize("masses,reach,robots", [("voxels 7", 13, 2), (512, 2, 2), (513, 2, 2), (256, 1, 2),
                                                 (257, 1, 2), (512, 1, 1)])
def test_xpbd_wide_line(masses, reach, robots, stress):
    print("xpbd wide line", masses, reach, stress, flush=True)
    if masses == "voxels 7":
        masses = 512
        case = workload_case(n_robots=robots, voxels=7, seed=4)
    else:
        case = Case([ring(masses, reach, 30)] * robots, mh.workload_materials(), mh.materials.WORKLOAD_ROWS)
    sim = gpu_sim(case, XPBD, 1e-4, robots_per_block=1)
    info = sim.info()
    assert info.kernel == mh.MH_KERNEL_MASS_GATHER and info.block_size == 768 and info.max_masses_per_block == masses
    sim.Step(61, trackStresses=stress)
    for got, want in zip(sim.collect_arrays(), mirror(case, XPBD, 61, 1e-4, stress=stress)):
        if want is not None:
            np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("block,voxels", [(256, 5), (512, 7), (768, 8)])
def test_force_wide_line(block, voxels):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    print("force wide line", block, voxels, cus, flush=True)
    case = workload_case(n_robots=2, voxels=voxels, seed=block)
    p, v, _ = mirror(case, mh.MH_SOLVER_FORCE, 41, 1e-4, LAND)
    n = len(p)
    for robots in (cus, cus + 1):
        sim = mh.Simulator(case.ms, mh.SimConfig(solver=mh.MH_SOLVER_FORCE, time_step=1e-4, kernel=mh.MH_KERNEL_MASS,
                                                 block_size=block, robots_per_block=1, **LAND))
        sim.SetElements(case.elements + case.elements[:1] * (robots - 2))
        assert sim.info().n_blocks == robots
        sim.Step(41)
        pos, vel, _ = sim.collect_arrays()
        assert np.array_equal(bits(pos[:n]), bits(p)) and np.array_equal(bits(vel[:n]), bits(v))
