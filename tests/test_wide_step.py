"""The force solver's step for launches of at most one workgroup per CU (256
on MI355X) against the one for more, bit for bit: the same robots alone in a
launch and among enough others, at list lengths that do not fill a batch, in
every block size, and with springs short enough to leave the fast
arithmetic's range."""
import numpy as np
import pytest

import mercury_amd as mh
from mercury_amd.robots import random_voxel_encodings, voxel_build
from helpers import LAND, bits

pytestmark = pytest.mark.gpu


def robots(n, voxels, seed):
    ms = mh.workload_materials()
    rng = np.random.default_rng(seed)
    return [voxel_build(ms, voxels + 1, 10.0, random_voxel_encodings(rng, voxels, 4, 0.3), mass=0.001)
            for _ in range(n)]


def trajectory(els, block, steps):
    sim = mh.Simulator(mh.workload_materials(),
                       mh.SimConfig(solver=mh.MH_SOLVER_FORCE, time_step=1e-4, kernel=mh.MH_KERNEL_MASS,
                                    block_size=block, robots_per_block=1, **LAND))
    sim.SetElements(els)
    sim.Step(steps)
    pos, vel, _ = sim.collect_arrays()
    return pos, vel, sim.info().n_blocks


@pytest.mark.parametrize("block,voxels", [(256, 1), (256, 3), (256, 5), (512, 6), (768, 8), (1024, 9)])
def test_few_and_many_workgroups_give_the_same_bits(block, voxels):
    print("wide step, block", block, "voxels", voxels, flush=True)
    els = robots(3, voxels, seed=block + voxels)
    # one robot with two masses a hair apart and one with all its masses in
    # a plane of tiny springs: squared lengths below 2^-30
    els[1].pos[1] = els[1].pos[0] + np.float32(1e-6)
    els[2].pos *= np.float32(1e-5)
    many = els + robots(1, voxels, seed=1) * 297
    pos_a, vel_a, blocks_a = trajectory(els, block, 61)
    pos_b, vel_b, blocks_b = trajectory(many, block, 61)
    assert blocks_a == 3 and blocks_b == 300
    assert np.isfinite(pos_a).all() and np.abs(vel_a).max() > 0
    assert np.array_equal(bits(pos_a), bits(pos_b[:len(pos_a)]))
    assert np.array_equal(bits(vel_a), bits(vel_b[:len(vel_a)]))
