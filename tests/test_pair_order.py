"""The lanes that advance the pairs' rest lengths: the last ones where the
last waves have few records, else the first.  Rings have lists of one length,
voxel robots of 7 to 26 springs; with and without idle waves, fewer pairs
than a wave and more than the lanes.  Exact against the FP32 mirror."""
import numpy as np
import pytest

import mercury_amd as mh
from helpers import LAND, Case, gpu_sim, mirror, workload_case

pytestmark = pytest.mark.gpu


def ring(n, reach, pairs):
    i = np.arange(n)
    a = 2 * np.pi * i / n
    pos = np.stack([0.016 * n * np.cos(a), 0.5 + 0.01 * (i % 7), 0.016 * n * np.sin(a)], 1).astype(np.float32)
    ab = np.concatenate([np.stack([i, (i + j) % n], 1) for j in range(1, reach + 1)])
    rest = np.linalg.norm(pos[ab[:, 0]] - pos[ab[:, 1]], axis=1)
    rest = np.repeat([rest[j * n:(j + 1) * n].mean() for j in range(reach)], n)
    rest = (rest * (1 + 1e-3 * (np.arange(len(rest)) % (pairs // reach)))).astype(np.float32)
    e = mh.Element(pos, np.ones(n, np.uint8), ab.astype(np.uint16), rest, np.full(len(ab), 8, np.uint8))
    e.mass = np.full(n, 0.01, np.float32)
    return e


CASES = [(shape, block, solver, stress)
         for shape, block in (((760, 3, 30), 768), ((600, 1, 2), 768), ((700, 8, 480), 768), ((250, 2, 500), 256),
                              ((1000, 2, 40), 1024), ((512, 3, 200), 512), ("voxels", 768), ("voxels", 256))
         for solver, stress in (("force", False), ("xpbd", False), ("xpbd", True), ("gather", False), ("gather", True))
         if solver != "gather" or block < 1024]  # the gather kernel's blocks


@pytest.mark.parametrize("shape,block,solver,stress", CASES, ids=str)
def test_pair_order_exact(shape, block, solver, stress):
    print("pair order", shape, block, solver, stress, flush=True)
    if shape == "voxels":
        case = workload_case(n_robots=3, voxels=8 if block == 768 else 5, seed=2)
    else:
        case = Case([ring(*shape)] * 2, mh.workload_materials(), mh.materials.WORKLOAD_ROWS)
    so = mh.MH_SOLVER_FORCE if solver == "force" else mh.MH_SOLVER_XPBD_REF
    env = LAND if solver == "force" else None
    kernel = mh.MH_KERNEL_MASS_GATHER if solver == "gather" else mh.MH_KERNEL_MASS
    sim = gpu_sim(case, so, 1e-4, env, kernel=kernel, block_size=block, robots_per_block=1)
    assert sim.info().kernel == kernel and sim.info().block_size == block
    sim.Step(61, trackStresses=stress)
    want = mirror(case, so, 61, 1e-4, env, stress=stress)
    assert np.abs(want[1]).max() > 0
    for got, w in zip(sim.collect_arrays(), want):
        if w is not None:
            np.testing.assert_array_equal(got, w)
