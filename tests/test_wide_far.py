"""The force solver's batched step on robots far from the origin (1.8e19 and
more from the padding records' ghost, squared distances overflow) whose lists
do not fill a batch: finite, and the FP32 mirror's bits.  Every mass has the
same number of springs, so that no list is padded to a longer one's length."""
import numpy as np
import pytest

import mercury_amd as mh
from helpers import LAND, Case, bits, gpu_sim, mirror

pytestmark = pytest.mark.gpu


def complete(n, x, seed):
    """n masses in the plane at x, every pair joined."""
    rng = np.random.default_rng(seed)
    pos = rng.uniform(0.1, 0.3, (n, 3)).astype(np.float32)
    pos[:, 0] = x
    a, b = np.triu_indices(n, 1)
    e = mh.Element(pos, np.ones(n, np.uint8), np.stack([a, b], 1).astype(np.uint16),
                   np.linalg.norm(pos[a, 1:] - pos[b, 1:], axis=1).astype(np.float32), np.full(len(a), 2, np.uint8))
    e.mass = np.full(n, 0.01, np.float32)
    return e


@pytest.mark.parametrize("block", [256, 512, 768])
@pytest.mark.parametrize("springs", [1, 3, 4, 5, 6, 7])
def test_far_robots_stay_finite(block, springs):
    print("far robots, block", block, "springs per mass", springs, flush=True)
    case = Case([complete(springs + 1, x, springs) for x in (0.0, 3e19, -1e25)], mh.workload_materials(),
                mh.materials.WORKLOAD_ROWS)
    sim = gpu_sim(case, mh.MH_SOLVER_FORCE, 1e-4, LAND, kernel=mh.MH_KERNEL_MASS, block_size=block, robots_per_block=1)
    sim.Step(21)
    pos, vel, _ = sim.collect_arrays()
    p, v, _ = mirror(case, mh.MH_SOLVER_FORCE, 21, 1e-4, LAND)
    assert np.isfinite(p).all() and np.abs(v).max() > 0
    assert np.array_equal(bits(pos), bits(p))
    assert np.array_equal(bits(vel), bits(v))
