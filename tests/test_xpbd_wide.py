"""XPBD gather kernel on packs of few masses (its wide form) and of more:
stresses tracked and not, and a robot that overflows, whose waves take the
general division.  Exact against the FP32 mirror (NaN equal to NaN)."""
import numpy as np
import pytest

import mercury_amd as mh
from helpers import gpu_sim, mirror, reference_case, workload_case

pytestmark = pytest.mark.gpu
XPBD = mh.MH_SOLVER_XPBD_REF


@pytest.mark.parametrize("stress", [False, True])
@pytest.mark.parametrize("voxels", [1, 2, 4, 5, 6, 8])
@pytest.mark.parametrize("family", ["workload", "reference"])
def test_xpbd_wide_exact(family, voxels, stress):
    print("xpbd wide", family, voxels, stress, flush=True)
    case = (workload_case if family == "workload" else reference_case)(n_robots=3, voxels=voxels, seed=5)
    n0 = int(case.a["mass_offset"][1])
    case.a["vel"][n0] = [3e38, -3e38, 1.0]  # second robot
    sim = gpu_sim(case, XPBD, 1e-4)
    sim.set_population(case.a)
    sim.Step(61, trackStresses=stress)
    p, v, s = mirror(case, XPBD, 61, 1e-4, stress=stress)
    for got, want in zip(sim.collect_arrays(), (p, v, s)):
        if want is not None:
            assert np.array_equal(got, want, equal_nan=True)
