"""K nearest neighbours of clouds whose distances coincide: few distinct
points (more than 64 candidates at one distance, taken level by level), each
point many times, coarse grids, and levels whose squared distances differ and
roots do not; and robots around the mass count where few neighbours are
searched by the scan.  Exact, as in test_knn_waves."""
import numpy as np
import pytest

from mercury_amd import robots
from test_knn_waves import sorted_knn

pytestmark = pytest.mark.gpu
SIZES = [40, 63, 64, 65, 300, 520, 1100, 2000]


def cloud(kind, n, rng):
    if kind.startswith("points"):
        p = rng.uniform(-1, 1, (int(kind[6:]), 3))[rng.integers(0, int(kind[6:]), n)]
    elif kind.startswith("copies"):
        p = np.repeat(rng.uniform(-1, 1, (n, 3)), int(kind[6:]), axis=0)[:n]
    elif kind.startswith("grid"):
        p = rng.integers(0, int(kind[4:]), (n, 3))
    elif kind == "roots":  # squared distances of neighbouring floats, one root
        x = np.float32(1.5) + np.float32(2.0 ** -23) * rng.integers(0, 5, n)
        p = np.stack([np.where(np.arange(n) % 2, x, 0), np.zeros(n), np.zeros(n)], 1)
    elif kind == "one_off":  # nearly all coincide
        p = np.zeros((n, 3))
        p[rng.integers(0, n, 3)] = [1, 2, 3]
    elif kind == "far":  # levels that overflow
        p = rng.choice([0.0, 1.0, 3e19, -3e19], (n, 3))
    return p.astype(np.float32)


@pytest.mark.parametrize("kind", ["points2", "points3", "points5", "points30", "copies4", "copies40", "grid2", "grid3",
                                  "roots", "one_off", "far"])
@pytest.mark.parametrize("k", [6, 15, 16, 25, 32])
def test_knn_ties_exact(kind, k):
    print("knn ties", kind, k, flush=True)
    rng = np.random.default_rng(k)
    pos = [cloud(kind, n, rng) for n in SIZES]
    mo = np.concatenate([[0], np.cumsum(SIZES)]).astype(np.uint32)
    nbr, dist = robots.knn_batch(mo, np.concatenate(pos), k)
    for r, p in enumerate(pos):
        en, ed = sorted_knn(p, k)
        np.testing.assert_array_equal(dist[mo[r]:mo[r + 1]], ed)
        np.testing.assert_array_equal(nbr[mo[r]:mo[r + 1]], en)
