"""K nearest neighbours at the sizes where the kernel changes: 64 candidates
per register, the switch between register counts (512, 1024, 1536, 2048
masses) and to the scan (over 2048 masses, under 6 neighbours).  Results are exact: the same FP32
distances, ranked by (distance, index), as a sort on the CPU gives."""
import numpy as np
import pytest

from mercury_amd import robots

pytestmark = pytest.mark.gpu

SIZES = [33, 64, 65, 257, 512, 513, 1024, 1025, 1537, 2048, 2049]


def sorted_knn(p, k):
    with np.errstate(all="ignore"):
        d = p[:, None, :] - p[None, :, :]
        d = d * d
        dist = np.sqrt(d[..., 0] + (d[..., 1] + d[..., 2]))
    dist[(dist == 0) | np.isnan(dist)] = np.inf
    order = np.argsort(dist, axis=1, kind="stable")[:, :k]
    dist = np.take_along_axis(dist, order, 1)
    return np.where(np.isinf(dist), 0xFFFF, order).astype(np.uint16), dist


def cloud(kind, n, rng):
    p = rng.uniform(-1, 1, (n, 3)).astype(np.float32)
    if kind == "lattice":  # many equal distances
        p = np.stack(np.unravel_index(np.arange(n), (13, 13, 13)), 1).astype(np.float32)
    elif kind == "one_distance":  # more than 64 candidates at the same distance
        p = np.tile(np.float32([[0, 0, 0], [1, 0, 0]]), (n, 1))[:n]
    elif kind == "coincident":
        p[:] = 0.25
    elif kind == "scales":  # underflow to zero and overflow to infinity
        p *= np.float32(10.0) ** rng.integers(-25, 25, (n, 1)).astype(np.float32)
    elif kind == "non_finite":
        p[rng.integers(0, n, 5), 0] = np.nan
        p[rng.integers(0, n, 5), 1] = np.inf
    elif kind == "clusters":
        p = (p * np.float32(0.01) + rng.integers(0, 3, (n, 1)).astype(np.float32)).astype(np.float32)
    return p


@pytest.mark.parametrize("kind", ["uniform", "lattice", "one_distance", "coincident", "scales", "non_finite", "clusters"])
@pytest.mark.parametrize("k", [5, 6, 25, 32])
def test_knn_exact(kind, k):
    print("knn", kind, k, flush=True)
    rng = np.random.default_rng(k)
    pos = [cloud(kind, n, rng) for n in SIZES]
    mo = np.concatenate([[0], np.cumsum(SIZES)]).astype(np.uint32)
    nbr, dist = robots.knn_batch(mo, np.concatenate(pos), k)
    for r, p in enumerate(pos):
        en, ed = sorted_knn(p, k)
        np.testing.assert_array_equal(dist[mo[r]:mo[r + 1]], ed)
        np.testing.assert_array_equal(nbr[mo[r]:mo[r + 1]], en)
