"""mh_mlp_forward_noalloc on both sides of the batch sizes where a network
that fits the fused kernels takes the layer-by-layer ones: the rows of
mh_mlp_forward, which scores in chunks that stay fused."""
import numpy as np
import pytest

import mercury_amd as mh
from mercury_amd.surrogate import MLP
from test_zz_no_alloc import DevArray, hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,batch", [
    ([1, 1], 8192), ([1, 1], 8193), ([7, 33], 8200), ([128, 128], 25024), ([128, 128], 25025), ([128, 130], 8193),
    ([256, 3], 8193), ([8, 8, 1], 16384), ([8, 8, 1], 16385), ([5, 33, 17, 3], 16400), ([9, 100, 2], 20001),
    ([6, 5, 7, 8, 2], 16385)], ids=lambda v: "-".join(map(str, v)) if isinstance(v, list) else str(v))
def test_routes_give_the_same_rows(sizes, batch):
    print("noalloc route", sizes, batch, flush=True)
    lib, rt = mh.load(), hip()
    rng = np.random.default_rng(batch)
    net = MLP(sizes, seed=4)
    x = rng.normal(size=(batch, sizes[0])).astype(np.float32)
    t = rng.normal(size=(300, sizes[-1])).astype(np.float32)
    net.train(x[:300], t, epochs=1, batch=100, lr=1e-2, seed=1)  # both forms of the weights are the trained ones
    want = net.forward(x)
    dx, dy = DevArray(rt, x.nbytes), DevArray(rt, want.nbytes)
    try:
        dx.put(x)
        dy.put(np.full_like(want, np.nan))
        assert lib.mh_mlp_forward_noalloc(net._h, dx.p, batch, dy.p, None) == 0, lib.mh_last_error()
        net.forward(x[:1])  # waits for the network's stream
        np.testing.assert_array_equal(dy.get(np.zeros_like(want)), want)
    finally:
        dx.free()
        dy.free()
