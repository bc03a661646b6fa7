"""mh_mlp_forward_noalloc with y inside x: every row of x is read before a row
of y is written, so the results are those of separate buffers, also after
training has changed the weights."""
import ctypes

import numpy as np
import pytest

import mercury_amd as mh
from mercury_amd.surrogate import MLP
from test_zz_no_alloc import DevArray, hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("where", ["start", "middle", "end"])
@pytest.mark.parametrize("sizes,batch", [([64, 256, 256, 1], 3001), ([5, 33, 17, 3], 700), ([32, 32, 32], 513)],
                         ids=lambda v: "-".join(map(str, v)) if isinstance(v, list) else str(v))
def test_output_inside_the_input(sizes, batch, where):
    print("noalloc, y inside x:", sizes, batch, where, flush=True)
    lib, rt = mh.load(), hip()
    rng = np.random.default_rng(batch)
    x = rng.normal(size=(batch, sizes[0])).astype(np.float32)
    t = rng.normal(size=(batch, sizes[-1])).astype(np.float32)
    net = MLP(sizes, seed=3)
    net.train(x, t, epochs=1, batch=batch // 3, lr=1e-2, seed=1)
    want = net.forward(x)
    room = 4 * batch * (sizes[0] - sizes[-1])
    at = {"start": 0, "middle": room // 8 * 4, "end": room}[where]
    dx = DevArray(rt, x.nbytes)
    try:
        dx.put(x)
        y = ctypes.c_void_p(dx.p.value + at)
        assert lib.mh_mlp_forward_noalloc(net._h, dx.p, batch, y, None) == 0, lib.mh_last_error()
        net.forward(x[:1])  # waits for the network's stream
        got = np.zeros_like(want)
        assert rt.hipMemcpy(got.ctypes.data, y, got.nbytes, 2) == 0
        np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))
    finally:
        dx.free()
