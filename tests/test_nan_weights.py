"""A weight that is not a number makes every output that depends on it not a
number, whatever its payload (rounding a NaN's bits to bf16 as if it were a
number turns some payloads into infinity or zero)."""
import numpy as np
import pytest

from mercury_amd import evolve, surrogate

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits", [0x7fc00000, 0x7f800001, 0x7fffffff, 0xffffffff])
@pytest.mark.parametrize("kind", ["64-256-256-1", "5-300-1", "cnn"])
def test_nan_weight_reaches_the_output(kind, bits):
    print("NaN weight", kind, hex(bits), flush=True)
    rng = np.random.default_rng(1)
    if kind == "cnn":
        net, x = surrogate.CNN(seed=2), evolve.random_genomes(rng, 9, 8)
        sizes = net.LAYERS
    else:
        shape = [int(v) for v in kind.split("-")]
        net, x = surrogate.MLP(shape, seed=2), rng.normal(size=(9, shape[0])).astype(np.float32)
        sizes = list(zip(shape[1:], shape[:-1]))
    p0, at = net.get_params(), 0
    for n_out, n_in in sizes:
        p = p0.copy()
        p.view(np.uint32)[at + n_in + (n_out > 1) * n_in // 2 - 1] = bits  # a weight of the first or second unit
        if kind == "cnn" and n_in == 135:  # every input channel of one offset: some voxel has one of them
            p.view(np.uint32)[at + 65:at + 70] = bits
        net.set_params(p)
        assert np.isnan(net.forward(x)).all(), (n_out, n_in)
        at += n_out * n_in + n_out
