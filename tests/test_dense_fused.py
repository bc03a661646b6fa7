"""The fused dense layers (mh_mlp_* for networks of up to 4 layers of at most
256 units) against the layer-by-layer kernels that wider networks take, bit
for bit, at the edges of their tiles: widths and batches that do not fill a
16-row tile, a 32-value slice or a row split, and the widest and deepest
networks they take.  The layer-by-layer kernels are held to the FP64 oracle
by the tests of the surrogate; a network reaches them when one of its layers
is widened past 256 by units whose weights are zero, which adds exact zeros
to every sum."""
import numpy as np
import pytest

from mercury_amd.surrogate import MLP
from helpers import adam_first_step_f32

pytestmark = pytest.mark.gpu

SHAPES = [[64, 256, 256, 1], [1, 1], [5, 33, 17, 3], [16, 32], [256, 256, 256, 256, 256], [7, 255, 18]]
BATCHES = [1, 15, 33, 130, 515]


def data(sizes, batch):
    rng = np.random.default_rng([batch, *sizes])
    x = rng.normal(size=(batch, sizes[0])).astype(np.float32)
    t = rng.normal(size=(batch, sizes[-1])).astype(np.float32)
    return MLP(sizes, seed=sum(sizes)), x, t


def widened(net):
    """The same network with layer k (the input where there is no hidden
    layer) widened to 300 units by zero weights; returns it and a function
    that takes its parameter vector back to the original's layout."""
    k = 1 if len(net.sizes) > 2 else 0
    n = net.sizes[k]
    sizes = list(net.sizes)
    sizes[k] = 300
    wide = MLP(sizes, seed=1)
    parts = []
    for (W, b), (Ww, bw) in zip(net.layers(), wide.layers()):
        P, q = np.zeros_like(Ww), np.zeros_like(bw)
        P[:W.shape[0], :W.shape[1]], q[:len(b)] = W, b
        parts += [P.reshape(-1), q]
    wide.set_params(np.concatenate(parts))

    def back(p):
        return np.concatenate([np.concatenate([Ww[:W.shape[0], :W.shape[1]].reshape(-1), bw[:len(b)]])
                               for (W, b), (Ww, bw) in zip(net.layers(), wide.layers(p))])

    def inputs(x):
        return x if k else np.pad(x, ((0, 0), (0, 300 - n)))
    return wide, inputs, back


@pytest.mark.parametrize("batch", BATCHES)
@pytest.mark.parametrize("sizes", SHAPES, ids=lambda s: "-".join(map(str, s)))
def test_fused_layers_equal_the_layer_by_layer_kernels(sizes, batch):
    print("fused dense", sizes, batch, flush=True)
    net, x, t = data(sizes, batch)
    wide, inputs, back = widened(net)
    np.testing.assert_array_equal(net.forward(x), wide.forward(inputs(x)))
    loss, g = net.loss_grad(x, t)
    loss_w, g_w = wide.loss_grad(inputs(x), t)
    assert loss == loss_w
    np.testing.assert_array_equal(g, back(g_w))
    # two epochs of shuffled batches with a dropped remainder
    step = max(1, batch // 3)
    assert net.train(x, t, epochs=2, batch=step, lr=1e-3, seed=5) == wide.train(inputs(x), t, epochs=2, batch=step,
                                                                              lr=1e-3, seed=5)
    np.testing.assert_array_equal(net.get_params(), back(wide.get_params()))
    np.testing.assert_array_equal(net.forward(x), wide.forward(inputs(x)))


@pytest.mark.parametrize("batch", [130, 515])
def test_fused_train_step_is_adam_on_its_own_gradient(batch):
    """Training updates the parameters inside the gradient kernel: one step
    must equal a float32 Adam step on loss_grad's gradient bit for bit (equal
    rows, so the shuffle does not matter), and a following forward pass must
    use the new weights, packed in both orders."""
    print("fused train step", batch, flush=True)
    net, x, t = data([5, 33, 17, 3], batch)
    x[:], t[:] = x[0], t[0]
    p0 = net.get_params()
    loss, g = net.loss_grad(x, t)
    assert net.train(x, t, epochs=1, batch=batch, lr=1e-2, seed=0) == loss
    p1 = net.get_params()
    np.testing.assert_array_equal(p1, adam_first_step_f32(p0, g, 1e-2))
    other = MLP(net.sizes, seed=1)
    other.set_params(p1)
    np.testing.assert_array_equal(net.forward(x), other.forward(x))
    np.testing.assert_array_equal(net.loss_grad(x, t)[1], other.loss_grad(x, t)[1])


def test_row_tiles_of_every_batch_size_give_the_same_rows():
    """The row tile grows with the batch (16, 32, 64 rows); a row's result
    does not depend on it."""
    print("fused row tiles", flush=True)
    net, x, _ = data([64, 256, 256, 1], 20011)
    y = net.forward(x)
    for n in (1, 17, 4096, 4097, 8192):
        np.testing.assert_array_equal(net.forward(x[:n]), y[:n])
