"""The convolutional network's scores, loss, gradient and trained parameters
against tests/golden/cnn_layerwise.json: the bits that the layer-by-layer
kernels (a matrix product or a column sum per launch, fp32 activations in
memory) gave on an MI355X before one kernel per direction replaced them.  The
fused kernels keep every product's operands and every sum's order."""
import hashlib
import json
import os

import numpy as np
import pytest

from mercury_amd import evolve, surrogate

pytestmark = pytest.mark.gpu
GOLDEN = json.load(open(os.path.join(os.path.dirname(__file__), "golden", "cnn_layerwise.json")))


def sha(a):
    return hashlib.sha256(np.ascontiguousarray(a, np.float32).tobytes()).hexdigest()


@pytest.mark.parametrize("n", [int(n) for n in GOLDEN])
def test_cnn_bits_of_the_layer_by_layer_kernels(n):
    print("cnn golden, batch of", n, flush=True)
    want = GOLDEN[str(n)]
    rng = np.random.default_rng(n)
    g = evolve.random_genomes(rng, n, 8)
    t = rng.normal(size=n).astype(np.float32)
    net = surrogate.CNN(seed=n)
    y = net.forward(g)
    assert [int(v) for v in y.view(np.uint32)[:4]] == want["scores"]
    assert sha(y) == want["scores_sha256"]
    loss, grad = net.loss_grad(g, t)
    assert float(np.float32(loss)).hex() == want["loss"] and sha(grad) == want["gradient_sha256"]
    loss = net.train(g, t, epochs=2, batch=max(1, n // 3), lr=1e-3, seed=5)
    assert float(np.float32(loss)).hex() == want["train_loss"] and sha(net.get_params()) == want["trained_sha256"]
