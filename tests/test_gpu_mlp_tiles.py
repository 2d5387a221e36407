"""The MLP's products with a weight matrix at the edges of their 32 x 32 tiles
and 16-deep slices, against the oracle that rounds its operands to BF16."""
import numpy as np
import pytest

import mlp_oracle as M
from test_gpu_learned import make_net

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,batch", [((4, 36, 64, 1), 1), ((32, 33, 31, 65), 33), ((8, 100, 60, 33), 64),
                                        ((17, 130, 260, 96), 31)])
def test_gradients_and_predictions(dims, batch):
    print(f"case mlp tiles dims={dims} batch={batch}", flush=True)
    net, p = make_net(dims, batch, seed=sum(dims))
    rng = np.random.default_rng(batch)
    X = rng.standard_normal((batch, dims[0])).astype(np.float32)
    Y = (rng.uniform(size=(batch, dims[3])) < 0.3).astype(np.float32)
    loss, g = net.gradients(X, Y)
    lo, go = M.loss_grad(p, X, Y, dims, bf16=True)
    net.close()
    # the same BF16 operands; FP32 sums in another order move a few of the
    # activations across a BF16 rounding (2^-9 relative): the suite's bound
    assert abs(loss - lo) <= 1e-4 * abs(lo)
    assert np.linalg.norm(g - go) <= 2e-3 * np.linalg.norm(go)
