"""The MLP's products with a weight matrix at the edges of their 32 x 32 tiles
and 16-deep slices, against the oracle that rounds its operands to BF16."""
import numpy as np
import pytest

import mlp_oracle as M
from test_gpu_learned import block_errors, make_net

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,batch", [((4, 36, 64, 1), 1), ((32, 33, 31, 65), 33), ((8, 100, 60, 33), 64),
                                        ((17, 130, 260, 96), 31), ((16, 136, 264, 96), 40),
                                        ((16, 136, 264, 97), 33)])  # 264: wide reads across, a last tile of 8
def test_gradients_and_predictions(dims, batch):
    print(f"case mlp tiles dims={dims} batch={batch}", flush=True)
    net, p = make_net(dims, batch, seed=sum(dims))
    rng = np.random.default_rng(batch)
    X = rng.standard_normal((batch, dims[0])).astype(np.float32)
    Y = (rng.uniform(size=(batch, dims[3])) < 0.3).astype(np.float32)
    loss, g = net.gradients(X, Y)
    lo, go = M.loss_grad(p, X, Y, dims, bf16=True)
    prob = net.predict_raw(X)
    net.close()
    # the same BF16 operands; FP32 sums in another order move a few of the
    # activations across a BF16 rounding (2^-9 relative): the suite's bounds,
    # for every block of the gradient and every prediction
    assert abs(loss - lo) <= 1e-4 * abs(lo)
    for k, e in block_errors(g, go, dims).items():
        assert e <= 2e-3, (k, e)
    assert np.max(np.abs(prob - M.predict(p, X, dims, bf16=True))) <= 2e-3


# ---- the order of the sums.  In ascending order every 1 added to 2^24 is lost
# (FP32 ties go to the even 2^24, truncation too), so the sum of this pattern
# is the last entry's: -2^24 + 2^24 = 0.  Summed in parts and joined, the ones
# survive.  One entry per 16-deep slice, so an MFMA adds a single product.
BIG = np.float32(2.0**24)


def pattern(k, step):
    v = np.zeros(k, np.float32)
    v[::step] = 1.0
    v[0] = BIG
    v[(k - 1) // step * step] = -BIG
    s = np.float32(0)
    for x in v:
        s = np.float32(s + x)
    assert s == 0 and v.astype(np.float64).sum() != 0
    return v


def pack(dims, **parts):
    o = M.layout(*dims)
    keys = ["W1", "b1", "W2", "b2", "W3", "b3", "n"]
    p = np.zeros(o["n"], np.float32)
    for a, b in zip(keys, keys[1:]):
        if a in parts:
            p[o[a]:o[b]] = np.broadcast_to(np.asarray(parts[a], np.float32),
                                           (o[b] - o[a],) if a[0] == "b" else
                                           {"W1": (dims[1], dims[0]), "W2": (dims[2], dims[1]),
                                            "W3": (dims[3], dims[2])}[a]).ravel()
    return p, o


@pytest.mark.parametrize("k", [100, 128, 1024])
@pytest.mark.parametrize("layer", [1, 2, 3])
def test_forward_sums_ascend(layer, k):
    print(f"case mlp forward order layer={layer} k={k}", flush=True)
    dims = [3, 5, 6, 4]
    dims[layer - 1] = k
    w = pattern(k, 16)
    # the layer's inputs are ones, the layers after it pass one value on
    parts = {f"W{layer}": w}
    if layer > 1:
        parts[f"b{layer - 1}"] = 1.0
    for later in range(layer + 1, 4):
        W = np.zeros((dims[later], dims[later - 1]), np.float32)
        W[:, 0] = 1.0
        parts[f"W{later}"] = W
    net, _ = make_net(tuple(dims), 3, seed=k)
    net.set_params(pack(dims, **parts)[0])
    assert np.all(net.predict_raw(np.ones((3, dims[0]), np.float32)) == 0.5)  # logits 0
    net.close()


@pytest.mark.parametrize("k,rows,h", [(64, 1, 5), (128, 2, 40), (1024, 1, 64), (64, 4096, 520)])
@pytest.mark.parametrize("layer", [2, 3])
def test_backward_sums_ascend(layer, k, rows, h):
    # rows x h beyond 2^21: the 64 x 64 tiles.  Sizes are powers of two: so are the errors (p - Y) / n.
    print(f"case mlp backward order layer={layer} k={k} rows={rows} h={h}", flush=True)
    dims = [2, h, k, 4] if layer == 2 else [2, 3, h, k]
    w = pattern(k, 16)[:, None]
    if layer == 3:
        parts = {"b1": 1.0, "b2": 1.0, "W3": w}
        z = w[:, 0]
    else:  # A1 = 2^-40: A2 = 1 and the logits stay 1
        parts = {"b1": 2.0**-40, "b2": 1.0, "W2": w, "W3": np.full((4, k), 2.0**-10)}
        z = np.full(4, k * 2.0**-10)
    p, o = pack(dims, **parts)
    net, _ = make_net(tuple(dims), rows, seed=k)
    net.set_params(p)
    prob = net.predict_raw(np.zeros((rows, 2), np.float32))
    assert np.array_equal(prob[0] > 0.5, z > 0) and np.array_equal(prob, np.broadcast_to(prob[:1], prob.shape))
    Y = prob - np.float32(1.0)  # every output error is (p - Y) / n: one value
    errors = (prob - Y)
    assert np.all(errors == errors[0, 0])
    g = net.gradients(np.zeros((rows, 2), np.float32), Y)[1]
    net.close()
    name = {3: "b2", 2: "b1"}[layer]
    end = {"b2": "W3", "b1": "W2"}[name]
    assert np.all(g[o[name]:o[end]] == 0.0)


@pytest.mark.parametrize("rows", [5, 16, 64, 133])
def test_bias_gradients_ascend(rows):
    print(f"case mlp bias order rows={rows}", flush=True)
    dims, batch = (2, 3, 5, 4), 2 ** int(np.ceil(np.log2(rows)))  # 1 / (batch x outputs) is a power of two
    n = batch * dims[3]
    v = np.zeros(batch, np.float32)
    v[:rows] = pattern(rows, 1)
    p, o = pack(dims, b3=200.0)  # every probability is 1
    net, _ = make_net(dims, batch, seed=rows)
    net.set_params(p)
    Y = np.repeat((1.0 - v * np.float32(n)).astype(np.float32)[:, None], dims[3], axis=1)
    assert np.array_equal((np.float32(1.0) - Y) / np.float32(n), np.repeat(v[:, None], dims[3], axis=1))
    g = net.gradients(np.zeros((batch, 2), np.float32), Y)[1]
    net.close()
    assert np.all(g[o["b3"]:o["n"]] == 0.0)
