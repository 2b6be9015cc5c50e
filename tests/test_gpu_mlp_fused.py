"""The two-kernel form of the network at the edges of its tiles (16 samples,
16 columns, 32-deep products), the layer-by-layer form of networks that do
not fit it, and the update fused into the gradients."""
import numpy as np
import pytest

from oracle import mlp_oracle as mo

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def V():
    import inovesa_amd as V
    return V


def _rel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def _data(B, dims, seed=1):
    rng = np.random.default_rng(seed)
    return (rng.uniform(-1, 1, (B, dims[0])).astype(np.float32),
            rng.standard_normal((B, dims[-1] - 1)).astype(np.float32),
            (rng.random(B) > 0.5).astype(np.float32))


# the last three do not fit (activations, layers): layer by layer
NETS = [(3, 2), (1, 5, 2), (3, 48, 33, 9), (33, 100, 17), (40, 256, 300, 65),
        (3, 31, 32, 33, 16, 17, 64, 65, 3), (3, 1200, 1100, 9),
        (3, 1600, 5), (3, 8, 8, 8, 8, 8, 8, 8, 8, 4)]


@pytest.mark.parametrize("dims", NETS)
@pytest.mark.parametrize("B", [1, 16, 33])
def test_network_edges_match_oracle(V, dims, B):
    # bounds of test_gpu_mlp.py: one BF16 rounding of an activation that
    # falls to the other side is 2^-9 of it
    net = V.MLP(dims, max_batch=48, seed=3)
    x, t, lab = _data(B, dims, seed=B)
    layers = mo.split(net.params(), dims)
    ref, _ = mo.forward(layers, x, emulate=True)
    assert _rel(net.forward(x), ref) <= 2e-3
    loss = net.loss_grad(x, t, lab, 0.5)
    rloss, rg = mo.loss_and_grads(layers, x, t, lab, 0.5, emulate=True)
    assert loss == pytest.approx(rloss, rel=1e-3)
    for (dW, db), (rW, rb) in zip(net.layers(net.grads()), rg):
        assert _rel(dW, rW) <= 2e-2
        assert _rel(db, rb) <= 2e-2


def test_forward_beyond_the_staging(V):
    dims = (3, 64, 65)
    net = V.MLP(dims, max_batch=16000, seed=5)
    x, _, _ = _data(15500, dims)   # 4.2 MB of inputs and outputs
    y = net.forward(x)
    for k in (0, 1023, 1024, 15499):
        np.testing.assert_array_equal(y[k:k + 1], net.forward(x[k:k + 1]))


@pytest.mark.parametrize("B", [1030, 2100, 4200])
def test_samples_per_workgroup(V, B):
    """4, 8 and 16 samples per workgroup (by the batch and 256 CUs): the
    same sums per sample, so the same outputs as a small batch; gradients
    against the oracle."""
    dims = (3, 40, 17, 9)
    net = V.MLP(dims, max_batch=B, seed=7)
    x, t, lab = _data(B, dims, seed=2)
    y = net.forward(x)
    for k in (0, 500, B - 3):
        np.testing.assert_array_equal(y[k:k + 3], net.forward(x[k:k + 3]))
    loss = net.loss_grad(x, t, lab, 0.5)
    rloss, rg = mo.loss_and_grads(mo.split(net.params(), dims), x, t, lab, 0.5,
                                  emulate=True)
    assert loss == pytest.approx(rloss, rel=1e-3)
    for (dW, db), (rW, rb) in zip(net.layers(net.grads()), rg):
        assert _rel(dW, rW) <= 2e-2
        assert _rel(db, rb) <= 2e-2


@pytest.mark.parametrize("dims", [(3, 48, 33, 9), (3, 1200, 1100, 9)])
def test_train_is_gradients_and_adam(V, dims):
    """One update over the whole set, fused, against loss_grad + adam_step.
    The sums run over the samples in another order: gradients differ by a
    few 2^-24 of their terms, and Adam's first update is lr g / (|g| + eps),
    which only differs where |g| is itself of that size."""
    x, t, lab = _data(45, dims, seed=8)
    a = V.MLP(dims, max_batch=48, seed=6)
    b = V.MLP(dims, max_batch=48, seed=6)
    loss = a.train(x, t, lab, batch=45, epochs=1, lr=1e-3, seed=4)
    assert loss[0] == pytest.approx(b.loss_grad(x, t, lab), rel=1e-6)
    assert _rel(a.grads(), b.grads()) <= 1e-5
    b.adam_step(lr=1e-3)
    d = np.abs(a.params() - b.params())
    assert d.max() <= 2.1e-3 and d.mean() <= 1e-5
    # the padded copies follow the parameters
    c = V.MLP(dims, max_batch=48, seed=1)
    c.set_params(a.params())
    np.testing.assert_array_equal(a.forward(x), c.forward(x))


@pytest.mark.parametrize("dims,B", [((3, 40, 17, 9), 32), ((2, 33, 2), 64),
                                    ((5, 7), 256), ((3, 64, 40, 5), 512),
                                    ((3, 40, 17, 9), 2048),
                                    ((3, 32, 9), 4096),
                                    ((3, 1200, 1100, 9), 64)])
def test_bias_gradients_add_the_samples_in_order(V, dims, B):
    """A bias gradient is the FP32 sum of its column of dZ over the samples,
    one after another, in either form and for any split of the batch over
    workgroups.  dZ of a batch of B = 2^k samples is 1/B times the bias
    gradient of each sample alone, exactly: the scale enters at the outputs
    and every later operation carries a power of two through unchanged."""
    net = V.MLP(dims, max_batch=B, seed=9)
    x, t, lab = _data(B, dims, seed=B)
    rows = []
    for k in range(B):
        net.loss_grad(x[k:k + 1], t[k:k + 1], lab[k:k + 1], 0.5)
        rows.append(np.concatenate([db for _, db in net.layers(net.grads())]))
    dz = np.array(rows, np.float32) / np.float32(B)
    ref = np.add.accumulate(dz, axis=0, dtype=np.float32)[-1]
    net.loss_grad(x, t, lab, 0.5)
    got = np.concatenate([db for _, db in net.layers(net.grads())])
    np.testing.assert_array_equal(got, ref)


@pytest.mark.parametrize("dims", [(3, 48, 33, 9), (3, 40, 64, 40, 5),
                                  (3, 64, 32, 9), (3, 1200, 1100, 9)])
def test_overflow_stays_infinite(V, dims):
    """An activation or gradient that overflows is an infinity in what
    follows from it, also where a width is no whole number of fragments and
    zero weights meet it in the columns between.  All weights, inputs and
    biases are positive, so no infinity meets its opposite or a zero."""
    net = V.MLP(dims, max_batch=40, seed=1)
    rng = np.random.default_rng(2)
    p = (0.01 + 0.01 * rng.random(net.params().size)).astype(np.float32)
    big = p.copy()
    big[:dims[0]] = 3e38            # the first hidden unit's weights
    net.set_params(big)
    x = np.full((20, dims[0]), 1e-30, np.float32)
    x[7] = 1.0
    y = net.forward(x)
    assert np.all(np.isposinf(y[7]))
    assert np.all(np.isfinite(np.delete(y, 7, axis=0)))
    # a target far away: the output gradient overflows
    net.set_params(p)
    x[:] = 0.5
    t = np.zeros((20, dims[-1] - 1), np.float32)
    t[7] = -3e38
    net.loss_grad(x, t, np.zeros(20, np.float32))
    for l, (dW, db) in enumerate(net.layers(net.grads())):
        # (not the row of the label, whose gradient is finite)
        out = slice(None, -1 if l + 2 == len(dims) else None)
        assert np.all(np.isposinf(dW[out])) and np.all(np.isposinf(db[out]))


@pytest.mark.parametrize("dims", [(3, 2), (1, 5, 2), (3, 48, 33, 9),
                                  (33, 100, 17), (3, 256, 256, 65),
                                  (3, 1200, 1100, 9)])
def test_adam_step_updates_the_operands(V, dims):
    """adam_step alone: the parameters by Adam's formula (two steps, FP32), and
    the BF16 copies that the products read follow them."""
    x, t, lab = _data(20, dims, seed=3)
    net = V.MLP(dims, max_batch=32, seed=2)
    m = v = np.zeros(net.params().size)
    for step in (1, 2):
        net.loss_grad(x, t, lab)
        p, g = net.params().astype(np.float64), net.grads().astype(np.float64)
        net.adam_step(lr=1e-2)
        m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
        ref = p - 1e-2 * (m / (1 - 0.9 ** step)) / (
            np.sqrt(v / (1 - 0.999 ** step)) + 1e-8)
        # an update is at most lr here and is made of a dozen FP32 operations
        # (1 - 0.999^t, a difference of near equals, carries the most: 6e-5)
        assert np.abs(net.params() - ref).max() <= 1e-2 * 1e-4 + 2.0**-23 * 4
    other = V.MLP(dims, max_batch=32, seed=5)
    other.set_params(net.params())
    np.testing.assert_array_equal(net.forward(x), other.forward(x))
    net.loss_grad(x, t, lab)
    other.loss_grad(x, t, lab)
    np.testing.assert_array_equal(net.grads(), other.grads())
