"""The surrogate's products at the edges of their blocks (32/64 rows, 64
columns, 16-deep steps, eight wavefronts over K): outputs, loss and gradients
of ragged networks against the fp32 PyTorch reference of test_gpu_mlp.py, at
its tolerances (the same BF16 roundings bound both)."""
import numpy as np
import pytest

from test_gpu_mlp import torch_reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,batch", [
    ((1, 1, 1, 1), 1),
    ((15, 17, 16, 2), 31),
    ((63, 65, 64, 1), 32),
    ((64, 96, 33, 65), 33),
    ((127, 128, 129, 64), 64),
    ((200, 130, 70, 193), 127),
    ((16, 640, 40, 130), 65),
])
def test_ragged_shapes_match_torch(dims, batch):
    from lightning_unification_amd import capi
    rs = np.random.default_rng(batch)
    net = capi.Mlp(dims, max_batch=batch, seed=11)
    p = net.params()
    p += rs.uniform(-0.1, 0.1, p.size).astype(np.float32)  # non-zero biases
    net.set_params(p)
    x = rs.uniform(-1, 1, (batch, dims[0])).astype(np.float32)
    t = rs.normal(size=(batch, dims[3])).astype(np.float32)
    w = rs.uniform(0.5, 1.5, dims[3]).astype(np.float32)
    net.set_loss_weights(w)
    y_ref, loss_ref, g_ref = torch_reference(net, p, x, t, w)
    assert np.max(np.abs(net.predict(x) - y_ref)) < 2e-3 * np.max(np.abs(y_ref))
    loss, g = net.gradients(x, t)
    assert abs(loss - loss_ref) < 1e-3 * loss_ref
    o = 0
    for l in range(3):
        for size in (dims[l] * dims[l + 1], dims[l + 1]):
            a, r = g[o:o + size], g_ref[o:o + size]
            o += size
            assert np.max(np.abs(a - r)) < 3e-2 * np.max(np.abs(r)), (l, size)
    net.close()


def test_rows_past_the_batch_stay_out():
    """A minibatch's blocks read rows of its neighbours; none of their values
    may reach the step, whatever they are.  One training step on the first 33
    rows equals the same step with NaN in every other row."""
    from lightning_unification_amd import capi
    rs = np.random.default_rng(5)
    dims, b = (20, 48, 64, 21), 33
    x = rs.uniform(-1, 1, (3 * b, dims[0])).astype(np.float32)
    t = rs.normal(size=(3 * b, dims[3])).astype(np.float32)
    got = []
    for fill in (0.0, np.nan):
        x[b:], t[b:] = fill, fill
        net = capi.Mlp(dims, max_batch=b, seed=2)
        net.load_data(x, t)
        loss = net.train(1, b, 1e-3)
        got.append((loss, net.params()))
        net.close()
    assert np.isfinite(got[1][0]) and got[0][0] == got[1][0]
    assert np.array_equal(got[0][1], got[1][1])


@pytest.mark.parametrize("seed", range(4))
def test_initial_weights_are_in_place(seed):
    """A network answers from its initial weights as soon as it exists."""
    from lightning_unification_amd import capi
    dims, b = (192, 512, 512, 193), 64
    x = np.random.default_rng(seed).uniform(-1, 1, (b, dims[0])).astype(np.float32)
    net = capi.Mlp(dims, max_batch=b, seed=seed)
    y = net.predict(x)
    y_ref = torch_reference(net, net.params(), x, np.zeros((b, dims[3]), np.float32), np.ones(dims[3], np.float32))[0]
    assert np.max(np.abs(y - y_ref)) < 2e-3 * np.max(np.abs(y_ref))
    net.close()


def test_an_overflowed_activation_stays_infinite():
    """All weights positive and one hidden value past the largest float: its
    row's outputs are +inf as the product has them, not NaN from the zeros that
    widths of 17 are padded with; the other rows are untouched."""
    from lightning_unification_amd import capi
    dims, b = (3, 17, 17, 5), 33
    net = capi.Mlp(dims, max_batch=b, seed=3)
    p = np.full(net.params().size, 0.25, np.float32)
    p[:dims[1]] = 0.0
    p[0] = 16.0  # feature 0 reaches hidden value 0 only
    net.set_params(p)
    x = np.full((b, 3), 0.5, np.float32)
    x[7, 0] = 3e38
    y = net.predict(x)
    x[7, 0] = 0.5
    ref = torch_reference(net, p, x, np.zeros((b, 5), np.float32), np.ones(5, np.float32))[0]
    assert np.all(np.isposinf(y[7]))
    rest = np.arange(b) != 7
    assert np.max(np.abs(y[rest] - ref[rest])) < 2e-3 * np.max(np.abs(ref))
    net.close()
