"""Gradients that were reset, through everything that may come next: a read, a backward pass (which overwrites them), two (of
which the second adds), an optimizer step with and without a pass in front of it, one of the two resets only, a clone, a recorded
step launched after eager resets; weight gradients cut into slices and written at once, convolution, dense and recurrent."""
import importlib

import numpy as np
import pytest

import helpers as hp

pytestmark = pytest.mark.gpu

ch = importlib.import_module("c-attl3_amd")

DENSE, SLICES, WHOLE = "dense", "convolution in slices", "convolution in one piece"


def _layer(kind, dtype):
    gen = hp.rng(3)
    if kind == DENSE:
        layer, shape = ch.DenseKernelLayer(dtype, (70,), 40), (24, 70)
    elif kind == SLICES:
        layer, shape = ch.ConvKernelLayer(dtype, (16, 16, 4), 8), (32, 16, 16, 4)
    else:
        layer, shape = ch.ConvKernelLayer(dtype, (3, 3, 40), 200), (4, 3, 3, 40)
    p = layer.get_params()
    p[0].set_values(hp.normal(gen, (p[0].get_rows(), p[0].get_cols()), dtype))
    x = hp.normal(gen, shape, dtype)
    g = hp.normal(gen, (shape[0],) + tuple(layer.get_output_dims()), dtype)
    return layer, p, ch.DeviceTensor.from_host(x), ch.DeviceTensor.from_host(g)


def _pass(layer, x, g):
    layer.pass_forward(x, True)
    layer.pass_back(g)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("kind", [DENSE, SLICES, WHOLE])
def test_what_follows_a_reset(kind, dtype):
    layer, p, x, g = _layer(kind, dtype)
    _pass(layer, x, g)
    once = [q.get_grad() for q in p]
    assert all(np.any(o != 0) for o in once)
    for q in p:
        q.reset_grad()
    assert all(np.all(q.get_grad() == 0) for q in p)                     # a read
    for q in p:
        q.reset_grad()
    _pass(layer, x, g)                                                   # a pass overwrites
    assert all(np.array_equal(q.get_grad(), o) for q, o in zip(p, once))
    for q in p:
        q.reset_grad()
    _pass(layer, x, g)
    _pass(layer, x, g)                                                   # the second adds
    tol = 8 * float(np.finfo(dtype).eps)
    assert all(np.allclose(q.get_grad(), 2 * o, rtol=tol, atol=tol * np.abs(o).max()) for q, o in zip(p, once))
    p[1].reset_grad()                                                    # one of the two
    _pass(layer, x, g)
    assert np.array_equal(p[1].get_grad(), once[1])
    assert np.allclose(p[0].get_grad(), 3 * once[0], rtol=2 * tol, atol=2 * tol * np.abs(once[0]).max())
    for q in p:
        q.reset_grad()
    clone = layer.clone()                                                # a deep copy has a gradient of zero, and one of its own
    assert all(np.all(q.get_grad() == 0) for q in clone.get_params())
    before = [q.get_values() for q in p]
    ch.ParameterList(p).optimizer_step("vanilla_sgd", (0.5,))            # a step on a gradient of zero
    assert all(np.array_equal(q.get_values(), b) for q, b in zip(p, before))
    _pass(layer, x, g)
    ch.ParameterList(p).optimizer_step("vanilla_sgd", (0.5,))
    eps = float(np.finfo(dtype).eps)
    for q, b, o in zip(p, before, once):
        assert np.all(np.abs(q.get_values() - (b - 0.5 * o)) <= 4 * eps * (np.abs(b) + np.abs(o)))
        assert np.all(q.get_grad() == 0)


def test_a_gradient_read_on_the_device_from_the_launch_that_sums_it():
    layer, p, x, g = _layer(SLICES, np.float32)
    _pass(layer, x, g)
    want = [q.get_grad() for q in p]
    for order in ((0, 1), (1, 0)):
        for q in p:
            q.reset_grad()
        _pass(layer, x, g)
        into = [ch.DeviceTensor((q.get_rows(), q.get_cols()), np.float32) for q in p]
        for i in order:
            assert ch.lib().cattle_hip_layer_get_param_grad(p[i]._layer._h, ch.binding._sz(i), into[i].ptr, ch.DEVICE) == 0
        for t, q, w in zip(into, p, want):
            assert np.array_equal(t.to_host(), w) and np.array_equal(q.get_grad(), w)


def test_resets_and_recorded_passes():
    """A recorded forward and backward pass adds to what is there; eager resets between launches hold."""
    layer, p, x, g = _layer(SLICES, np.float32)
    _pass(layer, x, g)
    once = [q.get_grad() for q in p]
    for q in p:
        q.reset_grad()
    with ch.Graph() as graph:
        _pass(layer, x, g)
    assert all(np.all(q.get_grad() == 0) for q in p)
    graph.launch()
    assert all(np.array_equal(q.get_grad(), o) for q, o in zip(p, once))
    graph.launch()
    assert all(np.allclose(q.get_grad(), 2 * o, rtol=1e-5, atol=1e-5 * np.abs(o).max()) for q, o in zip(p, once))
    for q in p:
        q.reset_grad()
    graph.launch()
    assert all(np.array_equal(q.get_grad(), o) for q, o in zip(p, once))
    for q in p:
        q.reset_grad()
    _pass(layer, x, g)                  # eager, then a launch that adds
    graph.launch()
    assert all(np.allclose(q.get_grad(), 2 * o, rtol=1e-5, atol=1e-5 * np.abs(o).max()) for q, o in zip(p, once))


@pytest.mark.parametrize("kind", [DENSE, SLICES, WHOLE])
def test_recorded_passes_with_the_optimizer_outside(kind):
    """Marked before the recording, zeroed by the optimizer while the graph lives, marked again once it is destroyed: each step
    starts from zero gradients, as the same steps without a recording do (sums of parts may be rounded in another order: 1e-5)."""
    layer, p, x, g = _layer(kind, np.float32)
    twin, tp, tx, tg = _layer(kind, np.float32)
    params, tparams = ch.ParameterList(p), ch.ParameterList(tp)

    def same():
        for q, t in zip(p, tp):
            v = t.get_values()
            assert np.allclose(q.get_values(), v, rtol=1e-5, atol=1e-5 * np.abs(v).max())

    def eager(n):
        for _ in range(n):
            _pass(layer, x, g)
            params.optimizer_step("vanilla_sgd", [1e-3])
    eager(2)
    with ch.Graph() as graph:
        _pass(layer, x, g)
    for _ in range(3):
        graph.launch()
        params.optimizer_step("vanilla_sgd", [1e-3])
    assert all(np.all(q.get_grad() == 0) for q in p)
    eager(1)
    graph.launch()
    params.optimizer_step("vanilla_sgd", [1e-3])
    graph.destroy()
    eager(2)
    assert all(np.all(q.get_grad() == 0) for q in p)
    for _ in range(9):
        _pass(twin, tx, tg)
        tparams.optimizer_step("vanilla_sgd", [1e-3])
    same()


def test_a_recurrent_network():
    net = ch.ConvLSTMNetwork(np.float32, (4, 4, 2), 8)
    gen = hp.rng(9)
    for k in range(8):
        w = net.kernel_params(k)[0]
        w.set_values(hp.normal(gen, (w.get_rows(), w.get_cols()), np.float32, 0.2))
    x, g = hp.normal(gen, (4, 3, 4, 4, 2), np.float32), hp.normal(gen, (4, 3, 4, 4, 8), np.float32)
    net.propagate(x)
    net.backpropagate(g)
    once = [q.get_grad() for q in net.get_params()]
    for q in net.get_params():
        q.reset_grad()
    net.propagate(x)
    net.backpropagate(g)
    assert all(np.array_equal(q.get_grad(), o) for q, o in zip(net.get_params(), once))
    for q in net.get_params():
        q.reset_grad()
    assert all(np.all(net.kernel_params(k)[b].get_grad() == 0) for k in range(8) for b in (0, 1))
