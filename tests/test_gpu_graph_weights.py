"""Recorded passes whose weights change between the launches: by set_values, by the optimizer calls of one and of many parameters, by
constraints set after the recording, by an optimizer inside another recorded step; with eager passes of the same layer in between. The
layers keep re-laid-out copies of their weights, and a launch must work on the values as they are whichever of these copies
were current when it was recorded. Every launch is held against the eager calls of a twin, bit for bit (same kernels, same
arguments, same order)."""
import importlib

import numpy as np
import pytest

import helpers as hp

pytestmark = pytest.mark.gpu

ch = importlib.import_module("c-attl3_amd")

DT = np.float32


class _Net(object):
    """One layer with weights, its input and an output gradient, on the device."""

    MAKE = {"conv": lambda: ch.ConvKernelLayer(DT, (8, 8, 4), 8), "dense": lambda: ch.DenseKernelLayer(DT, (64,), 64),
            "fused": lambda: ch.FusedKernelLayer([ch.ConvKernelLayer(DT, (8, 8, 4), 8), ch.ActivationLayer(DT, "relu", (8, 8, 8))]),
            # large enough for the input gradient that goes by the residue classes of the stride
            "strided": lambda: ch.ConvKernelLayer(DT, (32, 32, 32), 96, vertical_stride=2, horizontal_stride=2),
            "transposed": lambda: ch.TransConvKernelLayer(DT, (6, 6, 4), 4, 4, 4, 0, 0),
            "convlstm": lambda: ch.ConvLSTMNetwork(DT, (6, 6, 4), 8, foremost=False)}
    KINDS = tuple(MAKE)

    def __init__(self, kind, seed=11):
        self.kind, self.seed = kind, seed
        self.layer = self.MAKE[kind]()
        self.recurrent = kind == "convlstm"
        self.owner = self.layer.members[0] if kind == "fused" else self.layer
        self.params = self.owner.get_params()
        self.list = ch.ParameterList(self.params)
        self.set_weights(0)
        self.x, self.g = self.data(64 if kind == "strided" else 16)
        self.half = self.data(32 if kind == "strided" else 8)

    def data(self, N):
        gen = hp.rng(self.seed)
        lead = (N, 3) if self.recurrent else (N,)
        return tuple(ch.DeviceTensor.from_host(hp.normal(gen, lead + tuple(d), DT))
                     for d in (self.layer.get_input_dims(), self.layer.get_output_dims()))

    def set_weights(self, k):
        gen = hp.rng(1000 * self.seed + k)
        if self.recurrent:
            for i in range(8):
                w, _ = self.layer.kernel_params(i)
                w.set_values(hp.uniform(gen, (w.get_rows(), w.get_cols()), -0.3, 0.3, DT))
        else:
            w = self.params[0]
            w.set_values(hp.uniform(gen, (w.get_rows(), w.get_cols()), -0.3, 0.3, DT))

    def passes(self, x=None, g=None):
        x, g = x or self.x, g or self.g
        if self.recurrent:
            out = self.layer.propagate(x)
            return out, self.layer.backpropagate(g)
        out = self.layer.pass_forward(x, True)
        return out, self.layer.pass_back(g)

    def outcome(self, tensors):
        """On the host: outputs, input gradient, gradients (reset afterwards) and values."""
        got = [t.to_host() for t in tensors] + [p.get_grad() for p in self.params] + [p.get_values() for p in self.params]
        for p in self.params:
            p.reset_grad()
        return got


def _same(got, want, what):
    for i, (a, b) in enumerate(zip(got, want)):
        assert np.array_equal(a, b), "%s: result %d" % (what, i)


def _by_set_values(net, k):
    net.set_weights(k + 1)


def _by_single_updates(net, k):
    net.passes()
    for p in net.params:
        p.optimizer_step("vanilla_sgd", [1e-3])


def _by_constraints(net, k):
    net.params[0].set_constraints(value_clip=0.2 / (k + 1))


def _by_constrained_steps(net, k):
    net.params[0].set_constraints(value_clip=0.2)
    net.passes()
    net.list.optimizer_step("vanilla_sgd", [1e-3])


def _by_steps_at_another_batch_size(net, k):
    net.passes(*net.half)
    net.list.optimizer_step("vanilla_sgd", [1e-3])
    net.passes(*net.half)
    for p in net.params:
        p.reset_grad()


CHANGES = [_by_set_values, _by_single_updates, _by_constraints, _by_constrained_steps, _by_steps_at_another_batch_size]


@pytest.mark.parametrize("change", CHANGES, ids=lambda f: f.__name__[1:])
@pytest.mark.parametrize("kind", _Net.KINDS)
def test_a_launch_works_on_the_values_as_they_are(kind, change):
    if kind == "convlstm" and change in (_by_constraints, _by_constrained_steps):
        pytest.skip("a recurrent network takes no constraints")
    twin, net = _Net(kind), _Net(kind)
    for n in (twin, net):
        # a step, so that the optimizer's kernel keeps what it keeps, and a pass, so that everything is current
        n.passes()
        n.list.optimizer_step("vanilla_sgd", [1e-3])
        n.outcome(n.passes(*n.half))
        n.outcome(n.passes())
    with ch.Graph() as graph:
        recorded = net.passes()
    for k in range(3):
        change(twin, k)
        change(net, k)
        want = twin.outcome(twin.passes())
        graph.launch()
        _same(net.outcome(recorded), want, "launch %d after the change" % k)
        # an ordinary step from here on must be followed as well
        for n in (twin, net):
            n.list.optimizer_step("vanilla_sgd", [1e-3])
        want = twin.outcome(twin.passes())
        graph.launch()
        _same(net.outcome(recorded), want, "launch %d after a step behind the change" % k)
    graph.destroy()


@pytest.mark.parametrize("kind", _Net.KINDS)
def test_a_recording_prepares_nothing_for_eager_passes(kind):
    """The re-layouts that a recording holds have not run when it ends: an eager pass before the first launch makes its own."""
    twin, net = _Net(kind), _Net(kind)
    for n in (twin, net):
        n.outcome(n.passes())
        n.set_weights(5)
    with ch.Graph() as graph:
        recorded = net.passes()
    want = twin.outcome(twin.passes())
    _same(net.outcome(net.passes()), want, "eager pass before the first launch")
    graph.launch()
    _same(net.outcome(recorded), want, "first launch")
    for n in (twin, net):
        n.set_weights(6)
    want = twin.outcome(twin.passes())
    graph.launch()
    _same(net.outcome(recorded), want, "second launch")
    _same(net.outcome(net.passes()), want, "eager pass after it")
    graph.destroy()


@pytest.mark.parametrize("constrained", [False, True])
@pytest.mark.parametrize("kind", _Net.KINDS)
def test_eager_passes_follow_an_optimizer_on_a_graph(kind, constrained):
    """A recorded step moves the values at every launch: eager passes between the launches, and a second recording of passes
    alone, see them as they have become."""
    if kind == "convlstm" and constrained:
        pytest.skip("a recurrent network takes no constraints")
    twin, net = _Net(kind), _Net(kind)

    def step(n):
        n.passes()
        n.list.optimizer_step("vanilla_sgd", [1e-3])

    for n in (twin, net):
        if constrained:
            n.params[0].set_constraints(value_clip=0.25)
        step(n)
        n.outcome(n.passes())
    with ch.Graph() as passes:
        recorded = net.passes()
    with ch.Graph() as training:
        step(net)
    for k in range(3):
        step(twin)
        training.launch()
        want = twin.outcome(twin.passes())
        if k != 1:
            _same(net.outcome(net.passes()), want, "eager pass after launch %d" % k)
        passes.launch()
        _same(net.outcome(recorded), want, "recorded passes after launch %d" % k)
    passes.destroy()
    training.destroy()


def test_recurrent_steps_of_two_gate_orders():
    """The launch over few rows and the one over many want the recurrent weights' gates in blocks of different sizes, in one
    buffer: a network that runs at both batch sizes, eagerly and recorded."""
    hidden, side, T = 32, 16, 2
    net = ch.ConvLSTMNetwork(DT, (side, side, 4), hidden)
    gen = hp.rng(3)
    for k in range(8):
        w, _ = net.kernel_params(k)
        w.set_values(hp.uniform(gen, (w.get_rows(), hidden), -0.3, 0.3, DT))
    data = {N: ch.DeviceTensor.from_host(hp.normal(gen, (N, T, side, side, 4), DT)) for N in (200, 192, 8)}
    want = {}
    for N in data:
        want[N] = net.propagate(data[N], False).to_host()
        assert net.fused_steps()[0] == T - 1
        assert np.array_equal(net.propagate(data[N], False).to_host(), want[N])
    # the same samples in another batch, computed in the other order: the same to rounding, here a bound on sums of 9 x 32 products
    # of values below one through gates of slope one or less
    few = ch.DeviceTensor.from_host(np.asfortranarray(data[200].to_host()[:8]))
    assert np.max(np.abs(net.propagate(few, False).to_host() - want[200][:8])) <= 4 * (9 * hidden + 2) * 2.0 ** -24 * 9 * hidden * 0.3
    graphs = {}
    for N in data:
        net.propagate(data[N], False)
        with ch.Graph() as graphs[N]:
            want[N, "recorded"] = net.propagate(data[N], False)
    for N in (192, 200, 8, 200, 192, 192, 8):
        graphs[N].launch()
        assert np.array_equal(want[N, "recorded"].to_host(), want[N]), "launch at batch size %d" % N
        other = 200 if N != 200 else 8
        assert np.array_equal(net.propagate(data[other], False).to_host(), want[other]), "eager pass at batch size %d" % other
    for g in graphs.values():
        g.destroy()
