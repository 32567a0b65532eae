"""Dense layers whose products and weight gradients are single launches without slices or cut reductions (fp32): row and column
counts around the 16- and 32-row tiles, reductions around a step of four, a wavefront's share and the most that is taken, batch
sizes that allow no pairs of rows and no 16-byte loads, batches that leave a wavefront of the weight gradient partly or
wholly without samples; against 64 bits (DenseKernelLayer.hpp:78-115)."""
import importlib

import numpy as np
import pytest

import helpers as hp
from oracle import oracle

pytestmark = pytest.mark.gpu

ch = importlib.import_module("c-attl3_amd")

# batch, inputs, outputs
CASES = [(1, 32, 1000), (2, 33, 17), (15, 61, 40), (16, 64, 16), (17, 100, 130), (31, 1000, 9), (33, 67, 33), (256, 784, 512),
         (255, 500, 513), (4, 3072, 48), (60, 35, 32), (64, 31, 64), (68, 96, 100), (508, 40, 36), (512, 33, 700), (512, 600, 96)]


SMALL, SMALL_ORDERED = 1, 2       # ch.last_launches(): the launches that these cases are meant for
# in front of a rectifier (the sums keep the order of the tiled launches): the others are few tiles of few reduction indices, or whole tiles
ORDERED = [(17, 100, 130), (31, 1000, 9), (256, 784, 512), (255, 500, 513), (512, 600, 96)]


def _bound(k):
    """Of a sum of k products relative to the sum of their magnitudes: a rounding per addition, in any order, and one per product."""
    return (k + 2) * 2.0 ** -24


@pytest.mark.parametrize("act", [None, "relu", "elu"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(str(v) for v in c))
def test_small_dense_layers(case, act):
    N, K, F = case
    gen = hp.rng(77 + N + K + F)
    x = hp.normal(gen, (N, K), np.float32)
    w = hp.normal(gen, (K, F), np.float32, std=1.0 / np.sqrt(K))
    b = hp.normal(gen, (1, F), np.float32)
    g = hp.normal(gen, (N, F), np.float32)
    dense = ch.DenseKernelLayer(np.float32, (K,), F)
    wp, bp = dense.get_params()
    wp.set_values(w)
    bp.set_values(b)
    (layer,) = ch.fuse_layers([dense] + ([ch.ActivationLayer(np.float32, act, (F,), 0.5)] if act else []))
    y = layer.pass_forward(ch.DeviceTensor.from_host(x), True).to_host()
    assert (ch.last_launches()[0] == SMALL_ORDERED) == bool(act and case in ORDERED)
    assert (ch.last_launches()[0] == SMALL) == bool(not act and K >= 32)
    dx = layer.pass_back(ch.DeviceTensor.from_host(g)).to_host()
    if act or case == (256, 784, 512):      # (the others' weight gradients are one-wavefront tiles that ride with the input gradient)
        assert (ch.last_launches()[0] == SMALL) == (F >= 32)
        assert (ch.last_launches()[1] == SMALL) == (F >= 32 and N % 4 == 0)
    dw, db = wp.get_grad(), bp.get_grad()
    x64, w64, g64 = (np.asarray(a, np.float64) for a in (x, w, g))
    z = x64 @ w64 + b
    y_ref = np.asarray(oracle.act_forward(act, z, 0.5)).reshape(N, F) if act else z
    size = np.abs(x64) @ np.abs(w64) + np.abs(b)
    assert np.all(np.abs(y.reshape(N, F) - y_ref) <= _bound(K + 1) * size + 4 * 2.0 ** -24)
    # where z is rounding noise around zero, its side, and with it the derivative, is the device's to choose: a slack of the gradient
    dz, slack = g64, np.zeros_like(g64)
    if act:
        dz = g64 * np.where(z < 0, 0.0 if act == "relu" else y_ref + 0.5, 1.0)
        slack = np.abs(g64) * (np.abs(z) <= _bound(K + 1) * size)
    # the derivative's own error: its roundings, and for elu that of the output it is formed from
    extra = 4 * 2.0 ** -24 + (_bound(K + 1) * float(size.max()) / 0.5 if act == "elu" else 0.0)
    ones = np.ones((1, N))
    for got, ref, mag, loose, n in ((dx, dz @ w64.T, np.abs(dz) @ np.abs(w64.T), slack @ np.abs(w64.T), F),
                                    (dw, x64.T @ dz, np.abs(x64.T) @ np.abs(dz), np.abs(x64.T) @ slack, N),
                                    (db, ones @ dz, ones @ np.abs(dz), ones @ slack, N)):
        assert np.all(np.abs(got.reshape(ref.shape) - ref) <= (_bound(n) + extra) * mag + loose)
    # a second pass over the same batch adds the same gradient
    layer.pass_forward(ch.DeviceTensor.from_host(x), True)
    layer.pass_back(ch.DeviceTensor.from_host(g))
    for again, once, n, mag in ((wp.get_grad(), dw, N, np.abs(x64.T) @ np.abs(dz)), (bp.get_grad(), db, N, np.abs(dz).sum(0, keepdims=True))):
        assert np.all(np.abs(again - 2.0 * once) <= 2 * _bound(n) * mag)


def test_non_finite_operands_stay_in_their_rows():
    """An infinity in one sample, or in one row of the weights, reaches no other sample and no reduction index past the last."""
    N, K, F = 18, 50, 20
    gen = hp.rng(5)
    x, w = hp.normal(gen, (N, K), np.float32), hp.normal(gen, (K, F), np.float32)
    x[17, K - 1] = np.inf
    x[3, 0] = np.nan
    dense = ch.DenseKernelLayer(np.float32, (K,), F)
    dense.get_params()[0].set_values(w)
    y = dense.pass_forward(ch.DeviceTensor.from_host(np.asfortranarray(x)), False).to_host().reshape(N, F)
    bad = np.zeros(N, bool)
    bad[[3, 17]] = True
    assert np.all(np.isfinite(y[~bad])) and not np.any(np.isfinite(y[bad]))


@pytest.mark.parametrize("inputs", [900, 2000])
def test_layers_behind_a_max_pool_keep_the_order_of_their_sums(inputs):
    """The order is asked for, not guessed from sizes: a dense layer alone takes the small launch, one behind a pool the sums of the
    tiled launches, which a training pass in front of a rectifier takes too."""
    N, F = 64, 10
    gen = hp.rng(inputs)
    x = ch.DeviceTensor.from_host(hp.normal(gen, (N, inputs), np.float32))
    w, b = hp.normal(gen, (inputs, F), np.float32), hp.normal(gen, (1, F), np.float32)
    dense = ch.DenseKernelLayer(np.float32, (inputs,), F)
    dense.get_params()[0].set_values(w)
    dense.get_params()[1].set_values(b)
    alone = dense.pass_forward(x, True).to_host()
    (rectified,) = ch.fuse_layers([dense, ch.ActivationLayer(np.float32, "relu", (F,))])
    tiled = rectified.pass_forward(x, True).to_host()
    assert np.array_equal(dense.pass_forward(x, True).to_host(), alone)
    pool = ch.MaxPoolLayer(np.float32, (4, inputs // 4, 4))
    assert ch.fuse_layers([pool, dense])[1] is dense
    behind = dense.pass_forward(x, True).to_host()
    positive = behind > 0
    assert np.array_equal(behind[positive], tiled[positive]) and not np.array_equal(behind, alone)
    ref = np.asarray(x.to_host(), np.float64) @ w.astype(np.float64) + b
    size = np.abs(x.to_host()) @ np.abs(w) + np.abs(b)
    for got in (alone, behind):
        assert np.all(np.abs(got - ref) <= _bound(inputs + 1) * size)
    dense.keep_sum_order(False)
    assert np.array_equal(dense.pass_forward(x, True).to_host(), alone)
