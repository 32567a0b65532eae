"""The gradient of the softmax cross entropy for as many classes as a thread holds at once, one more, and around its edges,
against the formula in 64 bits (loss/SoftmaxCrossEntropyLoss.hpp:33-50); samples in which one output stands far out."""
import importlib

import numpy as np
import pytest

import helpers as hp

pytestmark = pytest.mark.gpu

ch = importlib.import_module("c-attl3_amd")


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("N,T,V", [(1, 1, 1), (33, 1, 7), (32, 1, 8), (5, 3, 9), (40, 1, 31), (64, 2, 32), (31, 1, 33), (7, 1, 100)])
def test_gradient_around_the_classes_that_a_thread_holds(N, T, V, dtype):
    gen = hp.rng(V + N)
    out = np.asfortranarray(hp.normal(gen, (N, T, V), dtype) * np.asarray(3, dtype))
    out[0, 0, V - 1] = 40
    obj = np.zeros((N, T, V), dtype, order="F")
    for n in range(N):
        for t in range(T):
            obj[n, t, gen.integers(0, V)] = 1
    got = ch.loss_d_function("softmax_cross_entropy", ch.DeviceTensor.from_host(out), ch.DeviceTensor.from_host(obj), scale=0.25,
                             sequential=True).to_host()
    o = out.astype(np.float64)
    e = np.exp(o - o.max(2, keepdims=True))
    ref = 0.25 * (e / (e.sum(2, keepdims=True) + 1e-5) - obj)
    # exp to a few roundings plus the argument's own (up to 52 of them), V additions, a division and a subtraction, of values up to one
    assert np.max(np.abs(got - ref)) <= 0.25 * (60 + V) * float(np.finfo(dtype).eps)
