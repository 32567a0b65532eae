"""Weight and bias gradients of convolutions with few weights over many positions (fp32), in slices of 64 samples of a position:
batches that fill a wavefront's samples, leave some of them out or take several wavefronts; one and two tiles of weights, up to
eight and up to sixteen filters; padding, strides and dilation; against the oracle in 64 bits (ConvKernelLayer.hpp:125-181)."""
import importlib

import numpy as np
import pytest

import helpers as hp
from oracle import oracle

pytestmark = pytest.mark.gpu

ch = importlib.import_module("c-attl3_amd")

# N, H, W, C, F, RH, RW, pv, ph, sv, sh, dv, dh
CASES = [(4, 9, 8, 1, 1, 3, 3, 1, 1, 1, 1, 0, 0), (60, 8, 9, 3, 3, 4, 4, 0, 0, 1, 1, 0, 0), (64, 12, 12, 3, 16, 3, 3, 1, 1, 1, 1, 0, 0),
         (68, 13, 11, 1, 3, 4, 4, 0, 0, 2, 2, 0, 0), (256, 13, 13, 3, 3, 4, 4, 0, 0, 1, 1, 0, 0), (512, 7, 7, 2, 9, 5, 5, 2, 2, 1, 1, 0, 0),
         (132, 10, 10, 16, 8, 2, 2, 0, 1, 1, 2, 0, 0), (96, 20, 20, 7, 5, 3, 3, 2, 2, 1, 1, 1, 1), (64, 6, 6, 33, 12, 1, 1, 0, 0, 1, 1, 0, 0)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(str(v) for v in c))
def test_gradients_of_few_weights(case):
    N, H, W, C, F, RH, RW, pv, ph, sv, sh, dv, dh = case
    gen = hp.rng(40 + N + C + F)
    x = hp.normal(gen, (N, H, W, C), np.float32)
    w = hp.normal(gen, (RH * RW * C, F), np.float32)
    OH, OW = hp.conv_dims(H, W, RH, RW, pv, ph, sv, sh, dv, dh)
    g = hp.normal(gen, (N, OH, OW, F), np.float32)
    layer = ch.ConvKernelLayer(np.float32, (H, W, C), F, RH, RW, pv, ph, sv, sh, dv, dh)
    wp, bp = layer.get_params()
    wp.set_values(w)
    layer.pass_forward(ch.DeviceTensor.from_host(x), True)
    layer.pass_back(ch.DeviceTensor.from_host(g))
    assert ch.last_launches()[1] == 4          # the launch that these cases are meant for, alone or in that of the input gradient
    geom = dict(RH=RH, RW=RW, pv=pv, ph=ph, sv=sv, sh=sh, dv=dv, dh=dh)
    x64, w64, g64, b64 = (np.asarray(a, np.float64) for a in (x, w, g, np.zeros((1, F))))
    _, cache = oracle.conv_forward(x64, w64, b64, return_cache=True, **geom)
    _, dw, db = oracle.conv_backward(x.shape, cache, w64, g64, **geom)
    # every sum against the sum of its magnitudes: a rounding per product and addition, in any order
    _, cache = oracle.conv_forward(np.abs(x64), w64, b64, return_cache=True, **geom)
    _, dw_mag, db_mag = oracle.conv_backward(x.shape, cache, w64, np.abs(g64), **geom)
    bound = (N * OH * OW + 2) * 2.0 ** -24
    assert np.all(np.abs(wp.get_grad() - dw) <= min(bound, 1e-5) * dw_mag)
    assert np.all(np.abs(bp.get_grad().reshape(np.shape(db)) - db) <= min(bound, 1e-5) * db_mag)
