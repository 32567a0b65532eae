"""3 x 3 convolutions of up to six channels whose products a wavefront takes whole (fp32): odd channel counts (the last
reduction step is half empty), rows and columns that leave partial tiles, any batch size, padding and dilation, as a forward pass
and as the input gradient of a layer with few filters; against the oracle in 64 bits (ConvKernelLayer.hpp:125-181)."""
import importlib

import numpy as np
import pytest

import helpers as hp
from oracle import oracle

pytestmark = pytest.mark.gpu

ch = importlib.import_module("c-attl3_amd")

# N, H, W, C, F, pv, ph, dv, dh
CASES = [(64, 32, 32, 3, 16, 1, 1, 0, 0), (1, 5, 6, 1, 9, 1, 1, 0, 0), (33, 9, 7, 2, 33, 0, 0, 0, 0), (7, 12, 10, 5, 40, 2, 1, 1, 0), (32, 8, 8, 6, 64, 3, 4, 2, 3),
         (40, 10, 9, 12, 4, 1, 1, 0, 0), (5, 11, 8, 17, 6, 0, 2, 0, 1), (33, 10, 9, 12, 4, 1, 1, 0, 0)]
FEW_CHANNELS = 3        # ch.last_launches(): the launch that these cases are meant for


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(str(v) for v in c))
def test_convolutions_of_few_channels(case):
    N, H, W, C, F, pv, ph, dv, dh = case
    gen = hp.rng(60 + N + C + F)
    x = hp.normal(gen, (N, H, W, C), np.float32)
    w = hp.normal(gen, (9 * C, F), np.float32)
    b = hp.normal(gen, (1, F), np.float32)
    OH, OW = hp.conv_dims(H, W, 3, 3, pv, ph, 1, 1, dv, dh)
    g = hp.normal(gen, (N, OH, OW, F), np.float32)
    layer = ch.ConvKernelLayer(np.float32, (H, W, C), F, 3, 3, pv, ph, 1, 1, dv, dh)
    wp, bp = layer.get_params()
    wp.set_values(w)
    bp.set_values(b)
    out = layer.pass_forward(ch.DeviceTensor.from_host(x), True).to_host()
    assert (ch.last_launches()[0] == FEW_CHANNELS) == (C <= 6)
    dx = layer.pass_back(ch.DeviceTensor.from_host(g)).to_host()
    # the input gradients of few filters, where no weight gradient rides in their launch (it does at a multiple of four samples)
    assert (ch.last_launches()[0] == FEW_CHANNELS) == (F <= 6 and N % 4 != 0)
    geom = dict(RH=3, RW=3, pv=pv, ph=ph, sv=1, sh=1, dv=dv, dh=dh)
    x64, w64, b64, g64 = (np.asarray(a, np.float64) for a in (x, w, b, g))
    ref, cache = oracle.conv_forward(x64, w64, b64, return_cache=True, **geom)
    dx_ref = oracle.conv_backward(x.shape, cache, w64, g64, **geom)[0]
    mag, cache = oracle.conv_forward(np.abs(x64), np.abs(w64), np.abs(b64), return_cache=True, **geom)
    dx_mag = oracle.conv_backward(x.shape, cache, np.abs(w64), np.abs(g64), **geom)[0]
    # a rounding per product and addition, in any order, of the sum of the magnitudes
    assert np.all(np.abs(out - ref) <= (9 * C + 3) * 2.0 ** -24 * mag)
    assert np.all(np.abs(dx - dx_ref) <= (9 * F + 2) * 2.0 ** -24 * dx_mag)
