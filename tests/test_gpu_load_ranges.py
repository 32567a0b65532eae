"""Loads at the ends of the operands: the kernels that fetch straight into the matrix instructions' registers choose, lane by lane, between
an offset inside the operand and one beyond any buffer. On the CPU the offsets of the 3 x 3 products are checked over small problems
(sides of one and two, paddings, dilations, odd channel counts); on the GPU shapes whose last rows, reduction indices, channels and
taps have no operand, with operands between values that are not numbers, against 64 bits."""
import ctypes
import importlib
import os
import shutil
import subprocess

import numpy as np
import pytest

import helpers as hp
from oracle import oracle

ch = importlib.import_module("c-attl3_amd")
HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
def test_offsets_of_tap_products(tmp_path):
    exe = str(tmp_path / "tap_ranges")
    subprocess.check_call([HIPCC, "-std=c++17", "-O1", "--offload-arch=gfx950", "--offload-host-only", "-I" + os.path.join(HERE, "..", "c-attl3_amd", "csrc"),
                           "-I" + os.path.join(HERE, "..", "include"), os.path.join(HERE, "compat", "tap_ranges.hip"), "-o", exe])
    run = subprocess.run([exe], stdout=subprocess.PIPE, universal_newlines=True, timeout=60)
    assert run.returncode == 0 and "all in range" in run.stdout, run.stdout[-2000:]


class _Between(object):
    """A device tensor with a kilobyte of NaN before it and behind it."""

    PAD = 256

    def __init__(self, values):
        self.shape = values.shape
        block = np.full(values.size + 2 * self.PAD, np.nan, np.float32)
        block[self.PAD:self.PAD + values.size] = values.reshape(-1, order="F")
        self._block = ch.DeviceTensor.from_host(block)
        self.ptr = ctypes.c_void_p(self._block.ptr.value + 4 * self.PAD)


def _within(got, ref, mag, terms):
    """A rounding per product and addition, in any order, of the sum of the magnitudes."""
    return bool(np.all(np.abs(got - ref) <= (terms + 3) * 2.0 ** -24 * mag))


# batch, inputs, outputs: fewer inputs than a tile of the weight gradient has; a remainder of the reduction's steps; fewer rows than a
# block, of one and of two row blocks; the kernel that keeps the order of the sums (training, behind a rectifier)
DENSE = [(4, 1, 32), (4, 3, 40), (36, 20, 33), (512, 23, 64), (256, 5, 40), (7, 33, 40), (5, 35, 4100), (33, 50, 4000), (1, 97, 10), (30, 66, 48), (17, 100, 130)]


@pytest.mark.gpu
@pytest.mark.parametrize("act", [False, True])
@pytest.mark.parametrize("case", DENSE, ids=lambda c: "x".join(str(v) for v in c))
def test_dense_layers(case, act):
    N, K, F = case
    gen = hp.rng(N + K + F)
    x, w, b, g = hp.normal(gen, (N, K), np.float32), hp.normal(gen, (K, F), np.float32), hp.normal(gen, (1, F), np.float32), hp.normal(gen, (N, F), np.float32)
    dense = ch.DenseKernelLayer(np.float32, (K,), F)
    dense.get_params()[0].set_values(w)
    dense.get_params()[1].set_values(b)
    (layer,) = ch.fuse_layers([dense] + ([ch.ActivationLayer(np.float32, "relu", (F,))] if act else []))
    out, dx = ch.DeviceTensor((N, F), np.float32), ch.DeviceTensor((N, K), np.float32)
    xd, gd = _Between(x), _Between(g)
    # (ch.last_launches(): the launches that these cases are meant for)
    layer.forward_into(xd, out)
    assert ch.last_products()[0] == 0       # none of them is a tile on the bf16 instructions
    assert ch.last_launches()[0] == ((2 if case == (17, 100, 130) else 0) if act else 1 if K >= 32 else 0)
    layer.backward_into(gd, dx)
    if act:
        assert ch.last_launches() == (1 if 32 <= F <= 3072 else 0, 1 if F >= 32 and N % 4 == 0 else 0)
    y = out.to_host()
    x64, w64, g64 = (np.asarray(a, np.float64) for a in (x, w, g))
    z, size = x64 @ w64 + b, np.abs(x64) @ np.abs(w64) + np.abs(b)
    assert _within(y, np.maximum(z, 0.0) if act else z, size, K + 1)
    if act:
        g64 = g64 * (y > 0)
    assert _within(dx.to_host(), g64 @ w64.T, np.abs(g64) @ np.abs(w64.T), F)
    assert _within(dense.get_params()[0].get_grad(), x64.T @ g64, np.abs(x64.T) @ np.abs(g64), N)
    assert _within(dense.get_params()[1].get_grad().ravel(), g64.sum(0), np.abs(g64).sum(0), N)


# N, H, W, C, F, pv, ph, dv, dh: sides of one and two, with odd and even channel counts; larger images whose last pair lacks a channel
CONV = [(33, 9, 1, 1, 16, 1, 1, 0, 0), (32, 1, 9, 1, 16, 1, 1, 0, 0), (16, 1, 1, 5, 12, 1, 1, 0, 0), (16, 1, 1, 4, 12, 1, 1, 0, 0), (12, 2, 2, 3, 24, 2, 2, 1, 1),
        (12, 2, 2, 3, 24, 1, 1, 0, 0), (8, 30, 1, 3, 9, 2, 1, 1, 0), (21, 7, 5, 3, 33, 1, 1, 0, 0), (64, 12, 12, 1, 10, 1, 1, 0, 0), (5, 9, 8, 5, 16, 2, 0, 0, 0),
        (16, 9, 1, 12, 5, 1, 1, 0, 0)]
# the last tap of a lone last channel reaches past the image
TILED = [(33, 9, 1, 1, 16, 1, 1, 0, 0), (16, 1, 1, 5, 12, 1, 1, 0, 0), (12, 2, 2, 3, 24, 2, 2, 1, 1), (8, 30, 1, 3, 9, 2, 1, 1, 0)]


@pytest.mark.gpu
@pytest.mark.parametrize("case", CONV, ids=lambda c: "x".join(str(v) for v in c))
def test_convolutions(case):
    N, H, W, C, F, pv, ph, dv, dh = case
    geom = dict(RH=3, RW=3, pv=pv, ph=ph, sv=1, sh=1, dv=dv, dh=dh)
    OH, OW = hp.conv_dims(H, W, 3, 3, pv, ph, 1, 1, dv, dh)
    gen = hp.rng(N + C + F)
    x, w, b, g = (hp.normal(gen, s, np.float32) for s in ((N, H, W, C), (9 * C, F), (1, F), (N, OH, OW, F)))
    layer = ch.ConvKernelLayer(np.float32, (H, W, C), F, 3, 3, pv, ph, 1, 1, dv, dh)
    layer.get_params()[0].set_values(w)
    layer.get_params()[1].set_values(b)
    out, dx = ch.DeviceTensor(g.shape, np.float32), ch.DeviceTensor(x.shape, np.float32)
    xd, gd = _Between(x), _Between(g)
    layer.forward_into(xd, out)
    assert (ch.last_launches()[0] == 3) == (C <= 6 and case not in TILED)
    layer.backward_into(gd, dx)
    x64, w64, b64, g64 = (np.asarray(a, np.float64) for a in (x, w, b, g))
    ref, cache = oracle.conv_forward(x64, w64, b64, return_cache=True, **geom)
    dx_ref, dw_ref, db_ref = oracle.conv_backward(x.shape, cache, w64, g64, **geom)
    mag, cache = oracle.conv_forward(np.abs(x64), np.abs(w64), np.abs(b64), return_cache=True, **geom)
    dx_mag, dw_mag, db_mag = oracle.conv_backward(x.shape, cache, np.abs(w64), np.abs(g64), **geom)
    assert _within(out.to_host(), ref, mag, 9 * C) and _within(dx.to_host(), dx_ref, dx_mag, 9 * F)
    assert _within(layer.get_params()[0].get_grad(), dw_ref, dw_mag, N * OH * OW)
    assert _within(layer.get_params()[1].get_grad().reshape(np.shape(db_ref)), db_ref, db_mag, N * OH * OW)


@pytest.mark.gpu
@pytest.mark.parametrize("side", [(9, 1), (1, 1), (2, 2), (5, 4)], ids=str)
def test_recurrent_steps_on_small_images(side):
    """Against the same network in 64 bits on the device, which has kernels of its own."""
    H, W = side
    gen = hp.rng(H + W)
    x = hp.normal(gen, (8, 3, H, W, 2), np.float32)
    got = []
    for dtype in (np.float32, np.float64):
        net = ch.ConvLSTMNetwork(dtype, (H, W, 2), 8, foremost=False)
        wgen = hp.rng(5)
        for k in range(8):
            w, _ = net.kernel_params(k)
            w.set_values(hp.uniform(wgen, (w.get_rows(), 8), -0.3, 0.3, np.float32))
        out = net.propagate(ch.DeviceTensor.from_host(x.astype(dtype, order="F")))
        assert dtype == np.float64 or net.fused_steps()[0] == 2
        dx = net.backpropagate(ch.DeviceTensor.from_host(np.ones(out.shape, dtype, order="F")))
        got.append((out.to_host(), dx.to_host()))
    for a, b in zip(*got):
        assert hp.rel_err(a, b) <= 1e-5
