"""fp32 convolutions and dense layers whose products run on the bf16 matrix instructions (an fp32 number as three bf16
numbers): against the oracle in double precision at the edges of the tiles, and where three bf16 numbers cannot stand in
for an fp32 number - infinities, NaNs, values near the largest and near the smallest.

The bound on the 2-norm error is that of fp32 sums: L roundings of relative size 2^-24 that add up like a random walk,
sqrt(L) 2^-24, for reductions of length L; and 20 x 2^-24 = 1.2e-6 for all longer ones, twice the largest error measured (a
weight gradient over 800,000 rows, 6.1e-7) and a third of what a missing product of parts makes (2^-18)."""
import ctypes
import importlib

import numpy as np
import pytest

import helpers as hp
from oracle import oracle

pytestmark = pytest.mark.gpu

ch = importlib.import_module("c-attl3_amd")


def _run(x, w, b, go, geom):
    H, W, C = x.shape[1:]
    layer = ch.ConvKernelLayer(np.float32, (H, W, C), w.shape[1], geom["RH"], geom["RW"], geom["pv"], geom["ph"], geom["sv"], geom["sh"],
                               geom["dv"], geom["dh"])
    wp, bp = layer.get_params()
    wp.set_values(w)
    bp.set_values(b)
    out = layer.pass_forward(x, True)
    dx = layer.pass_back(go)
    return {"out": out, "dx": dx, "dw": wp.get_grad(), "db": bp.get_grad()}


def _truth(x, w, b, go, geom):
    x, w, b, go = (np.asarray(a, np.float64) for a in (x, w, b, go))
    out, cache = oracle.conv_forward(x, w, b, return_cache=True, **geom)
    dx, dw, db = oracle.conv_backward(x.shape, cache, w, go, **geom)
    return {"out": out, "dx": dx, "dw": dw, "db": db}


def _geom(R=3, pad=1, stride=1, dilation=0):
    return dict(RH=R, RW=R, pv=pad, ph=pad, sv=stride, sh=stride, dv=dilation, dh=dilation)


def _inputs(N, H, W, C, F, geom, seed, scale=1.0):
    g = hp.rng(seed)
    R = geom["RH"]
    OH, OW = hp.conv_dims(H, W, R, R, geom["pv"], geom["ph"], geom["sv"], geom["sh"], geom["dv"], geom["dh"])
    return (hp.normal(g, (N, H, W, C), np.float32, scale), hp.normal(g, (R * R * C, F), np.float32, (2.0 / (R * R * C)) ** 0.5),
            hp.normal(g, (1, F), np.float32, scale), hp.normal(g, (N, OH, OW, F), np.float32, scale))


def _check(got, ref, lengths):
    for k, L in lengths.items():
        e = np.linalg.norm(np.asarray(got[k], np.float64) - ref[k]) / np.linalg.norm(ref[k])
        assert e <= 2.0 ** -24 * min(max(L, 16) ** 0.5, 20.0), (k, e, L)


CASES = [
    # N, H, W, C, F, geometry: sizes around the tiles' edges, on either kind of instruction
    (64, 32, 33, 8, 128, _geom()), (64, 33, 32, 7, 97, _geom()), (66, 32, 33, 8, 65, _geom()), (64, 33, 34, 6, 64, _geom()),
    (67, 31, 33, 6, 63, _geom()), (32, 10, 9, 16, 130, _geom()), (50, 9, 11, 24, 44, _geom()), (33, 7, 9, 11, 33, _geom()),
    (96, 16, 12, 32, 32, _geom()), (31, 13, 7, 40, 17, _geom()), (8, 9, 8, 64, 9, _geom()),
    # receptors of one tap, many taps, dilated; strides (a gradient by residue classes where the work allows it)
    (40, 14, 14, 96, 200, _geom(1, 0)), (16, 9, 9, 40, 72, _geom(5, 2)), (32, 12, 12, 24, 48, _geom(3, 2, 1, 1)),
    (64, 24, 22, 48, 96, _geom(3, 1, 2)), (64, 18, 18, 40, 100, _geom(4, 2, 2)), (21, 15, 13, 30, 50, _geom(3, 1, 2)),
    (70, 20, 19, 35, 96, _geom(3, 1, 2)), (66, 26, 23, 34, 70, _geom(4, 2, 2)),
    # reductions just above where the path begins, and cut into parts
    (32, 6, 6, 48, 96, _geom(1, 0)), (4, 6, 6, 300, 48, _geom()), (130, 2, 2, 256, 256, _geom()),
]


@pytest.mark.parametrize("case", CASES, ids=["%dx%dx%dx%d-f%d-r%dp%ds%dd%d" % (c[:5] + (c[5]["RH"], c[5]["pv"], c[5]["sv"], c[5]["dv"])) for c in CASES])
def test_layers_at_tile_edges(case):
    N, H, W, C, F, geom = case
    x, w, b, go = _inputs(N, H, W, C, F, geom, 7 * N + F)
    rows = N * go.shape[1] * go.shape[2]
    _check(_run(x, w, b, go, geom), _truth(x, w, b, go, geom),
           {"out": w.shape[0], "dx": geom["RH"] * geom["RW"] * F, "dw": rows, "db": rows})


TILES = [
    # N, H, W, C, F, receptor, tiles of the forward product, the input gradient and the weight gradient (rows * 1000 + columns; 0: fp32
    # instructions). Every tile, with batches that are multiples of four, even and odd, rows and columns that are no multiples of
    # the tile, whole rounds of tiles and cut ones behind them
    (76, 20, 22, 75, 69, 1, 256128, 256128, 96128), (25, 30, 24, 51, 195, 1, 256128, 64064, 96128),
    (33, 33, 36, 10, 74, 3, 256128, 64064, 96128), (34, 29, 30, 51, 191, 1, 256128, 64064, 64064),
    (52, 24, 16, 80, 167, 1, 256064, 128032, 96128), (49, 23, 22, 89, 99, 1, 256064, 256064, 96128),
    (118, 24, 18, 9, 34, 3, 256064, 128032, 0), (40, 21, 34, 48, 76, 1, 128064, 0, 0), (118, 32, 32, 55, 57, 1, 128064, 128064, 64064),
    (92, 15, 8, 13, 79, 3, 64064, 0, 0), (61, 11, 12, 106, 129, 1, 64064, 64064, 0), (43, 19, 20, 55, 19, 3, 128032, 64064, 64064),
    (49, 30, 27, 83, 17, 3, 64064, 256128, 128064), (63, 19, 29, 88, 15, 3, 64064, 256128, 128064),
    (44, 18, 40, 83, 10, 3, 64064, 256064, 128064), (92, 36, 26, 10, 23, 3, 128032, 128032, 128064),
    (64, 20, 20, 32, 64, 3, 64064, 64064, 64064), (66, 20, 21, 48, 96, 3, 256064, 64064, 96128),
    (37, 9, 27, 125, 214, 3, 256128, 256128, 192128), (92, 36, 17, 55, 101, 3, 256128, 256064, 192128),
]


@pytest.mark.parametrize("case", TILES, ids=["%dx%dx%dx%d-f%d-r%d" % c[:6] for c in TILES])
def test_every_tile(case):
    N, H, W, C, F, R, forward, dgrad, wgrad = case
    geom = _geom(R, R // 2)
    x, w, b, go = _inputs(N, H, W, C, F, geom, 3 * N + F)
    layer = ch.ConvKernelLayer(np.float32, (H, W, C), F, R, R, R // 2, R // 2)
    wp, bp = layer.get_params()
    wp.set_values(w)
    bp.set_values(b)
    out = layer.pass_forward(x, True)
    took = [ch.last_products()[0]]
    dx = layer.pass_back(go)
    took += ch.last_products()
    assert took == [forward, dgrad, wgrad]
    rows = N * H * W
    _check({"out": out, "dx": dx, "dw": wp.get_grad(), "db": bp.get_grad()}, _truth(x, w, b, go, geom),
           {"out": w.shape[0], "dx": R * R * F, "dw": rows, "db": rows})


@pytest.mark.parametrize("which", ["out", "dx", "dw"])
def test_single_products(which):
    """Every result is one product of two fp32 numbers with all 24 bits in use: at most 2^-24 for the products of parts that are
    left out and 2^-24 for the sum's rounding; a missing product of parts would be 2^-18 or more."""
    N, C, F = 512, 4096, 256
    g = hp.rng(29)
    one = lambda shape: hp.uniform(g, shape, 1, 2, np.float32) * np.where(g.random(shape) < 0.5, -1, 1).astype(np.float32)
    x, w, go = one((N, C)), one((C, F)), one((N, F))
    layer = ch.DenseKernelLayer(np.float32, (C,), F)
    wp, bp = layer.get_params()
    bp.set_values(np.zeros((1, F), np.float32))

    def single(a, axis):
        """a with one entry per row (axis 1) or column (axis 0) kept"""
        keep = np.zeros(a.shape, bool)
        at = g.integers(0, a.shape[axis], a.shape[1 - axis])
        keep[(np.arange(a.shape[0]), at) if axis == 1 else (at, np.arange(a.shape[1]))] = True
        return np.asfortranarray(np.where(keep, a, 0).astype(np.float32))

    if which == "out":
        x = single(x, 1)
    elif which == "dx":
        go = single(go, 1)
    else:
        x = single(x, 0)
    wp.set_values(w)
    out = layer.pass_forward(x, True)
    product = ch.last_products()[0]
    dx = layer.pass_back(go)
    assert {"out": product, "dx": ch.last_products()[0], "dw": ch.last_products()[1]}[which] > 0
    x, w, go = (a.astype(np.float64) for a in (x, w, go))
    got, ref = {"out": lambda: (out, x @ w), "dx": lambda: (dx, go @ w.T), "dw": lambda: (wp.get_grad(), x.T @ go)}[which]()
    assert (np.abs(got - ref) <= 2.0 ** -23 * np.abs(ref)).all()


@pytest.mark.parametrize("shape", [(64, 33, 32, 8, 96), (64, 20, 20, 32, 64), (66, 20, 21, 48, 96), (33, 7, 9, 16, 48)], ids=str)
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan], ids=str)
def test_values_that_are_not_finite(shape, value):
    """An infinity or NaN in the input and in the upstream gradient reaches exactly the results that it reaches in fp32, with
    the same values, and no others."""
    geom = _geom()
    x, w, b, go = _inputs(*shape, geom, 3)
    x[3, 2, 1, 5] = value
    go[1, 4, 3, 7] = value
    got, ref = _run(x, w, b, go, geom), _truth(x, w, b, go, geom)
    for k in got:
        a, r = np.asarray(got[k], np.float64), ref[k]
        bad = ~np.isfinite(r)
        assert bad.any() and np.array_equal(np.isnan(a), np.isnan(r)) and np.array_equal(a[np.isinf(r)], r[np.isinf(r)]), k
        e = np.linalg.norm((a - r)[~bad]) / np.linalg.norm(r[~bad]) if (~bad).any() else 0.0
        assert e <= 2.0 ** -24 * (x.shape[0] * x.shape[1] * x.shape[2]) ** 0.5, (k, e)


class _Offset(object):
    """A device tensor that begins `elements` fp32 elements behind a 256-byte boundary."""

    def __init__(self, shape, elements, values=None):
        self.shape = shape
        self._block = ch.DeviceTensor((int(np.prod(shape)) + 4,), np.float32)
        self.ptr = ctypes.c_void_p(self._block.ptr.value + 4 * elements)
        if values is not None:
            values = np.asfortranarray(values)
            ch.binding._check(ch.lib().cattle_hip_upload(self.ptr, ctypes.c_void_p(values.ctypes.data), ctypes.c_size_t(values.nbytes)))

    def to_host(self):
        a = np.empty(self.shape, np.float32, order="F")
        ch.binding._check(ch.lib().cattle_hip_download(ctypes.c_void_p(a.ctypes.data), self.ptr, ctypes.c_size_t(a.nbytes)))
        return a


@pytest.mark.parametrize("offset", [1, 2])
@pytest.mark.parametrize("shape", [(64, 33, 32, 8, 96), (32, 20, 21, 24, 130), (66, 24, 24, 16, 48)], ids=str)
def test_unaligned_tensors(shape, offset):
    """Caller's tensors on 4- and 8-byte boundaries only: no 16-byte loads, and so no walk of the weight gradient by positions."""
    geom = _geom()
    x, w, b, go = _inputs(*shape, geom, 19)
    layer = ch.ConvKernelLayer(np.float32, x.shape[1:], shape[4])
    wp, bp = layer.get_params()
    wp.set_values(w)
    bp.set_values(b)
    xd, gd, out, dx = _Offset(x.shape, offset, x), _Offset(go.shape, offset, go), _Offset(go.shape, offset), _Offset(x.shape, offset)
    layer.forward_into(xd, out)
    layer.backward_into(gd, dx)
    rows = shape[0] * shape[1] * shape[2]
    _check({"out": out.to_host(), "dx": dx.to_host(), "dw": wp.get_grad(), "db": bp.get_grad()}, _truth(x, w, b, go, geom),
           {"out": w.shape[0], "dx": 9 * shape[4], "dw": rows, "db": rows})


def _slice_error(got, ref):
    got, ref = np.asarray(got, np.float64), np.asarray(ref, np.float64)
    return np.linalg.norm(got - ref) / np.linalg.norm(ref)


TINY = [2.0 ** -82, 2.0 ** -112, 2.0 ** -119]       # lower bf16 parts of an unscaled number: normal, lost in part, denormal
TINY_SHAPES = [(64, 33, 32, 8, 96), (50, 9, 11, 24, 44)]


@pytest.mark.parametrize("tiny", TINY, ids=str)
@pytest.mark.parametrize("shape", TINY_SHAPES, ids=str)
def test_tiny_values(shape, tiny):
    """All operands of one side so small that the lower parts of an unscaled split are bf16 denormals: fp32 keeps their bits."""
    geom = _geom()
    x, w, b, go = _inputs(*shape, geom, 5, tiny)
    rows = x.shape[0] * x.shape[1] * x.shape[2]
    _check(_run(x, w, b, go, geom), _truth(x, w, b, go, geom), {"out": w.shape[0], "dx": 9 * shape[4]})
    got = _run(x, w, b, go / np.float32(tiny), geom)
    _check(got, _truth(x, w, b, go / np.float32(tiny), geom), {"dw": rows})


@pytest.mark.parametrize("tiny", TINY, ids=str)
@pytest.mark.parametrize("shape", TINY_SHAPES, ids=str)
def test_tiny_times_huge_values(shape, tiny):
    """Tiny operands against huge ones, with results of ordinary size."""
    geom = _geom()
    x, w, b, go = _inputs(*shape, geom, 8)
    rows = x.shape[0] * x.shape[1] * x.shape[2]
    t, huge = np.float32(tiny), np.float32(1 / tiny)
    got = _run(x * t, w * huge, b, go * t, geom)
    _check(got, _truth(x * t, w * huge, b, go * t, geom), {"out": w.shape[0], "dx": 9 * shape[4]})
    _check(_run(x * t, w, b, go * huge, geom), _truth(x * t, w, b, go * huge, geom), {"dw": rows})


@pytest.mark.parametrize("tiny", TINY, ids=str)
@pytest.mark.parametrize("shape", TINY_SHAPES, ids=str)
def test_tiny_values_among_ordinary_ones(shape, tiny):
    """One tiny sample, filter and channel among ordinary ones, in the same tiles: each keeps the precision of its own."""
    N, H, W, C, F = shape
    geom = _geom()
    x, w, b, go = _inputs(*shape, geom, 9)
    b[:] = 0
    t = np.float32(tiny)
    rows = N * H * W
    bound = lambda L: 2.0 ** -24 * max(L, 16) ** 0.5

    xs, gs = x.copy(order="F"), go.copy(order="F")
    xs[3] *= t
    gs[3] *= t
    got, ref = _run(xs, w, b, gs, geom), _truth(xs, w, b, gs, geom)
    assert _slice_error(got["out"][3], ref["out"][3]) <= bound(9 * C)
    assert _slice_error(got["dx"][3], ref["dx"][3]) <= bound(9 * F)

    xs, ws, gs = x.copy(order="F"), w.copy(order="F"), go.copy(order="F")
    xs[..., 2] *= t                     # (rows 18 to 26 of the weights and their gradient)
    ws[:, 5] *= t
    gs[..., 5] *= t
    got, ref = _run(xs, ws, b, gs, geom), _truth(xs, ws, b, gs, geom)
    assert _slice_error(got["out"][..., 5], ref["out"][..., 5]) <= bound(9 * C)
    assert _slice_error(got["dw"][18:27, :5], ref["dw"][18:27, :5]) <= bound(rows)
    assert _slice_error(got["dw"][:18, 5], ref["dw"][:18, 5]) <= bound(rows)


def test_values_near_the_largest():
    """Above the largest bf16 number, where rounding to bf16 gives an infinity."""
    geom = _geom()
    x, w, b, go = _inputs(50, 9, 11, 24, 44, geom, 6)
    x[7, 3, 2, 4] = np.float32(3.4e38)
    w *= np.float32(1e-3)
    got, ref = _run(x, w, b, go, geom), _truth(x, w, b, go, geom)
    assert np.isfinite(np.asarray(got["out"])).all()
    for n in (7, 8):
        a, r = np.asarray(got["out"][n], np.float64), ref["out"][n]
        assert np.linalg.norm(a - r) <= 2.0 ** -24 * w.shape[0] ** 0.5 * np.linalg.norm(r), n


@pytest.mark.parametrize("N,C,F", [(512, 4096, 256), (77, 333, 77), (300, 1000, 500), (2048, 96, 33), (1774, 1105, 542), (341, 2179, 850)])
def test_dense(N, C, F):
    g = hp.rng(N + F)
    x, w = hp.normal(g, (N, C), np.float32), hp.normal(g, (C, F), np.float32, (2.0 / C) ** 0.5)
    b, go = hp.normal(g, (1, F), np.float32), hp.normal(g, (N, F), np.float32)
    layer = ch.DenseKernelLayer(np.float32, (C,), F)
    wp, bp = layer.get_params()
    wp.set_values(w)
    bp.set_values(b)
    got = {"out": layer.pass_forward(x, True), "dx": layer.pass_back(go), "dw": wp.get_grad(), "db": bp.get_grad()}
    x, w, b, go = (a.astype(np.float64) for a in (x, w, b, go))
    _check(got, {"out": x @ w + b, "dx": go @ w.T, "dw": x.T @ go, "db": go.sum(0, keepdims=True)}, {"out": C, "dx": F, "dw": N, "db": N})


@pytest.mark.parametrize("behind", ["relu", "relu pool", "batch norm relu"])
@pytest.mark.parametrize("shape", [(64, 32, 32, 8, 96), (64, 64, 32, 8, 64), (32, 8, 16, 24, 100), (96, 16, 16, 12, 30)], ids=str)
def test_fused_epilogues(shape, behind):
    """The kernel layer with what is fused behind it against the same layers one by one, in fp32 both."""
    N, H, W, C, F = shape
    x, w, b, go = _inputs(N, H, W, C, F, _geom(), 11)

    def layers():
        out = [ch.ConvKernelLayer(np.float32, (H, W, C), F)]
        if "batch norm" in behind:
            out.append(ch.BatchNormLayer(np.float32, (H, W, F)))
        out.append(ch.ActivationLayer(np.float32, "relu", (H, W, F)))
        if "pool" in behind:
            out.append(ch.MeanPoolLayer(np.float32, (H, W, F)))
        out[0].get_params()[0].set_values(w)
        out[0].get_params()[1].set_values(b)
        return out

    def forward(ls):
        a = x
        for l in ls:
            a = l.pass_forward(a, True)
        return np.asarray(a)

    def backward(ls, conv, g):
        for l in reversed(ls):
            g = l.pass_back(g)
        return np.asarray(g), conv.get_params()[0].get_grad()

    plain, members = layers(), layers()
    fused = ch.fuse_layers(members)
    assert len(fused) == 1
    one, many = {"out": forward(fused)}, {"out": forward(plain)}
    g = np.asfortranarray(go if "pool" not in behind else go[:, ::2, ::2])
    if "pool" not in behind:
        # where the rounding of one pass carried a value across the rectifier's kink the gradients differ: no gradient there
        crossed = (one["out"] > 0) != (many["out"] > 0)
        assert crossed.mean() < 1e-4
        g[crossed] = 0
    one["dx"], one["dw"] = backward(fused, members[0], g)
    many["dx"], many["dw"] = backward(plain, plain[0], g)
    # two fp32 passes, each within the bound of its own. A pool hides which values crossed (its gradients are compared exactly by
    # test_fused_epilogues_of_whole_numbers); a batch norm's sums carry the rounding of its statistics to all gradients
    for k, L in {"out": 9 * C, "dx": 9 * F, "dw": N * H * W}.items():
        e = np.linalg.norm(one[k].astype(np.float64) - many[k]) / np.linalg.norm(many[k].astype(np.float64))
        slack = 2 if k == "out" or behind == "relu" else 200
        assert e <= slack * 2.0 ** -24 * min(L ** 0.5, 20.0), (k, e)


@pytest.mark.parametrize("behind", ["relu", "relu pool"])
@pytest.mark.parametrize("shape", [(64, 32, 32, 8, 96), (64, 64, 32, 8, 64), (32, 8, 16, 24, 100), (96, 16, 16, 12, 30)], ids=str)
def test_fused_epilogues_of_whole_numbers(shape, behind):
    """Small whole numbers, whose products and sums are exact: the fused group and the layers one by one agree to the last bit."""
    N, H, W, C, F = shape
    g = hp.rng(23)
    whole = lambda lo, hi, s: np.asfortranarray(g.integers(lo, hi + 1, s).astype(np.float32))
    x, w, b = whole(-3, 3, (N, H, W, C)), whole(-2, 2, (9 * C, F)), whole(-2, 2, (1, F))
    pool = "pool" in behind
    go = 4 * whole(-3, 3, (N, H // 2, W // 2, F) if pool else (N, H, W, F))

    def run(fuse):
        ls = [ch.ConvKernelLayer(np.float32, (H, W, C), F), ch.ActivationLayer(np.float32, "relu", (H, W, F))]
        if pool:
            ls.append(ch.MeanPoolLayer(np.float32, (H, W, F)))
        ls[0].get_params()[0].set_values(w)
        ls[0].get_params()[1].set_values(b)
        called = ch.fuse_layers(ls) if fuse else ls
        a, d = x, go
        for l in called:
            a = l.pass_forward(a, True)
        for l in reversed(called):
            d = l.pass_back(d)
        return a, d, ls[0].get_params()[0].get_grad(), ls[0].get_params()[1].get_grad()

    for got, ref in zip(run(True), run(False)):
        assert np.array_equal(np.asarray(got), np.asarray(ref))


def _pooled_layers(shape, w, b):
    H, W, C, F = shape
    layers = [ch.ConvKernelLayer(np.float32, (H, W, C), F), ch.ActivationLayer(np.float32, "relu", (H, W, F)), ch.MaxPoolLayer(np.float32, (H, W, F))]
    layers[0].get_params()[0].set_values(w)
    layers[0].get_params()[1].set_values(b)
    return layers


@pytest.mark.parametrize("N", [32, 30, 33])
def test_max_pool_group_leaves_its_kernel_layer_as_it_was(N):
    """A kernel layer grouped with a max pool runs on the fp32 instructions there; called by itself, before or after the
    group, it gives the bits of a layer that was never grouped."""
    H, W, C, F = 16, 16, 24, 100
    x, w, b, go = _inputs(N, H, W, C, F, _geom(), 13)
    pooled = go[:, ::2, ::2]

    def alone(conv):
        out = conv.pass_forward(x, True)
        dx = conv.pass_back(go)
        dw = conv.get_params()[0].get_grad()
        for p in conv.get_params():
            p.reset_grad()
        return out, dx, dw

    plain, members = _pooled_layers((H, W, C, F), w, b), _pooled_layers((H, W, C, F), w, b)
    expected = alone(plain[0])
    group = ch.fuse_layers(members)
    assert len(group) == 1
    for _ in range(2):
        for got, ref in zip(alone(members[0]), expected):
            assert np.array_equal(got, ref)
        group[0].pass_forward(x, True)
        group[0].pass_back(pooled)
        for p in members[0].get_params():
            p.reset_grad()


@pytest.mark.parametrize("N", [32, 30, 33])
def test_max_pool_group_against_its_layers(N):
    """Values whose products and sums are exact on either kind of instruction (small whole numbers): the group and the layers one
    by one agree to the last bit, ties between equal values included."""
    H, W, C, F = 16, 16, 24, 100
    g = hp.rng(17)
    x = np.asfortranarray(g.integers(-3, 4, (N, H, W, C)).astype(np.float32))
    w = np.asfortranarray(g.integers(-2, 3, (9 * C, F)).astype(np.float32))
    b = np.asfortranarray(g.integers(-2, 3, (1, F)).astype(np.float32))
    go = np.asfortranarray(g.integers(-3, 4, (N, H // 2, W // 2, F)).astype(np.float32))

    def run(layers, conv):
        a, d = x, go
        for l in layers:
            a = l.pass_forward(a, True)
        for l in reversed(layers):
            d = l.pass_back(d)
        return a, d, conv.get_params()[0].get_grad(), conv.get_params()[1].get_grad()

    plain, members = _pooled_layers((H, W, C, F), w, b), _pooled_layers((H, W, C, F), w, b)
    for got, ref in zip(run(ch.fuse_layers(members), members[0]), run(plain, plain[0])):
        assert np.array_equal(np.asarray(got), np.asarray(ref))


def test_smaller_batches_run_while_a_graph_lives():
    """Scratch buffers that were grown at the largest batch stay where they are while a graph lives. A smaller batch whose slices
    on the bf16 instructions would need more than that takes the fp32 plan instead of being refused."""
    H, W, C, F = 10, 10, 87, 239
    geom = _geom()
    tiny = ch.DenseKernelLayer(np.float32, (4,), 3)
    tx, ty = ch.DeviceTensor.from_host(np.ones((4, 4), np.float32, order="F")), ch.DeviceTensor((4, 3), np.float32)
    tiny.forward_into(tx, ty, False)
    layer = ch.ConvKernelLayer(np.float32, (H, W, C), F)
    x, w, b, go = _inputs(61, H, W, C, F, geom, 21)
    layer.get_params()[0].set_values(w)
    layer.get_params()[1].set_values(b)
    layer.pass_forward(x, True)
    layer.pass_back(go)
    graph = ch.Graph()
    with graph:
        tiny.forward_into(tx, ty, False)
    try:
        for N in (60, 53, 45, 38, 30, 24):
            for p in layer.get_params():
                p.reset_grad()
            xs, gs = np.asfortranarray(x[:N]), np.asfortranarray(go[:N])
            layer.pass_forward(xs, True)
            dx = layer.pass_back(gs)
            ref = _truth(xs, w, b, gs, geom)
            _check({"dx": dx, "dw": layer.get_params()[0].get_grad()}, ref, {"dx": 9 * F, "dw": N * H * W})
    finally:
        graph.destroy()
