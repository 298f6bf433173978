"""The products that run on the bf16 matrix cores with their float32 operands
split in three: sizes at the edges of its tiles and of the rules that pick it,
and values the split cannot carry (infinities, NaN, sums that overflow)."""

from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    from ttrl_amd.engine.device import open_device

    return open_device(0)


def _patches(x, k, s):
    """(B, H, W, C) -> (B * OH * OW, k * k * C) in float64, k order (kh, kw, c)."""
    oh = (x.shape[1] - k) // s + 1
    ow = (x.shape[2] - k) // s + 1
    cols = [x[:, i:i + s * oh:s, j:j + s * ow:s] for i in range(k) for j in range(k)]
    return np.stack(cols, 3).reshape(x.shape[0] * oh * ow, -1).astype(np.float64)


def _scatter(cols, shape, k, s):
    """The adjoint of _patches: columns added back onto an image batch."""
    b, h, w, c = shape
    oh, ow = (h - k) // s + 1, (w - k) // s + 1
    cols = cols.reshape(b, oh, ow, k * k, c)
    out = np.zeros(shape)
    for i in range(k):
        for j in range(k):
            out[:, i:i + s * oh:s, j:j + s * ow:s] += cols[:, :, :, i * k + j]
    return out


def _bound(terms, magnitude):
    """Rounding of a float32 sum of `terms` products in any order: terms + 16
    roundings (the split's dropped parts, at most 2^-24 of each product, and
    the epilogue among the 16) of at most 2^-24 of the sum of magnitudes."""
    return (terms + 16) * 2.0 ** -24 * magnitude


def _backward(dev, x, dy, wt, k, s, u8, scale=1.0, mask=None, bank=None):
    """-> (dW, db, dX or None) of the convolution; with `bank`, the weight
    gradient's partials formed by the launch that reads gradient banks."""
    from ttrl_amd import _lib
    from ttrl_amd.engine.tensor import DeviceArray, to_device

    B = x.shape[0]
    c, h, w = (x.shape[1], x.shape[2], x.shape[3]) if u8 else (x.shape[3], x.shape[1], x.shape[2])
    o = dy.shape[1]
    geom = _lib.ConvGeom(B, c, h, w, o, k, s, 0, _lib.LAYOUT_NCHW_U8 if u8 else _lib.LAYOUT_NHWC_F32)
    xd, dyd = to_device(x, dev, x.dtype), to_device(dy, dev)
    dw, db = DeviceArray(dev, (c * k * k, o)), DeviceArray(dev, (1, o))
    if u8:
        dev.call("ttrl_conv2d_backward_weight", C.byref(geom), xd.vp, C.c_float(scale), dyd.vp, None, dw.vp, db.vp,
                 C.c_float(0.0))
        return dw.numpy(), db.numpy(), None
    wd, dx = to_device(wt, dev), DeviceArray(dev, x.shape)
    md = None if mask is None else to_device(mask, dev)
    mp = None if md is None else md.vp
    if bank is None:
        dev.call("ttrl_conv2d_backward", C.byref(geom), xd.vp, C.c_float(scale), dyd.vp, None, wd.vp, dw.vp, db.vp,
                 C.c_float(0.0), dx.vp, mp, C.c_float(0.0))
    else:
        src = _lib.GradSource()
        dev.call("ttrl_conv2d_backward_deferred", C.byref(geom), xd.vp, C.c_float(scale), dyd.vp, None, wd.vp, dw.vp,
                 db.vp, dx.vp, mp, C.c_float(0.0), bank, C.byref(src))
        assert src.kind == _lib.GRAD_SPLITS and src.splits > 1
        dev.call("ttrl_grad_sources_materialize", 1, C.byref(src))
    return dw.numpy(), db.numpy(), dx.numpy()


# (batch, channels, size, out, kernel, stride): batches on both sides of each
# rule's line (test_which_core_forms_a_gradient), rows and columns one past a
# tile, input channels that are and are not whole fragments of columns, strides
# whose residue classes differ.
CONVS = [(301, 32, 8, 64, 3, 1), (302, 32, 8, 64, 3, 1), (166, 32, 8, 64, 3, 1), (167, 32, 8, 64, 3, 1), (400, 32, 7, 32, 2, 1), (251, 36, 9, 96, 5, 1),
         (110, 32, 20, 64, 4, 2), (700, 64, 5, 32, 3, 1), (170, 20, 14, 64, 2, 2), (130, 96, 11, 20, 3, 1)]


@pytest.mark.parametrize("b,c,size,o,k,s", CONVS)
@pytest.mark.parametrize("bank", [None, 1])
def test_convolution_gradients(dev, b, c, size, o, k, s, bank):
    rng = np.random.default_rng(b)
    x = rng.standard_normal((b, size, size, c)).astype(np.float32)
    wt = rng.standard_normal((k * k * c, o)).astype(np.float32)
    a = _patches(x, k, s)
    dy = rng.standard_normal((a.shape[0], o)).astype(np.float32)
    mask = x if bank is None else None
    dw, db, dx = _backward(dev, x, dy, wt, k, s, False, 0.5, mask, bank)
    g = dy.astype(np.float64)
    assert np.all(np.abs(dw - 0.5 * (a.T @ g)) <= _bound(a.shape[0], np.abs(a).T @ np.abs(g)))
    assert np.all(np.abs(db[0] - g.sum(0)) <= _bound(a.shape[0], np.abs(g).sum(0)))
    w64 = wt.astype(np.float64)
    want = 0.5 * _scatter(g @ w64.T, x.shape, k, s)
    magnitude = _scatter(np.abs(g) @ np.abs(w64).T, x.shape, k, s)
    if mask is not None:
        want = np.where(mask > 0, want, 0.0)
    assert np.all(np.abs(dx - want) <= _bound(k * k * o, magnitude))


@pytest.mark.parametrize("b,c,h,w,o", [(15, 4, 84, 84, 32), (61, 4, 84, 84, 32), (62, 4, 84, 84, 32), (25, 3, 100, 100, 16),
                                       (60, 3, 100, 100, 16), (700, 1, 36, 36, 32), (90, 4, 84, 52, 20),
                                       (110, 4, 84, 52, 20), (97, 2, 84, 84, 64)])
def test_frames_weight_gradient(dev, b, c, h, w, o):
    rng = np.random.default_rng(b)
    x = rng.integers(0, 256, (b, c, h, w), dtype=np.uint8)
    a = _patches(x.transpose(0, 2, 3, 1), 8, 4).reshape(-1, 64, c).transpose(0, 2, 1).reshape(-1, c * 64)
    dy = rng.standard_normal((a.shape[0], o)).astype(np.float32)
    dw, db, _ = _backward(dev, x, dy, None, 8, 4, True, 1.0 / 255.0)
    g = dy.astype(np.float64)
    scale = np.float64(np.float32(1.0 / 255.0))
    assert np.all(np.abs(dw - scale * (a.T @ g)) <= scale * _bound(a.shape[0], np.abs(a).T @ np.abs(g)))
    assert np.all(np.abs(db[0] - g.sum(0)) <= _bound(a.shape[0], np.abs(g).sum(0)))


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 3.3e38, 1e-38])
def test_values_outside_the_split(dev, value):
    """A value bf16 parts cannot carry gives what float32 gives in the sums
    that read it, and leaves the others alone."""
    rng = np.random.default_rng(3)
    x = rng.standard_normal((200, 9, 9, 32)).astype(np.float32)
    x[..., 5] = 1.0  # no lower parts: inf * 0 must not appear
    wt = rng.uniform(0.25, 0.5, (9 * 32, 64)).astype(np.float32)
    a = _patches(x, 3, 1)
    dy = rng.standard_normal((a.shape[0], 64)).astype(np.float32)
    dy[1234, 7] = value
    dw, db, dx = _backward(dev, x, dy, wt, 3, 1, False)
    g, w64 = dy.astype(np.float64), wt.astype(np.float64)
    with np.errstate(all="ignore"):
        wants = ((dw, a.T @ g, a.shape[0], np.abs(a).T @ np.abs(g)),
                 (db[0], g.sum(0), a.shape[0], np.abs(g).sum(0)),
                 (dx, _scatter(g @ w64.T, x.shape, 3, 1), 9 * 64, _scatter(np.abs(g) @ w64.T, x.shape, 3, 1)))
        for got, want, terms, magnitude in wants:
            bad = ~np.isfinite(want.astype(np.float32))
            assert np.array_equal(np.isnan(got[bad]), np.isnan(want[bad]))
            some = bad & ~np.isnan(want)
            assert np.array_equal(np.sign(got[some]), np.sign(want[some]))
            fine = ~bad & (magnitude < 1e38)
            assert np.all(np.abs(got - want)[fine] <= _bound(terms, magnitude[fine]))


class _Layer:
    """One layer's operands on the device and its gradient entry points; the
    gradients of a call under `fp32`, or by the rule that picks the core."""

    def __init__(self, dev, b, c, size, o, k, s, u8=False, p=0):
        from ttrl_amd.engine.tensor import to_device

        rng = np.random.default_rng(b + size)
        self.dev, self.dims = dev, (b, c, size, o, k, s, u8, p)
        oh = (size + 2 * p - k) // s + 1
        x = rng.integers(0, 256, (b, c, size, size), dtype=np.uint8) if u8 else \
            rng.standard_normal((b, size, size, c)).astype(np.float32)
        self.x = to_device(x, dev, x.dtype)
        self.wt = to_device(rng.standard_normal((k * k * c, o)).astype(np.float32), dev)
        self.dy = to_device(rng.standard_normal((b * oh * oh, o)).astype(np.float32), dev)

    def geom(self, fp32):
        from ttrl_amd import _lib

        b, c, size, o, k, s, u8, p = self.dims
        layout = _lib.LAYOUT_NCHW_U8 if u8 else _lib.LAYOUT_NHWC_F32
        return C.byref(_lib.ConvGeom(b, c, size, size, o, k, s, p, layout | (_lib.CONV_FP32_ORDER if fp32 else 0)))

    def _out(self, shape):
        from ttrl_amd.engine.tensor import DeviceArray

        return DeviceArray(self.dev, shape)

    def weight(self, fp32):
        dw, db = self._out(self.wt.shape), self._out((1, self.dims[3]))
        self.dev.call("ttrl_conv2d_backward_weight", self.geom(fp32), self.x.vp, C.c_float(1.0), self.dy.vp, None, dw.vp,
                      db.vp, C.c_float(0.0))
        return dw.numpy()

    def input(self, fp32):
        dx = self._out(self.x.shape)
        self.dev.call("ttrl_conv2d_backward_input", self.geom(fp32), self.dy.vp, None, self.wt.vp, dx.vp, None,
                      C.c_float(1.0), C.c_float(0.0))
        return dx.numpy()

    def both(self, bank=None):
        """ttrl_conv2d_backward, or with a bank ttrl_conv2d_backward_deferred
        (no dW: its partials stay in the bank) -> dW, dX."""
        from ttrl_amd import _lib

        dw, db, dx = self._out(self.wt.shape), self._out((1, self.dims[3])), self._out(self.x.shape)
        args = (self.geom(False), self.x.vp, C.c_float(1.0), self.dy.vp, None, self.wt.vp, dw.vp, db.vp)
        if bank is None:
            self.dev.call("ttrl_conv2d_backward", *args, C.c_float(0.0), dx.vp, None, C.c_float(0.0))
            return dw.numpy(), dx.numpy()
        src = _lib.GradSource()
        self.dev.call("ttrl_conv2d_backward_deferred", *args, dx.vp, None, C.c_float(0.0), bank, C.byref(src))
        return None, dx.numpy()


# Frames and float layers, and whether the split core forms their weight
# gradient and their input gradient (None: there is none).
CORES = [((32, 4, 84, 32, 8, 4, True), False, None),   # 105 M products
         ((61, 4, 84, 32, 8, 4, True), False, None),   # 199.9 M
         ((62, 4, 84, 32, 8, 4, True), True, None),
         ((75, 3, 52, 32, 8, 4, True), False, None),   # 66 M
         ((512, 3, 52, 32, 8, 4, True), True, None),   # a weight of 192 x 32 bytes' products
         ((512, 1, 84, 32, 8, 4, True), False, None),  # 420 M, but a weight of 64 x 32
         ((32, 32, 20, 64, 4, 2), False, False),       # 85 M; 100 tiles
         ((47, 32, 20, 64, 4, 2), False, False),       # 125 M; 148 tiles
         ((48, 32, 20, 64, 4, 2), False, True),        # 150 tiles
         ((64, 32, 20, 64, 4, 2), False, True),        # 170 M; 200 tiles
         ((256, 32, 20, 64, 4, 2), True, True),
         ((96, 64, 9, 64, 3, 1), False, False),        # 173 M; 122 tiles
         ((128, 64, 9, 64, 3, 1), True, True),         # 231 M; 162 tiles
         ((512, 16, 12, 32, 3, 1), False, True),       # 236 M, but a weight of 144 x 32; 576 tiles
         ((300, 32, 18, 20, 4, 2), True, False),       # 20 outputs: dX reads 32 at a time
         ((512, 32, 8, 32, 2, 2), False, True)]        # K 32; 256 tiles


@pytest.mark.parametrize("dims,dw,dx", CORES)
def test_which_core_forms_a_gradient(dev, dims, dw, dx):
    """Sums on the two cores differ in their last bits, so whether a gradient
    is the one under TTRL_CONV_FP32_ORDER shows which core formed it."""
    layer = _Layer(dev, *dims)
    assert np.array_equal(layer.weight(False), layer.weight(True)) == (not dw)
    if dx is not None:
        assert np.array_equal(layer.input(False), layer.input(True)) == (not dx)


@pytest.mark.parametrize("dims,dw,dx", [row for row in CORES if row[2] or (row[1] and row[2] is not None)])
@pytest.mark.parametrize("bank", [None, 2])
def test_both_gradients_choose_their_cores_apart(dev, dims, dw, dx, bank):
    """The call for both gradients: what the split core forms for a call of its
    own it forms there too, bit for bit, except where the call has timed one
    launch of both on the FP32 core as faster."""
    layer = _Layer(dev, *dims)
    both_dw, both_dx = layer.both(bank)
    b, c, size, o, k, s = dims
    key = f"ttrl_conv2d_backward:pair|0|{b}|{c}|{size}|{size}|{o}|{k}|{k}|{s}|0|0|0|{int(bank is not None)}|split"
    plan = [row.split("\t")[0].split()[0] for row in dev.export_plans().splitlines() if row.endswith(key)]
    assert len(plan) == 1
    separate = plan[0] == "0"
    if dx:
        assert np.array_equal(both_dx, layer.input(False)) == separate
    if dw and bank is None:
        assert np.array_equal(both_dw, layer.weight(False)) == separate
    assert separate or not (dw and dx)  # both well past the lines


@pytest.mark.parametrize("dims", [(62, 4, 84, 32, 8, 4, True), (256, 32, 20, 64, 4, 2), (128, 64, 9, 64, 3, 1)])
def test_the_flag_gives_the_fp32_core(dev, dims):
    """Output gradients one float off 16-byte alignment keep any layer on the
    FP32 core, by the same plan: TTRL_CONV_FP32_ORDER gives its bits."""
    from ttrl_amd.engine.tensor import to_device

    layer = _Layer(dev, *dims)
    want = layer.weight(True), None if layer.dims[6] else layer.input(True)
    dy = layer.dy.numpy()
    layer.dy = to_device(np.concatenate([[np.float32(0.0)], dy.ravel()]), dev).view(1, dy.shape)
    assert np.array_equal(layer.weight(False), want[0])
    if want[1] is not None:
        assert np.array_equal(layer.input(False), want[1])


# Output gradients masked by the layer's own ReLU (a copy in the workspace, the
# partials below it), outputs added to, kernels whose classes take several
# launches (stride 3: nine), and padding (the weight gradient then on the FP32
# core): (batch, channels, size, out, kernel, stride, padding).
FORMS = [(256, 32, 20, 64, 4, 2, 0), (128, 64, 9, 64, 3, 1, 0), (400, 32, 15, 64, 3, 3, 0), (400, 24, 13, 32, 5, 4, 0),
         (64, 32, 20, 64, 3, 1, 1), (300, 20, 12, 32, 4, 2, 1)]


@pytest.mark.parametrize("b,c,size,o,k,s,p", FORMS)
@pytest.mark.parametrize("entry", ["both", "apart", "deferred"])
def test_masks_sums_strides_and_padding(dev, b, c, size, o, k, s, p, entry):
    from ttrl_amd import _lib
    from ttrl_amd.engine.tensor import DeviceArray, to_device

    rng = np.random.default_rng(b + size)
    x = rng.standard_normal((b, size, size, c)).astype(np.float32)
    xp = np.pad(x, ((0, 0), (p, p), (p, p), (0, 0)))
    a = _patches(xp, k, s)
    wt = rng.standard_normal((k * k * c, o)).astype(np.float32)
    dy, y = (rng.standard_normal((a.shape[0], o)).astype(np.float32) for _ in range(2))
    geom = C.byref(_lib.ConvGeom(b, c, size, size, o, k, s, p, _lib.LAYOUT_NHWC_F32))
    xd, dyd, yd, wd = (to_device(v, dev) for v in (x, dy, y, wt))
    dw, db, dx = DeviceArray(dev, wt.shape), DeviceArray(dev, (1, o)), DeviceArray(dev, x.shape)
    for out in (dw, db, dx):
        out.fill(3.0)
    beta = np.float32(0.0 if entry == "deferred" else 0.5)  # the deferred weight gradient is written fresh
    half = C.c_float(0.5)
    if entry == "both":
        dev.call("ttrl_conv2d_backward", geom, xd.vp, half, dyd.vp, yd.vp, wd.vp, dw.vp, db.vp, half, dx.vp, xd.vp, half)
    elif entry == "apart":
        dev.call("ttrl_conv2d_backward_weight", geom, xd.vp, half, dyd.vp, yd.vp, dw.vp, db.vp, half)
        dev.call("ttrl_conv2d_backward_input", geom, dyd.vp, yd.vp, wd.vp, dx.vp, xd.vp, half, half)
        other = DeviceArray(dev, x.shape)
        other.fill(3.0)
        fp32 = C.byref(_lib.ConvGeom(b, c, size, size, o, k, s, p, _lib.LAYOUT_NHWC_F32 | _lib.CONV_FP32_ORDER))
        dev.call("ttrl_conv2d_backward_input", fp32, dyd.vp, yd.vp, wd.vp, other.vp, xd.vp, half, half)
        assert not np.array_equal(dx.numpy(), other.numpy())  # every form is the split core's
    else:
        src = _lib.GradSource()
        dev.call("ttrl_conv2d_backward_deferred", geom, xd.vp, half, dyd.vp, yd.vp, wd.vp, dw.vp, db.vp, dx.vp, xd.vp,
                 half, 3, C.byref(src))
        if src.kind != _lib.GRAD_NONE:
            dev.call("ttrl_grad_sources_materialize", 1, C.byref(src))
    g = np.where(y > 0, dy, np.float32(0.0)).astype(np.float64)
    w64 = wt.astype(np.float64)
    crop = (slice(None), slice(p, p + size), slice(p, p + size))
    dx64, mag = (_scatter(f(g) @ f(w64).T, xp.shape, k, s)[crop] for f in (lambda v: v, np.abs))
    # the float32 epilogue rounds twice more, on the old value among them
    for got, want, terms, m in ((dw, 0.5 * (a.T @ g) + beta * 3.0, a.shape[0], np.abs(a).T @ np.abs(g) + 6.0),
                                (db, g.sum(0)[None] + beta * 3.0, a.shape[0], np.abs(g).sum(0)[None] + 6.0),
                                (dx, np.where(x > 0, 0.5 * dx64, 0.0) + 1.5, k * k * o, mag + 6.0)):
        assert np.all(np.abs(got.numpy() - want) <= _bound(terms, m))


def test_short_sums_of_the_worst_operands(dev):
    """Sums of 32 products (one step of the core) of operands whose mantissa
    leaves most in the lower parts (0x00ffff).  In 2^-24 of the sum: 1 for the
    products left out, 1 for each of at most four additions of the main sum, 1
    for adding the lower products' sum."""
    rng = np.random.default_rng(5)
    one = np.array([0x3F80FFFF], np.uint32).view(np.float32)[0]
    x = np.ones((1600, 8, 8, 64), np.float32)
    wt = one * np.exp2(rng.integers(-3, 4, (4 * 64, 32))).astype(np.float32)
    dy = one * np.exp2(rng.integers(-3, 4, (1600 * 16, 32))).astype(np.float32)
    _, _, dx = _backward(dev, x, dy, wt, 2, 2, False)
    want = _scatter(dy.astype(np.float64) @ wt.astype(np.float64).T, x.shape, 2, 2)
    assert np.max(np.abs(dx - want) / want) <= 6 * 2.0 ** -24


def test_sums_of_one_sign_are_not_biased(dev):
    """Rounding to nearest errs to either side alike: over n sums of positive
    terms, each off by at most E * 2^-24 of itself, the mean error lies within
    five standard deviations, 5 E / sqrt(n) * 2^-24 (E = 12 bounds the largest
    of either gradient)."""
    rng = np.random.default_rng(6)
    k, s = 4, 2
    x = np.abs(rng.standard_normal((256, 20, 20, 32))).astype(np.float32)
    wt = np.abs(rng.standard_normal((k * k * 32, 64))).astype(np.float32)
    a = _patches(x, k, s)
    dy = np.abs(rng.standard_normal((a.shape[0], 64))).astype(np.float32)
    dw, _, dx = _backward(dev, x, dy, wt, k, s, False)
    g = dy.astype(np.float64)
    for got, want in ((dw, a.T @ g), (dx, _scatter(g @ wt.astype(np.float64).T, x.shape, k, s))):
        e = (got - want) / want * 2.0 ** 24
        assert np.max(np.abs(e)) <= 12
        assert abs(e.mean()) <= 5 * 12 / np.sqrt(e.size)


@pytest.mark.parametrize("power", [100, 112, 120])
def test_gradients_of_tiny_values(dev, power):
    """Output gradients down to 2^-120, whose lower parts bf16 cannot hold:
    2-norm error of float32 sums, at most sqrt(terms) * 2^-24 of the sum's own
    norm (9,800 terms in parts of 200 at most: 14 * 2^-24 = 9e-7), as 1e-6."""
    rng = np.random.default_rng(9)
    k, s = 3, 1
    x = rng.standard_normal((200, 9, 9, 32)).astype(np.float32)
    wt = rng.standard_normal((k * k * 32, 64)).astype(np.float32)
    a = _patches(x, k, s)
    dy = (rng.standard_normal((a.shape[0], 64)) * 2.0 ** -power).astype(np.float32)
    dw, _, dx = _backward(dev, x, dy, wt, k, s, False)
    g = dy.astype(np.float64)
    for got, want in ((dw, a.T @ g), (dx, _scatter(g @ wt.astype(np.float64).T, x.shape, k, s))):
        assert np.linalg.norm(got - want) <= 1e-6 * np.linalg.norm(want)
