"""The f16-split matrix kernels (float32 values as scaled f16 pairs): every
tile of the implicit GEMM and every form of the 3x3 patch kernel, pinned
through SIMDYOLO_HIP_TILE, against float64.

Bound: a value's pair is within 2^-23 of it, the product left out below 2^-22
of the product, so a sum of products is within 2^-20.5 of the sum of their
magnitudes before the accumulators round.  These round once per 16 terms and
product, each time by at most 2^-24 of the running sum: up to 2^-18.4 of the
magnitudes at K = 1152 if the sum grows evenly and every rounding had the same
sign.  They do not: the largest error over the forms and shapes below is 2^-22.7
of the magnitudes, 2^-19.9 where test_scales mixes far-apart ones, and 2^-19 is
asked for.  Rows or pixels out of the pairs' range are computed in float32,
one rounding per term or two: 2^-17 for them (within).
"""
import numpy as np
import pytest

from simdyolo_amd import CONV_IGEMM, SyError, synth

pytestmark = pytest.mark.gpu

X3_BASE, C3_BASE = 64, 96
X3_TILES = [(128, 128, 2, 2), (64, 64, 2, 2), (64, 128, 2, 2), (128, 32, 4, 1), (64, 32, 2, 1)]
# (pixels, channels, wave grid, waves per block)
C3_FORMS = [(128, 64, 2, 2, 1), (128, 32, 4, 1, 1), (64, 32, 2, 1, 1), (64, 64, 2, 2, 1), (64, 96, 2, 3, 1),
            (32, 32, 1, 1, 4), (32, 32, 1, 1, 8)]


def c3_name(form):
    bm, bn, wm, wn, kw = C3_FORMS[form]
    return f"conv3_x3_{bm}x{bn}_{wm}{wn}" + (f"_ks{kw}" if kw > 1 else "")


def conv64(x, w, b, stride, silu, res):
    """(result, sum of the products' magnitudes) in float64, NCHW."""
    x, w = x.astype(np.float64), w.astype(np.float64)
    n, ic, h, wd = x.shape
    oc, _, k, _ = w.shape
    p = k // 2
    oh, ow = (h + 2 * p - k) // stride + 1, (wd + 2 * p - k) // stride + 1
    y = np.zeros((n, oc, oh, ow)) + b.astype(np.float64)[None, :, None, None]
    mag = np.abs(y)
    xp = np.pad(x, ((0, 0), (0, 0), (p, p), (p, p)))
    with np.errstate(invalid="ignore", over="ignore"):
        for i in range(k):
            for j in range(k):
                t = xp[:, :, i:i + stride * (oh - 1) + 1:stride, j:j + stride * (ow - 1) + 1:stride]
                y += np.einsum("nchw,oc->nohw", t, w[:, :, i, j])
                mag += np.einsum("nchw,oc->nohw", np.abs(t), np.abs(w[:, :, i, j]))
        if silu:
            y = y / (1.0 + np.exp(-y))
    if res is not None:
        y = y + res
        mag = mag + np.abs(res)
    return y, mag


def run(hip, monkeypatch, tile, x, w, b, stride=1, silu=True, res=None):
    """The conv on channel slices of wider buffers; (result, kernel names)."""
    monkeypatch.setenv("SIMDYOLO_HIP_TILE", str(tile))
    n, ic, h, wd = x.shape
    oc, _, k, _ = w.shape
    hip.begin_frame()
    try:
        conv = hip.conv_create(w, b, (stride, stride), (k // 2,) * 4, silu=silu)
        hip.conv_set_algo(conv, CONV_IGEMM)
        oh, ow = hip.conv_out_size(conv, h, wd)
        xv = hip.alloc(n, ic + 4, h, wd).slice(4, ic)
        hip.upload(x, xv)
        yv = hip.alloc(n, oc + 13, oh, ow).slice(9, oc)
        rv = None
        if res is not None:
            rv = hip.alloc(n, oc + 7, oh, ow).slice(3, oc)
            hip.upload(res, rv)
        hip.profile_enable(True)
        hip.profile_read()
        try:
            hip.conv(conv, xv, yv, rv)
            hip.flush()
            names = set(hip.profile_read())
        finally:
            hip.profile_enable(False)
        return hip.download(yv), names
    finally:
        hip.end_frame()


def data(n, ic, h, w, oc, k, seed):
    return (synth.activations((n, ic, h, w), seed), synth.kaiming((oc, ic, k, k), seed + 1),
            synth.activations((oc,), seed + 2) * np.float32(0.1))


def near(got, exp, mag, floor=0.0):
    off = np.abs(got.astype(np.float64) - exp)
    allowed = 2.0 ** -19 * mag + floor
    assert np.isfinite(got).all() and (off <= allowed).all(), (off / allowed).max()


# (n, ic, h, w, oc, k, stride), mode: ragged pixels, channels and depth.
GEMM = [((2, 40, 13, 11, 72, 1, 1), 2), ((1, 4, 1, 1, 1, 1, 1), 2), ((1, 512, 9, 7, 132, 1, 1), 2),
        ((1, 64, 19, 21, 40, 3, 2), 1), ((2, 20, 11, 9, 24, 3, 1), 0), ((1, 16, 33, 18, 32, 3, 2), 0)]


@pytest.mark.parametrize("res", [False, True], ids=["plain", "res"])
@pytest.mark.parametrize("form,mode", GEMM, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
@pytest.mark.parametrize("tile", range(len(X3_TILES)))
def test_gemm_tiles(hip, monkeypatch, tile, form, mode, res):
    n, ic, h, w, oc, k, s = form
    x, wt, b = data(n, ic, h, w, oc, k, 100 + tile)
    r = synth.activations((n, oc, (h - 1) // s + 1, (w - 1) // s + 1), 7) if res else None
    exp, mag = conv64(x, wt, b, s, True, r)
    got, names = run(hip, monkeypatch, X3_BASE + tile, x, wt, b, s, True, r)
    assert names == {"igemm_m%d_x3_%dx%d_%d%d" % ((mode,) + X3_TILES[tile])}
    near(got, exp, mag)


# (n, ic, h, w, oc): one pixel, images smaller than a tile, tiles across images, ragged edges; input channels of one
# partial group to three chunks.
PATCH = [(1, 4, 1, 1, 1), (3, 16, 2, 5, 33), (5, 20, 20, 20, 24), (2, 32, 17, 33, 64), (1, 64, 45, 75, 80),
         (2, 80, 9, 16, 96), (1, 144, 8, 8, 128)]


@pytest.mark.parametrize("res", [False, True], ids=["plain", "res"])
@pytest.mark.parametrize("shape", PATCH, ids=lambda v: "x".join(map(str, v)))
@pytest.mark.parametrize("form", range(len(C3_FORMS)))
def test_patch_forms(hip, monkeypatch, form, shape, res):
    n, ic, h, w, oc = shape
    x, wt, b = data(n, ic, h, w, oc, 3, 200 + form)
    r = synth.activations((n, oc, h, w), 8) if res else None
    exp, mag = conv64(x, wt, b, 1, True, r)
    got, names = run(hip, monkeypatch, C3_BASE + form, x, wt, b, 1, True, r)
    assert names == {c3_name(form)}
    near(got, exp, mag)


# (n, ic, h, w, oc): odd and even extents, one pixel, tiles across images, three chunks.
PATCH_S2 = [(1, 4, 1, 1, 1), (3, 16, 2, 5, 33), (5, 20, 20, 20, 24), (2, 32, 35, 66, 64), (1, 80, 45, 75, 96),
            (2, 36, 9, 17, 40)]


@pytest.mark.parametrize("res", [False, True], ids=["plain", "res"])
@pytest.mark.parametrize("shape", PATCH_S2, ids=lambda v: "x".join(map(str, v)))
@pytest.mark.parametrize("form", range(len(C3_FORMS)))
def test_patch_forms_stride_2(hip, monkeypatch, form, shape, res):
    n, ic, h, w, oc = shape
    x, wt, b = data(n, ic, h, w, oc, 3, 250 + form)
    r = synth.activations((n, oc, (h + 1) // 2, (w + 1) // 2), 9) if res else None
    exp, mag = conv64(x, wt, b, 2, True, r)
    got, names = run(hip, monkeypatch, C3_BASE + form, x, wt, b, 2, True, r)
    assert names == {c3_name(form)}
    near(got, exp, mag)


@pytest.mark.parametrize("tile", [X3_BASE + 1, C3_BASE + 3, C3_BASE + 5], ids=["gemm", "patch", "patch_ks4"])
@pytest.mark.parametrize("scale", [0.0, 1e-30, 1e-6, 3e4, 1e30], ids=str)
def test_scales(hip, monkeypatch, tile, scale):
    """Magnitudes outside the first guess of the scale, the second half of the
    channels 2^12 times larger (the sums so far change scale), and one value
    10^6 times the others."""
    x, wt, b = data(1, 128, 12, 20, 40, 3, 300)
    x = (x * np.float32(scale)).astype(np.float32)
    x[:, 64:] *= np.float32(4096)
    x[0, 5, 3, 4] *= np.float32(1e6)
    b = b * np.float32(0)
    exp, mag = conv64(x, wt, b, 1, False, None)
    got, _ = run(hip, monkeypatch, tile, x, wt, b, 1, False)
    near(got, exp, mag, 1e-45)


@pytest.mark.parametrize("tile", [X3_BASE + 1, C3_BASE + 3, C3_BASE + 5], ids=["gemm", "patch", "patch_ks4"])
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 3.4e38], ids=str)
def test_non_finite_input(hip, monkeypatch, tile, value):
    """Infinities, NaN and the top of the float32 range give what float32
    arithmetic gives, at the outputs that they reach and no others."""
    x, wt, b = data(1, 32, 10, 19, 24, 3, 400)
    x[0, 3, 1, 1] = value
    exp, mag = conv64(x, wt, b, 1, False, None)
    exp = np.where(np.abs(exp) > np.finfo(np.float32).max, np.sign(exp) * np.inf, exp)
    got, _ = run(hip, monkeypatch, tile, x, wt, b, 1, False)
    same_non_finite(got, exp)
    fine = np.isfinite(exp)
    # Elements of a tile that holds such a value are computed in float32.
    assert (np.abs(got[fine] - exp[fine]) <= 2.0 ** -17 * mag[fine]).all()


def same_non_finite(got, exp):
    np.testing.assert_array_equal(np.isnan(got), np.isnan(exp))
    np.testing.assert_array_equal(np.isposinf(got), np.isposinf(exp))
    np.testing.assert_array_equal(np.isneginf(got), np.isneginf(exp))


@pytest.mark.parametrize("value", [np.inf, np.nan], ids=str)
def test_non_finite_weight_keeps_float32(hip, value):
    """A 1x1 convolution with such a weight is tuned over the float32 kernels
    (its grid would otherwise take the split ones)."""
    x, wt, b = data(8, 64, 80, 80, 32, 1, 401)
    wt[5, 3, 0, 0] = value
    exp, mag = conv64(x, wt, b, 1, False, None)
    hip.begin_frame()
    try:
        conv = hip.conv_create(wt, b)
        xv = hip.upload(x)
        y = hip.alloc(8, 32, 80, 80)
        hip.conv(conv, xv, y)
        got = hip.download(y)
    finally:
        hip.end_frame()
    same_non_finite(got, exp)
    fine = np.isfinite(exp)
    assert (np.abs(got[fine] - exp[fine]) <= 2.0 ** -17 * mag[fine]).all()


def test_transposed_conv(hip, monkeypatch):
    """The 2x2 transposed conv's sub-pixel scatter behind a split GEMM tile."""
    monkeypatch.setenv("SIMDYOLO_HIP_TILE", str(X3_BASE + 1))
    ic, oc, h, w = 36, 20, 7, 9
    x = synth.activations((2, ic, h, w), 500)
    wt = synth.activations((ic, oc, 2, 2), 501)
    b = synth.activations((oc,), 502)
    exp = np.einsum("nchw,coij->nohiwj", x.astype(np.float64), wt).reshape(2, oc, 2 * h, 2 * w)
    mag = np.einsum("nchw,coij->nohiwj", np.abs(x).astype(np.float64), np.abs(wt)).reshape(2, oc, 2 * h, 2 * w)
    hip.begin_frame()
    try:
        conv = hip.conv_transpose2x2_create(wt, b)
        hip.conv_set_algo(conv, CONV_IGEMM)
        y = hip.alloc(2, oc, 2 * h, 2 * w)
        hip.conv(conv, hip.upload(x), y)
        got = hip.download(y)
    finally:
        hip.end_frame()
    near(got, exp + b[None, :, None, None], mag + np.abs(b)[None, :, None, None])


@pytest.mark.parametrize("tile", range(len(X3_TILES)))
def test_upsampled_part(hip, monkeypatch, tile):
    """A 1x1 conv whose first 64 channels come from a half-resolution view."""
    monkeypatch.setenv("SIMDYOLO_HIP_AUTOTUNE", "0")
    monkeypatch.setenv("SIMDYOLO_HIP_TILE", str(X3_BASE + tile))
    n, cu, c, h, w, oc = 2, 64, 20, 14, 18, 40
    xu, x = synth.activations((n, cu, h // 2, w // 2), 600), synth.activations((n, c, h, w), 601)
    _, wt, b = data(n, cu + c, h, w, oc, 1, 602)
    full = np.concatenate([xu.repeat(2, 2).repeat(2, 3), x], 1)
    exp, mag = conv64(full, wt, b, 1, True, None)
    hip.begin_frame()
    try:
        conv = hip.conv_create(wt, b, silu=True)
        xv = hip.alloc(n, cu + c, h, w)
        hip.upload(x, xv.slice(cu, c))
        xuv = hip.upload(xu)
        yv = hip.alloc(n, oc, h, w)
        hip.profile_enable(True)
        hip.profile_read()
        try:
            hip.conv_upsampled(conv, xuv, xv, yv)
            hip.flush()
            names = set(hip.profile_read())
        finally:
            hip.profile_enable(False)
        got = hip.download(yv)
    finally:
        hip.end_frame()
    assert names == {"igemm_m3_x3_%dx%d_%d%d" % X3_TILES[tile]}
    near(got, exp, mag)


def within(got, exp, mag):
    """Float32-like: 2^-17 of the sum of the magnitudes that the output itself
    reads (K <= 576 rounded float32 terms), whatever else its tile holds."""
    off = np.abs(got.astype(np.float64) - exp)
    assert np.isfinite(got).all() and (off <= 2.0 ** -17 * mag).all(), (off / (2.0 ** -17 * mag + 1e-300)).max()


# kernel, (ic, h, w, oc, k, stride): every addressing mode of the GEMM; the patch kernel at both strides, with
# one chunk of channels, several, and channel groups shared out over four and eight waves.
RANGE = [(X3_BASE + 1, (64, 12, 20, 40, 1, 1)), (X3_BASE + 3, (32, 9, 14, 24, 3, 1)), (X3_BASE + 4, (20, 9, 14, 24, 3, 2)),
         (X3_BASE + 0, (96, 10, 13, 132, 1, 1)), (C3_BASE + 0, (64, 12, 20, 72, 3, 1)), (C3_BASE + 1, (48, 9, 14, 24, 3, 1)),
         (C3_BASE + 4, (16, 9, 14, 40, 3, 1)), (C3_BASE + 0, (20, 17, 21, 24, 3, 2)), (C3_BASE + 3, (64, 12, 20, 40, 3, 2)),
         (C3_BASE + 5, (64, 9, 14, 24, 3, 1)), (C3_BASE + 6, (60, 9, 14, 40, 3, 1)), (C3_BASE + 5, (64, 12, 20, 40, 3, 2))]
RANGE_IDS = [f"{t}-" + "x".join(map(str, f)) for t, f in RANGE]


def range_case(form, seed):
    ic, h, w, oc, k, s = form
    x, wt, b = data(2, ic, h, w, oc, k, seed)
    r = synth.activations((2, oc, (h - 1) // s + 1, (w - 1) // s + 1), seed + 3)
    return x, wt, b, s, r


@pytest.mark.parametrize("value", [6e4, 1e10, 1e20], ids=str)
@pytest.mark.parametrize("tile,form", RANGE, ids=RANGE_IDS)
def test_outlier_leaves_other_outputs(hip, monkeypatch, tile, form, value):
    """One large value in image 0: its own outputs, the other pixels of its
    image and the other image are as close to float64 as float32 would be."""
    x, wt, b, s, r = range_case(form, 700)
    x[0, 3, 1, 1] = value
    exp, mag = conv64(x, wt, b, s, True, r)
    got, _ = run(hip, monkeypatch, tile, x, wt, b, s, True, r)
    within(got, exp, mag)


@pytest.mark.parametrize("small", [1e-4, 1e-7, 1e-30], ids=str)
@pytest.mark.parametrize("large", [1.0, 1e3])
@pytest.mark.parametrize("tile,form", RANGE, ids=RANGE_IDS)
def test_images_of_far_apart_magnitudes(hip, monkeypatch, tile, form, large, small):
    x, wt, b, s, _ = range_case(form, 800)
    x[0] *= np.float32(large)
    x[1] *= np.float32(small)
    b *= np.float32(0)
    exp, mag = conv64(x, wt, b, s, False, None)
    got, _ = run(hip, monkeypatch, tile, x, wt, b, s, False)
    within(got, exp, mag)


@pytest.mark.parametrize("tile,form", RANGE, ids=RANGE_IDS)
def test_small_pixels_among_zeros(hip, monkeypatch, tile, form):
    """Pixels of 1e-9 in an image of zeros with one pixel of ordinary size."""
    x, wt, b, s, _ = range_case(form, 900)
    x[1] = 0
    x[0, :, :, 4:] = 0
    x[0, :, 2:] *= np.float32(1e-9)
    b *= np.float32(0)
    exp, mag = conv64(x, wt, b, s, False, None)
    got, _ = run(hip, monkeypatch, tile, x, wt, b, s, False)
    within(got, exp, mag)


@pytest.mark.parametrize("value", [np.inf, np.nan, 3.4e38], ids=str)
@pytest.mark.parametrize("tile,form", RANGE, ids=RANGE_IDS)
def test_non_finite_input_modes(hip, monkeypatch, tile, form, value):
    x, wt, b, s, r = range_case(form, 1000)
    x[1, 3, 2, 2] = value
    exp, mag = conv64(x, wt, b, s, False, r)
    exp = np.where(np.abs(exp) > np.finfo(np.float32).max, np.sign(exp) * np.inf, exp)
    got, _ = run(hip, monkeypatch, tile, x, wt, b, s, False, r)
    same_non_finite(got, exp)
    fine = np.isfinite(exp)
    assert (np.abs(got[fine] - exp[fine]) <= 2.0 ** -17 * mag[fine]).all()


@pytest.mark.parametrize("value", [1e10, np.inf], ids=str)
def test_transposed_conv_outlier(hip, monkeypatch, value):
    monkeypatch.setenv("SIMDYOLO_HIP_TILE", str(X3_BASE + 1))
    ic, oc, h, w = 36, 20, 7, 9
    x = synth.activations((2, ic, h, w), 1100)
    x[0, 5, 3, 2] = value
    wt = synth.activations((ic, oc, 2, 2), 1101)
    with np.errstate(invalid="ignore"):
        exp = np.einsum("nchw,coij->nohiwj", x.astype(np.float64), wt).reshape(2, oc, 2 * h, 2 * w)
    mag = np.einsum("nchw,coij->nohiwj", np.abs(x).astype(np.float64), np.abs(wt)).reshape(2, oc, 2 * h, 2 * w)
    hip.begin_frame()
    try:
        conv = hip.conv_transpose2x2_create(wt, np.zeros(oc, np.float32))
        hip.conv_set_algo(conv, CONV_IGEMM)
        y = hip.alloc(2, oc, 2 * h, 2 * w)
        hip.conv(conv, hip.upload(x), y)
        got = hip.download(y)
    finally:
        hip.end_frame()
    same_non_finite(got, exp)
    fine = np.isfinite(exp)
    assert (np.abs(got[fine] - exp[fine]) <= 2.0 ** -17 * mag[fine]).all()


@pytest.mark.parametrize("part", ["upsampled", "rest"])
@pytest.mark.parametrize("value", [1e10, np.inf], ids=str)
def test_upsampled_part_outlier(hip, monkeypatch, value, part):
    monkeypatch.setenv("SIMDYOLO_HIP_AUTOTUNE", "0")
    monkeypatch.setenv("SIMDYOLO_HIP_TILE", str(X3_BASE + 1))
    n, cu, c, h, w, oc = 2, 64, 20, 14, 18, 40
    xu, x = synth.activations((n, cu, h // 2, w // 2), 1200), synth.activations((n, c, h, w), 1201)
    (xu if part == "upsampled" else x)[0, 7, 3, 5] = value
    _, wt, b = data(n, cu + c, h, w, oc, 1, 1202)
    full = np.concatenate([xu.repeat(2, 2).repeat(2, 3), x], 1)
    exp, mag = conv64(full, wt, b, 1, False, None)
    hip.begin_frame()
    try:
        conv = hip.conv_create(wt, b)
        xv = hip.alloc(n, cu + c, h, w)
        hip.upload(x, xv.slice(cu, c))
        yv = hip.alloc(n, oc, h, w)
        hip.conv_upsampled(conv, hip.upload(xu), xv, yv)
        got = hip.download(yv)
    finally:
        hip.end_frame()
    same_non_finite(got, exp)
    fine = np.isfinite(exp)
    assert (np.abs(got[fine] - exp[fine]) <= 2.0 ** -17 * mag[fine]).all()


# (ic, h, w, oc, kernel, strides, pads, dilation): forms that only the GEMM runs.
GENERAL = [(16, 13, 17, 24, (3, 3), (1, 1), (2, 2, 2, 2), (2, 2)), (32, 11, 9, 40, (1, 3), (1, 1), (0, 1, 0, 1), (1, 1)),
           (20, 12, 15, 33, (3, 2), (3, 1), (0, 1, 2, 0), (1, 1)), (64, 17, 18, 32, (5, 5), (4, 3), (2, 2, 2, 2), (1, 1))]


@pytest.mark.parametrize("form", GENERAL, ids=lambda f: "x".join(map(str, f[:4])) + "k%dx%d" % f[4])
@pytest.mark.parametrize("tile", range(len(X3_TILES)))
def test_gemm_general_geometry(hip, monkeypatch, tile, form):
    ic, h, w, oc, k, s, pads, d = form
    monkeypatch.setenv("SIMDYOLO_HIP_TILE", str(X3_BASE + tile))
    x = synth.activations((2, ic, h, w), 1300)
    wt, b = synth.kaiming((oc, ic) + k, 1301), synth.activations((oc,), 1302) * np.float32(0.1)
    top, left, bottom, right = pads
    xp = np.pad(x.astype(np.float64), ((0, 0), (0, 0), (top, bottom), (left, right)))
    oh, ow = [(n - e * (q - 1) - 1) // t + 1 for n, q, t, e in zip(xp.shape[2:], k, s, d)]
    exp = np.zeros((2, oc, oh, ow)) + b[None, :, None, None]
    mag = np.abs(exp)
    for i in range(k[0]):
        for j in range(k[1]):
            t = xp[:, :, i * d[0]:i * d[0] + s[0] * (oh - 1) + 1:s[0], j * d[1]:j * d[1] + s[1] * (ow - 1) + 1:s[1]]
            exp += np.einsum("nchw,oc->nohw", t, wt[:, :, i, j].astype(np.float64))
            mag += np.einsum("nchw,oc->nohw", np.abs(t), np.abs(wt[:, :, i, j]).astype(np.float64))
    hip.begin_frame()
    try:
        conv = hip.conv_create(wt, b, s, pads, d)
        hip.conv_set_algo(conv, CONV_IGEMM)
        assert hip.conv_out_size(conv, h, w) == (oh, ow)
        y = hip.alloc(2, oc, oh, ow)
        hip.conv(conv, hip.upload(x), y)
        got = hip.download(y)
    finally:
        hip.end_frame()
    near(got, exp, mag)


# (n, ic, h, w, oc, k, stride): sizes that only the split kernels are timed at.
@pytest.mark.parametrize("form", [(8, 36, 76, 80, 32, 1, 1), (8, 36, 150, 146, 40, 3, 2)], ids=["1x1", "3x3s2"])
def test_capture_with_the_choice_of_another_conv(hip, form):
    """A convolution that runs first inside a capture, of a shape that another
    one tuned: its split weights are not packed yet, and packing uploads."""
    n, ic, h, w, oc, k, s = form
    x, wt, b = data(n, ic, h, w, oc, k, 1400)
    w2 = synth.kaiming((oc, ic, k, k), 1410)
    xs = [x] + [synth.activations(x.shape, 1411 + i) for i in range(2)]
    hip.begin_frame()
    try:
        first, second = (hip.conv_create(t, b, (s, s), (k // 2,) * 4) for t in (wt, w2))
        xv = hip.upload(x)
        yv = hip.alloc(n, oc, *hip.conv_out_size(first, h, w))
        hip.conv(first, xv, yv)
        near(hip.download(yv), *conv64(x, wt, b, s, False, None))
        hip.graph_begin()
        try:
            hip.conv(second, xv, yv)
        finally:
            g = hip.graph_end()
        for x in xs:
            hip.upload(x, xv)
            hip.graph_launch(g)
            near(hip.download(yv), *conv64(x, w2, b, s, False, None))
        # Outside the capture it takes the recorded choice.
        hip.profile_enable(True)
        hip.profile_read()
        try:
            hip.conv(second, xv, yv)
            hip.flush()
            names = set(hip.profile_read())
        finally:
            hip.profile_enable(False)
        assert all("_x3_" in name for name in names), names
        near(hip.download(yv), *conv64(xs[-1], w2, b, s, False, None))
    finally:
        hip.end_frame()


def test_tuning_tables_of_other_forms_are_refused(hip, tmp_path):
    """A saved table numbers the kernels: one whose lists were of another
    length, or from before the split kernels, would name others."""
    table, other = tmp_path / "table.txt", tmp_path / "other.txt"
    hip.tune_save(str(table))
    hip.tune_load(str(table))
    head, *rows = table.read_text().splitlines()
    kind, fields = head.split()[:2], head.split()[2:]
    changed = [kind + fields[:i] + [str(int(fields[i]) + 1)] + fields[i + 1:] for i in range(len(fields))]
    for old in changed + [[kind[0], "tune2"] + fields[:2]]:
        other.write_text("\n".join([" ".join(old)] + rows) + "\n")
        with pytest.raises(SyError):
            hip.tune_load(str(other))
    other.write_text("\r\n".join([head] + rows) + "\r\n")
    hip.tune_load(str(other))


def test_patch_choice_at_a_wide_pitch(hip, tmp_path):
    """A 3x3 choice is kept by shape: the same call on views whose pitch passes the patch kernel's 32-bit offsets
    (two images of 512 MiB) takes the routing rule."""
    n, ic, h, w, oc = 2, 32, 256, 258, 32
    x, wt, b = data(n, ic, h, w, oc, 3, 1500)
    exp, mag = conv64(x, wt, b, 2, False, None)
    table = tmp_path / "table.txt"
    hip.begin_frame()
    try:
        y = hip.alloc(n, oc, h // 2, w // 2)
        narrow, wide = (hip.alloc(n, pitch, h, w).slice(0, ic) for pitch in (ic, 2048))
        hip.upload(x, narrow)
        hip.upload(x, wide)
        hip.conv(hip.conv_create(wt, b, (2, 2), (1, 1, 1, 1)), narrow, y)
        # The tuned choice of this shape: form 3 of the patch kernel, whichever won.
        hip.tune_save(str(table))
        rows = table.read_text().splitlines()
        rows = [r.split()[0] + f" {CONV_IGEMM} {C3_BASE + 3} 1" if f":{n},{h},{w},0 " in r else r for r in rows]
        table.write_text("\n".join(rows) + "\n")
        hip.tune_load(str(table))
        conv = hip.conv_create(wt, b, (2, 2), (1, 1, 1, 1))
        names = []
        for xv in (narrow, wide):
            hip.profile_enable(True)
            hip.profile_read()
            try:
                hip.conv(conv, xv, y)
                hip.flush()
                names.append(set(hip.profile_read()))
            finally:
                hip.profile_enable(False)
            within(hip.download(y), exp, mag)
        assert names[0] == {c3_name(3)} and not any(k.startswith("conv3_x3_") for k in names[1]), names
    finally:
        hip.end_frame()
