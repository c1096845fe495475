"""The fused attention kernel at the edges of its tiles (32 queries, 32-key
tiles over four waves, key and head dims below its 32 and 64), with non-finite
and far-scaled operands, and the geometry past it that keeps the GEMMs.

Bound: scores carry at most 2^-19 of sum |q||k| scale (products within 2^-24,
32 of them summed in float32), a probability e^(s - m) that error twice, and the
output 2^-19 of the weighted sum of |v| more.
"""
import numpy as np
import pytest

from simdyolo_amd import synth

pytestmark = pytest.mark.gpu


def reference(qkv, heads, kd, hd, scale):
    """(output, bound) in float64, [B, heads * hd, N]."""
    b, _, h, w = qkv.shape
    t = qkv.astype(np.float64).reshape(b, heads, 2 * kd + hd, h * w)
    q, k, v = t[:, :, :kd], t[:, :, kd:2 * kd], t[:, :, 2 * kd:]
    with np.errstate(invalid="ignore", over="ignore"):
        s = np.matmul(q.transpose(0, 1, 3, 2), k) * float(scale)
        off = np.matmul(np.abs(q).transpose(0, 1, 3, 2), np.abs(k)) * float(scale) * 2.0 ** -19 + 2.0 ** -21
        p = np.exp(s - s.max(-1, keepdims=True))
        p /= p.sum(-1, keepdims=True)
        o = np.matmul(v, p.transpose(0, 1, 3, 2))
        bound = np.matmul(np.abs(v), (p * (2 * off.max(-1, keepdims=True) + 2.0 ** -19)).transpose(0, 1, 3, 2))
    return o.reshape(b, heads * hd, h, w), bound.reshape(b, heads * hd, h, w), v.reshape(b, heads * hd, h, w)


def run(hip, qkv, heads, kd, hd, scale):
    b, c, h, w = qkv.shape
    hip.begin_frame()
    try:
        x = hip.alloc(b, c + 8, h, w).slice(4, c)
        hip.upload(qkv, x)
        o = hip.alloc(b, heads * hd + 3, h, w).slice(1, heads * hd)
        v = hip.alloc(b, heads * hd + 5, h, w).slice(2, heads * hd)
        hip.profile_enable(True)
        hip.profile_read()
        try:
            hip.attention(x, heads, kd, hd, float(scale), o, v)
            hip.flush()
            names = set(hip.profile_read())
        finally:
            hip.profile_enable(False)
        return hip.download(o), hip.download(v), names
    finally:
        hip.end_frame()


# (batch, heads, key dim, head dim, h, w): one token, fewer key tiles than waves, one past a tile, ragged dims.
CASES = [(1, 1, 32, 64, 1, 1), (2, 2, 4, 4, 3, 11), (1, 3, 20, 36, 8, 16), (2, 1, 32, 64, 3, 43), (1, 2, 32, 64, 20, 20),
         (1, 2, 28, 60, 33, 31)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
def test_fused(hip, case):
    b, heads, kd, hd, h, w = case
    qkv = synth.activations((b, heads * (2 * kd + hd), h, w), 31 * h + w)
    scale = np.float32(kd ** -0.5)
    exp, bound, vexp = reference(qkv, heads, kd, hd, scale)
    got, v, names = run(hip, qkv, heads, kd, hd, scale)
    assert names == {"attention"}
    np.testing.assert_array_equal(v, vexp.astype(np.float32))
    assert (np.abs(got - exp) <= bound).all(), (np.abs(got - exp) / bound).max()


@pytest.mark.parametrize("scales", [(1e-6, 1e6, 1e-20), (30.0, 1.0, 1e4), (0.0, 1.0, 1.0), (1e-30, 1e-30, 1e-30)], ids=str)
def test_operand_scales(hip, scales):
    """q, k and v far from the first guess of their scales, values that grow by 2^14 over the key tiles."""
    heads, kd, hd = 2, 32, 64
    qkv = synth.activations((1, heads, 2 * kd + hd, 12, 16), 5)
    qkv[:, :, :kd] *= np.float32(scales[0])
    qkv[:, :, kd:2 * kd] *= np.float32(scales[1])
    qkv[:, :, 2 * kd:] *= np.float32(scales[2])
    qkv[:, :, 2 * kd:, 6:] *= np.float32(16384)
    qkv = qkv.reshape(1, -1, 12, 16)
    exp, bound, _ = reference(qkv, heads, kd, hd, np.float32(kd ** -0.5))
    got, _, _ = run(hip, qkv, heads, kd, hd, np.float32(kd ** -0.5))
    floor = 2.0 ** -38 * float(np.abs(qkv.reshape(1, heads, -1, 192)[:, :, 2 * kd:]).max())
    assert (np.abs(got - exp) <= bound + floor).all()


@pytest.mark.parametrize("step", [0.5, 2.0, 3.0, 60.0, -2.0])
def test_creeping_maximum(hip, step):
    """Scores that rise by `step` from one 32-key tile to the next: below, at about and far past the slack within
    which a running maximum stays."""
    heads, kd, hd = 1, 32, 64
    qkv = synth.activations((1, 2 * kd + hd, 20, 24), 8)
    qkv[:, :kd] = np.float32(1.0)
    qkv[:, kd:2 * kd] *= np.float32(0.25)
    qkv[:, kd] += (np.float32(step) * (np.arange(480) // 32)).reshape(20, 24).astype(np.float32)
    exp, bound, _ = reference(qkv, heads, kd, hd, np.float32(1.0))
    got, _, _ = run(hip, qkv, heads, kd, hd, np.float32(1.0))
    assert (np.abs(got - exp) <= bound).all(), (np.abs(got - exp) / bound).max()


@pytest.mark.parametrize("power", [20, 21, 60])
def test_large_scale(hip, power):
    """Past 2^20 the rows are computed in plain float32 (32 products: below the bound of the split)."""
    heads, kd, hd = 2, 32, 64
    qkv = synth.activations((1, heads, 2 * kd + hd, 5, 9), 9)
    qkv[:, :, :kd] *= np.float32(2.0 ** -power)
    qkv = qkv.reshape(1, -1, 5, 9)
    exp, bound, _ = reference(qkv, heads, kd, hd, np.float32(2.0 ** power))
    got, _, _ = run(hip, qkv, heads, kd, hd, np.float32(2.0 ** power))
    assert (np.abs(got - exp) <= bound).all(), (np.abs(got - exp) / bound).max()


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan], ids=str)
@pytest.mark.parametrize("part", ["q", "k", "v"])
def test_non_finite(hip, part, value):
    heads, kd, hd = 1, 32, 64
    qkv = synth.activations((1, 2 * kd + hd, 7, 9), 6)
    qkv[0, {"q": 3, "k": kd + 3, "v": 2 * kd + 3}[part], 2, 5] = value
    exp, _, _ = reference(qkv, heads, kd, hd, np.float32(kd ** -0.5))
    got, _, _ = run(hip, qkv, heads, kd, hd, np.float32(kd ** -0.5))
    np.testing.assert_array_equal(np.isnan(got), np.isnan(exp))
    fine = np.isfinite(exp)
    np.testing.assert_array_equal(got[~fine & ~np.isnan(exp)], exp[~fine & ~np.isnan(exp)])
    np.testing.assert_allclose(got[fine], exp[fine], rtol=0, atol=1e-5)  # 63 products of order 1 in float32


def test_wider_dims_keep_the_gemms(hip):
    heads, kd, hd = 1, 40, 72
    qkv = synth.activations((2, 2 * kd + hd, 9, 7), 7)
    exp, bound, vexp = reference(qkv, heads, kd, hd, np.float32(kd ** -0.5))
    got, v, names = run(hip, qkv, heads, kd, hd, np.float32(kd ** -0.5))
    assert "attn_softmax" in names
    np.testing.assert_array_equal(v, vexp.astype(np.float32))
    assert (np.abs(got - exp) <= bound).all()


@pytest.mark.parametrize("sign", [1.0, -1.0])
@pytest.mark.parametrize("step", [4.0, -4.0, 8.0])
def test_large_scores(hip, sign, step):
    """Scores of 2^25 magnitude, where floats lie 4 apart, in key tiles 0 and 4 (the same wave's): the step between
    the tiles is larger than the slack of the running maximum, but not than the rounding of maximum plus slack."""
    heads, kd, hd = 1, 32, 64
    qkv = synth.activations((1, 2 * kd + hd, 8, 20), 10)
    qkv[:, :kd] = np.float32(sign * 1024)
    qkv[:, kd:2 * kd] = np.float32(1024)
    late = (np.arange(160) >= 128).reshape(8, 20)
    qkv[:, kd, late] += np.float32(sign * step / 1024)
    got, _, _ = run(hip, qkv, heads, kd, hd, np.float32(1.0))
    # Every product and sum of these scores is a float32: no error but the exponentials' and the weighted sum's.
    t = qkv.astype(np.float64).reshape(2 * kd + hd, 160)
    s = t[:kd].T @ t[kd:2 * kd]
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    exp, mag = t[2 * kd:] @ p.T, np.abs(t[2 * kd:]) @ p.T
    err = np.abs(got.reshape(hd, 160) - exp)
    assert np.isfinite(got).all() and (err <= 2.0 ** -18 * mag).all(), (err / mag).max()


@pytest.mark.parametrize("where", ["o in qkv", "o in v"])
def test_output_over_an_operand(hip, where):
    """The output over the query channels of its own input, or over v's copy, is written after all reads."""
    heads, kd, hd = 2, 32, 32
    c = heads * (2 * kd + hd)
    qkv = synth.activations((2, c, 9, 40), 12)
    exp, bound, _ = reference(qkv, heads, kd, hd, np.float32(kd ** -0.5))
    hip.begin_frame()
    try:
        x, v = hip.alloc(2, c, 9, 40), hip.alloc(2, heads * hd, 9, 40)
        o = x.slice(0, heads * hd) if where == "o in qkv" else v
        for _ in range(2):
            hip.upload(qkv, x)
            hip.attention(x, heads, kd, hd, float(np.float32(kd ** -0.5)), o, v)
            got = hip.download(o)
            assert (np.abs(got - exp) <= bound).all(), (np.abs(got - exp) / bound).max()
    finally:
        hip.end_frame()


RANGES = {
    # One query 2^29 times the others', whose own scores are of order 1.
    "queries": lambda q, k, v: (np.where(np.arange(96) == 5, 3e4, 2.0 ** -14) * q, 2.0 ** 14 * k, v),
    # Every query attends to key 40 alone, whose values are 10^-12 of the others'.
    "value rows": lambda q, k, v: (q + 8, np.where(np.arange(96) == 40, 8.0, -1.0) + 0 * k,
                                   np.where(np.arange(96) == 40, 1e-12, 1.0) * v),
    # Channels from 1 down to 10^-20.
    "value channels": lambda q, k, v: (q, k, np.logspace(0, -20, 64)[None, :, None] * v),
    # One value of 10^20: only its channel and no other sees it.
    "outlier": lambda q, k, v: (q, k, np.where((np.arange(96) == 70) & (np.arange(64) == 3)[:, None], 1e20, v)),
    # A sum of 96 such values overflows, their average does not.
    "largest": lambda q, k, v: (q, k, 1e37 * (1 + 0.1 * v)),
}


@pytest.mark.parametrize("name", RANGES)
def test_precision_is_each_operands_own(hip, name):
    """Operands of far-apart magnitudes: every output within the bound of its own products, no floor added."""
    heads, kd, hd = 2, 32, 64
    x = synth.activations((heads, 2 * kd + hd, 96), 11)
    q, k, v = RANGES[name](x[:, :kd], x[:, kd:2 * kd], x[:, 2 * kd:])
    qkv = np.concatenate([np.broadcast_to(t, (heads, d, 96)) for t, d in ((q, kd), (k, kd), (v, hd))], 1)
    qkv = qkv.astype(np.float32).reshape(1, -1, 8, 12)
    exp, bound, _ = reference(qkv, heads, kd, hd, np.float32(kd ** -0.5))
    got, _, _ = run(hip, qkv, heads, kd, hd, np.float32(kd ** -0.5))
    assert np.isfinite(got).all() and (np.abs(got - exp) <= bound).all(), (np.abs(got - exp) / bound).max()
