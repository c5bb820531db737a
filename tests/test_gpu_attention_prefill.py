"""Prompt attention on the matrix cores in every workgroup shape: ends of key tiles (rows past the last key are zeros from the buffer), the
reference of the exponents that moves late or never, and weights below the normal f16 range, against 64 bits."""
import numpy as np
import pytest

from kalosm_amd._lib import F16, F32, MASK_CAUSAL, check
from kalosm_amd.fusor import MaskKind, Tensor

pytestmark = pytest.mark.gpu


def exact(q, k, v, scale, causal):
    h, g, t, s = q.shape[1], k.shape[1], q.shape[2], k.shape[2]
    q, k, v = (a[0].astype(np.float64) for a in (q, k, v))
    z = q @ np.repeat(k, h // g, 0).transpose(0, 2, 1) * scale
    if causal:
        z[:, np.arange(s)[None] > np.arange(t)[:, None] + s - t] = -np.inf
    e = np.exp(z - z.max(2, keepdims=True))
    return (e / e.sum(2, keepdims=True)) @ np.repeat(v, h // g, 0)


def run(dev, q, k, v, dtype, scale, causal, shape):
    dev.set_option("attn_kernel", shape)
    try:
        qt, kt, vt = (Tensor.from_slice(dev, a, dtype) for a in (q, k, v))
        return qt.flash_attention(kt, vt, scale, MaskKind.Causal if causal else None).as_slice()[0].astype(np.float64)
    finally:
        dev.set_option("attn_kernel", 0)


def close(got, want, dtype, scores):
    """f16: weights, values and outputs each rounded by at most 2^-11 of themselves, against the outputs' root mean square: weights of
    a row add up to one, so their roundings move an output by less than 2^-11 of the largest value (4.5 of N(0, 1)).  f32: the operands keep 22
    bits, a score of size `scores` and so its weight an error of scores * 2^-21."""
    tol = 2.0 ** -11 * (4.5 + 2 * np.abs(want)) if dtype == "f16" else 4.5 * 2.0 ** -21 * (2 + scores)
    assert np.isfinite(got).all() and (np.abs(got - want) <= tol).all(), np.abs(got - want).max()


@pytest.mark.parametrize("dtype", ["f16", "f32"])
@pytest.mark.parametrize("shape", [0, 6, 7, 8, 9])
@pytest.mark.parametrize("t,s,d,causal", [(33, 33, 128, True), (64, 64, 64, True), (129, 129, 128, True), (200, 331, 128, True), (257, 257, 64, False),
                                          (40, 127, 128, False), (383, 383, 128, True)])
def test_every_shape_at_the_ends_of_its_tiles(dev, dtype, shape, t, s, d, causal):
    rng = np.random.default_rng(t * 1000 + s)
    q, k, v = (rng.standard_normal((1, n, m, d)).astype(np.float16 if dtype == "f16" else np.float32) for n, m in ((4, t), (2, s), (2, s)))
    want = exact(q, k, v, d ** -0.5, causal)
    close(run(dev, q, k, v, dtype, d ** -0.5, causal, shape), want, dtype, 6)


@pytest.mark.parametrize("dtype", ["f16", "f32"])
@pytest.mark.parametrize("shape", [6, 7, 8, 9])
@pytest.mark.parametrize("steps", [[0.0, 4.0, 11.0, 11.5], [9.0, 0.0, 0.0, -3.0], [0.0, 7.0, 14.0, 21.0, 28.0, 35.0]])
def test_reference_of_the_exponents(dev, dtype, shape, steps):
    """A maximum that grows by less, by just less and by more than 2^8 (in powers of two) from one tile of keys to the next, or falls; far below it
    are thousands of weights of 2^-17, which are subnormal in f16 and still make up a part of the denominator."""
    rng = np.random.default_rng(len(steps))
    d, tiles = 128, len(steps)
    s = 128 * tiles + 3000
    q = np.zeros((1, 4, 70, d), np.float32)
    q[..., 0] = 1.0
    k = np.zeros((1, 2, s, d), np.float32)
    top = max(steps)
    k[0, :, :, 0] = top - 17
    for i, x in enumerate(steps):
        k[0, :, 128 * i + 64, 0] = x
    k[0, :, :, 0] = np.round(k[0, :, :, 0] * np.log(2.0) * 64) / 64  # exact in f16
    v = (1 + 0.25 * rng.standard_normal((1, 2, s, d))).astype(np.float32)
    if dtype == "f16":
        q, k, v = (a.astype(np.float16) for a in (q, k, v))
    want = exact(q, k, v, 1.0, False)
    got = run(dev, q, k, v, dtype, 1.0, False, shape)
    # subnormal weights, and what is left of them for the second operand of f32, are multiples of 2^-24: each is off by up to 2^-25, s of them
    tol = (2.0 ** -10 * np.abs(want).max() if dtype == "f16" else 2.0 ** -20 * (2 + top)) + s * 2.0 ** -25
    assert np.abs(got - want).max() <= tol, np.abs(got - want).max()


@pytest.mark.parametrize("shape", [0, 6, 7, 8, 9])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("below", [25.5, 24.6])
@pytest.mark.parametrize("dtype,s", [("f32", 16384), ("f16", 131072)])
def test_denominator_of_small_weights(dev, dtype, s, below, d, shape):
    """f16 keys, one of them ahead of all others by 2^25.5 or 2^24.6: weights that f16 rounds to zero, or to 2^-24.  They are in the denominator as they are;
    values of 1 and -1 in turn take them out of the numerator, exactly.  Left are the roundings of a sum between 1 and 2, 2^-24 a tile of 64 keys, of
    exponents and outputs.  Weights rounded ahead of the sum move it by 1.6e-4 (s = 16384, where 1.7e-5 are allowed) and 1.3e-3 (6.1e-4) at least."""
    q, k, v = (np.zeros((1, n, m, d), np.float16) for n, m in ((4, 64), (2, s), (2, s)))
    q[..., 0] = 1.0
    k[..., 0] = np.float16(-below * np.log(2.0))
    k[0, :, 3, 0] = 0.0
    v[..., 0::2, :], v[..., 1::2, :] = 1.0, -1.0
    v[0, :, 2, :], v[0, :, 3, :] = 0.0, 0.75  # (and the leading key's neighbour, so that as many are 1 as are -1)
    tail = (s - 1) * np.exp(float(k[0, 0, 0, 0]))
    qt, kt, vt = Tensor.from_slice(dev, q.astype(np.float32) if dtype == "f32" else q, dtype), Tensor.from_slice(dev, k, "f16"), Tensor.from_slice(dev, v, "f16")
    dev.set_option("attn_kernel", shape)
    try:
        got = qt.flash_attention(kt, vt, 1.0).as_slice().astype(np.float64)
    finally:
        dev.set_option("attn_kernel", 0)
    want = 0.75 / (1.0 + tail)
    assert np.abs(got - want).max() <= want * (s / 64 * 2.0 ** -24 + 2.0 ** -20 + (2.0 ** -11 if dtype == "f16" else 0)), (got.max() / want - 1, got.min() / want - 1)


@pytest.mark.parametrize("qt,kt,kernel", [("f32", "f16", 0), ("f16", "f16", 0), ("f32", "f32", 0), ("f32", "f32", 2)])
@pytest.mark.parametrize("view,t,s,d", [("odd", 33, 200, 128), ("odd", 129, 129, 64), ("odd", 70, 70, 128), ("back", 129, 129, 128), ("back", 40, 63, 64),
                                        ("far", 33, 66, 64)])
def test_views_of_any_address_and_stride(dev, view, qt, kt, kernel, t, s, d):
    """K and V that begin one element behind an address of 16 bytes, whose positions run backwards, or are 2^21 elements apart, as a caller in C may pass them;
    the elements around them are not finite."""
    rng = np.random.default_rng(t + s + d)
    q, k, v = (rng.standard_normal((1, n, m, d)).astype(np.float16 if ty == "f16" else np.float32) for n, m, ty in ((4, t, qt), (2, s, kt), (2, s, kt)))
    if kt == "f16" or kernel == 2:
        q, k, v = (a.astype(np.float16).astype(a.dtype) for a in (q, k, v))
    want = exact(q, k, v, d ** -0.5, True)
    qd, out, size = Tensor.from_slice(dev, q, qt), Tensor(dev, q.shape, qt), k.itemsize
    if view == "far": # both heads of K, then both of V, at each position
        sh, st, held = d, 1 << 21, np.zeros((s, 1 << 21), k.dtype)
        for i, a in enumerate((k, v)):
            held[:, 2 * d * i:2 * d * (i + 1)] = a[0].transpose(1, 0, 2).reshape(s, 2 * d)
        base = [Tensor.from_slice(dev, held, kt)]
        ptr = [base[0].ptr, base[0].ptr + 2 * d * size]
    else:
        at, sh, st = 1 if view == "odd" else 0, s * d, d if view == "odd" else -d
        base, ptr = [], []
        for a in (k, v):
            held = np.full(2 * s * d + 64, np.nan, k.dtype)
            held[at:at + 2 * s * d] = (a if view == "odd" else a[:, :, ::-1]).reshape(-1)
            base.append(Tensor.from_slice(dev, held, kt))
            ptr.append(base[-1].ptr + (at if view == "odd" else (s - 1) * d) * size)
    code = {"f32": F32, "f16": F16}
    dev.set_option("attn_kernel", kernel)
    try:
        check(dev._lib.fh_flash_attention_ex(dev._h, code[qt], code[kt], qd.ptr, 4 * t * d, t * d, d, ptr[0], ptr[1], 0, sh, st, 1, 4, 2, t, s, d, d ** -0.5,
                                             MASK_CAUSAL, None, out.ptr))
    finally:
        dev.set_option("attn_kernel", 0)
    close(out.as_slice()[0].astype(np.float64), want, "f16" if kernel else kt, 6)


@pytest.mark.parametrize("shape", [0, 6, 7, 8, 9])
@pytest.mark.parametrize("dtype", ["f16", "f32"])
def test_rows_are_their_own(dev, dtype, shape):
    """A row's bits do not depend on what the rows beside it hold: not on scores of theirs that grow from tile to tile, not on infinities or NaN."""
    rng = np.random.default_rng(9)
    q, k, v = (rng.standard_normal((1, n, m, 128)).astype(np.float16 if dtype == "f16" else np.float32) for n, m in ((4, 70), (2, 700), (2, 700)))
    base = run(dev, q, k, v, dtype, 128 ** -0.5, False, shape)
    q[0, :, 5] *= 30
    q[0, 1, 40, 3], q[0, 2, 41, 4] = np.inf, np.nan
    got = run(dev, q, k, v, dtype, 128 ** -0.5, False, shape)
    rest = [r for r in range(70) if r not in (5, 40, 41)]
    assert np.array_equal(got[:, rest], base[:, rest])
    assert not np.array_equal(got[:, 5], base[:, 5]) and np.isfinite(got[:, 5]).all() and np.isnan(got[2, 41]).all()


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("t,s", [(33, 128), (33, 129), (129, 129), (200, 331), (128, 384)])
def test_f32_rounded_to_f16(dev, t, s, d, causal):
    """attn_kernel = 2: f32 operands rounded to f16, from 129 keys on in two key groups.  (Values of f16, so that the rounding changes none of them.)"""
    rng = np.random.default_rng(t + s + d)
    q, k, v = (rng.standard_normal((1, n, m, d)).astype(np.float16).astype(np.float32) for n, m in ((4, t), (2, s), (2, s)))
    close(run(dev, q, k, v, "f32", d ** -0.5, causal, 2), exact(q, k, v, d ** -0.5, causal), "f16", 6)
