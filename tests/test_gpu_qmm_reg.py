"""GPU parity: the matmul that decodes weights in registers (csrc/fh_qmm_reg.hip) against a float64 product of the oracle's
dequantised weights.

Bound: the operands are exact up to 2^-22 of each activation; products are added in f32, sixteen times 2 or 3 in a chain within a 256,
then up to eight of those (each with its offsets, which cancel most of it) and the sums of eight; the wide products up to k / 256 of them,
or, with a scale per 32, half of k / 32 (f32 rows: all).  Rounding errors (2^-24 each, of either sign) grow with the
root of their number: 1e-6 of the root of the sum of the squared products (the result's root mean square where there are many of
them; one result alone may be next to nothing by cancellation) covers k = 16384.  The largest single difference is held to ten
times that (ten standard deviations)."""
import numpy as np
import pytest

from kalosm_amd import synth
from kalosm_amd.fusor import Device, QMatrix, Tensor

pytestmark = pytest.mark.gpu
TYPES = [synth.Q4_0, synth.Q5_0, synth.Q8_0, synth.Q4_K, synth.Q5_K, synth.Q6_K]


def operands(dev, ty, m, n, k, act, x=None):
    raw = synth.random_weight(ty, n, k, seed=n + k, sigma=2e-3)
    x = synth.random_activation(m, k, seed=m) if x is None else x
    q = QMatrix.from_raw_bytes(dev, (n, k), raw, ty)
    if act == "f32":
        return q, Tensor.from_slice(dev, x), x, raw
    bits = synth.to_bf16_bits(x)
    return q, Tensor.from_slice(dev, bits, dtype="bf16"), synth.from_bf16_bits(bits), raw


def run(dev, q, xt, option, cut=0):
    out = Tensor.filled_bytes(dev, (xt.shape[0], q.shape()[0]), 0xFF)  # poisoned: unwritten elements show as NaN
    dev.set_option("matmul_kernel", option)
    dev.set_option("matmul_cut", cut)
    try:
        return xt.q_mat_mul(q, out=out).as_slice()
    finally:
        dev.set_option("matmul_kernel", 0)
        dev.set_option("matmul_cut", 0)


def cut_of(mt, kw, parts):
    """Row tiles of activations a workgroup, groups of its wavefronts along k, workgroups along k."""
    return mt + 16 * kw + 256 * parts


@pytest.mark.parametrize("act", ["f32", "bf16"])
@pytest.mark.parametrize("ty", TYPES, ids=lambda t: synth.TYPE_NAMES[t])
@pytest.mark.parametrize("m,n,k,option", [
    (1, 1, 256, 16),       # one row, one output, one 256
    (17, 33, 1280, 16),    # five 256s in parts of their own (how k is shared out otherwise: test_cuts); a second row tile of one row
    (48, 272, 2304, 16),   # three row tiles; nine 256s
    (65, 96, 4096, 16),    # five row tiles in two workgroups of three
    (130, 520, 1024, 16),  # nine row tiles in three workgroups
    (33, 40, 16384, 16),   # the longest k, in parts
    (1, 1, 256, 15),       # the wide products (option 15): the same
    (64, 256, 512, 15),    # exactly a tile
    (65, 257, 768, 15),    # one past it; three 256s
    (515, 80, 4096, 15),   # activations laid out eight rows a workgroup, half of k held by a thread, ...
    (513, 48, 8192, 15),   # ... all of it, ...
    (1027, 33, 8448, 15),  # ... read twice; rows past the last eight
])
def test_product(dev, oracle, ty, act, m, n, k, option):
    q, xt, x, raw = operands(dev, ty, m, n, k, act)
    got = run(dev, q, xt, option).astype(np.float64)
    x, w = x.astype(np.float64), oracle.dequantize(ty, raw).reshape(n, k).astype(np.float64)
    want, rms = x @ w.T, np.sqrt(np.mean((x * x) @ (w * w).T))
    assert np.isfinite(got).all()
    assert np.sqrt(np.mean((got - want) ** 2)) <= 1e-6 * rms
    assert np.abs(got - want).max() <= 1e-5 * rms


@pytest.mark.parametrize("act", ["f32", "bf16"])
@pytest.mark.parametrize("ty", TYPES, ids=lambda t: synth.TYPE_NAMES[t])
@pytest.mark.parametrize("mt", [1, 2, 3, 4])
@pytest.mark.parametrize("kw,parts", [(1, 1), (1, 3), (2, 1), (2, 3), (4, 1), (4, 3)])
def test_cuts(dev, oracle, ty, act, mt, kw, parts):
    """Every way a product can be cut: 13 256s over one to twelve groups (most of them uneven, so that some multiply a 256 with a scale of
    zero), a row tile past the last whole workgroup, weight rows past the last tile of one."""
    m, n, k = 16 * mt + 3, 136, 256 * 13
    q, xt, x, raw = operands(dev, ty, m, n, k, act)
    got = run(dev, q, xt, 16, cut_of(mt, kw, parts)).astype(np.float64)
    x, w = x.astype(np.float64), oracle.dequantize(ty, raw).reshape(n, k).astype(np.float64)
    want, rms = x @ w.T, np.sqrt(np.mean((x * x) @ (w * w).T))
    assert np.isfinite(got).all()
    assert np.sqrt(np.mean((got - want) ** 2)) <= 1e-6 * rms
    assert np.abs(got - want).max() <= 1e-5 * rms


@pytest.mark.parametrize("ty,act,m,n,k,taken", [
    (synth.Q8_0, "bf16", 1, 64, 1024, True), (synth.Q8_0, "bf16", 1, 64, 768, False),
    (synth.Q4_K, "f32", 17, 64, 1024, True), (synth.Q4_K, "f32", 16, 64, 1024, False),
    (synth.Q5_K, "f32", 5, 64, 1024, True), (synth.Q5_0, "f32", 4, 64, 1024, False), (synth.Q5_0, "f32", 12, 64, 768, False),
    (synth.Q4_K, "f32", 511, 8192, 2048, True), (synth.Q4_K, "f32", 512, 8192, 2048, False), (synth.Q4_K, "f32", 640, 64, 2048, True),
    (synth.Q5_0, "f32", 192, 8192, 2048, True), (synth.Q5_0, "f32", 193, 8192, 2048, False),
    (synth.Q8_0, "bf16", 1280, 64, 1024, True), (synth.Q6_K, "f32", 513, 64, 1024, False),
    (synth.Q4_K, "bf16", 1300, 8192, 1024, True), (synth.Q4_K, "bf16", 1300, 1024, 1024, False), (synth.Q4_K, "bf16", 1300, 4096, 8448, False),
    (synth.Q4_K, "f32", 1000, 8192, 1024, True), (synth.Q4_K, "f32", 1000, 8176, 1024, False),
    (synth.Q4_K, "f32", 512, 4096, 2048, True), (synth.Q4_K, "f32", 513, 4096, 2048, True),          # either side of whole tiles of 256 rows
    (synth.Q4_K, "f32", 600, 8192, 2048, False), (synth.Q5_K, "f32", 384, 11008, 2048, False),       # a second round of workgroups: the fragments are quicker
    (synth.Q5_K, "f32", 300, 11008, 2048, True), (synth.Q8_0, "bf16", 1000, 8192, 2048, True),
    (synth.Q8_0, "bf16", 1000, 7168, 8448, False), (synth.Q8_0, "bf16", 1100, 7168, 8448, True),     # 224 whole tiles, 280
    (synth.Q6_K, "bf16", 768, 10880, 1024, False), (synth.Q6_K, "bf16", 640, 4096, 1024, True),
])
def test_rule(dev, ty, act, m, n, k, taken):
    """Both sides of the dispatch's lines: the bits of this kernel (option 14) or others."""
    q, xt, _, _ = operands(dev, ty, m, n, k, act)
    assert np.array_equal(run(dev, q, xt, 0).view(np.uint32), run(dev, q, xt, 14).view(np.uint32)) == taken


@pytest.mark.parametrize("option,cut", [(15, 0), (16, 0), (16, cut_of(3, 4, 1)), (16, cut_of(2, 2, 2))], ids=["wide", "model", "k over 4", "k over 2 x 2"])
@pytest.mark.parametrize("ty,m", [(synth.Q4_K, 40), (synth.Q6_K, 40), (synth.Q8_0, 40), (synth.Q5_0, 12), (synth.Q5_K, 12)],
                         ids=lambda t: synth.TYPE_NAMES.get(t, t))
def test_rows_are_independent(dev, ty, m, option, cut):
    """Zeros stay zero, a power of two passes through exactly, and an infinity or a NaN stays in its row - also where a group of
    wavefronts has fewer 256s than others (five over four), and with a power of two per 32 (12 rows of the 5-bit formats)."""
    n, k = 96, 1280
    x = synth.random_activation(m, k, seed=5)
    q, xt, _, _ = operands(dev, ty, m, n, k, "f32", x.copy())
    base = run(dev, q, xt, option, cut)
    x[3] = 0.0
    x[4] *= np.float32(2.0 ** 20)
    x[5, 7] = np.inf
    x[6, 9] = np.nan
    got = run(dev, q, Tensor.from_slice(dev, x), option, cut)
    assert not got[3].any()
    assert np.array_equal(got[4], base[4] * np.float32(2.0 ** 20))
    assert not np.isfinite(got[5]).any() and np.isnan(got[6]).all()
    rest = [r for r in range(m) if r not in (3, 4, 5, 6)]
    assert np.array_equal(got[rest], base[rest])


@pytest.mark.parametrize("option", [15, 16])
@pytest.mark.parametrize("m", [65, 100])
@pytest.mark.parametrize("ffn", [256, 1280])
def test_swiglu_epilogue(dev, m, ffn, option):
    """gate | up of one launch, SwiGLU at the store, against the two halves as matrices of their own, whose k may be in other
    parts: each product within 1e-6 of the exact one, so two layers of three products within 1e-5 of each other."""
    from kalosm_amd.llama import Model

    cfg = dict(n_layers=2, d_model=1024, n_heads=8, n_kv_heads=4, head_dim=128, ffn=ffn, vocab=320, ctx=256, eps=1e-5, theta=1e4)
    tokens = np.random.default_rng(m).integers(0, 320, m)
    models = [Model.random_init(dev, cfg, seed=2, sigma=2e-3, fuse_gate_up=fuse) for fuse in (True, False)]
    dev.set_option("matmul_kernel", option)
    try:
        got = [model.forward(tokens) for model in models]
    finally:
        dev.set_option("matmul_kernel", 0)
    assert np.isfinite(got[0]).all()
    assert np.sqrt(np.mean((got[0] - got[1]) ** 2)) <= 1e-5 * np.sqrt(np.mean(got[1] ** 2))


@pytest.mark.parametrize("ty", [synth.Q5_0, synth.Q5_K], ids=lambda t: synth.TYPE_NAMES[t])
def test_five_bit_rows_without_memory(ty):
    """5 to 12 rows of the 5-bit formats: where the memory for their activations cannot be had (a bound, a capture ahead of any eager
    call) they are a launch each, which needs none, and with it they leave the graphs of other calls alone."""
    dev = Device.gpu(0)
    try:
        raw = synth.random_weight(ty, 64, 1024, seed=1, sigma=2e-3)
        q = QMatrix.from_raw_bytes(dev, (64, 1024), raw, ty)
        x = synth.random_activation(12, 1024, seed=2)
        xt, out = Tensor.from_slice(dev, x), Tensor(dev, (12, 64))
        rows = np.concatenate([Tensor.from_slice(dev, x[r:r + 1]).q_mat_mul(q).as_slice() for r in range(12)])
        dev.set_option("scratch_limit", 1)
        assert np.array_equal(run(dev, q, xt, 0).view(np.uint32), rows.view(np.uint32))
        dev.set_option("scratch_limit", 0)
        dev.graph_begin()
        xt.q_mat_mul(q, out=out)
        graph = dev.graph_end()
        for _ in range(2):
            in_one = run(dev, q, xt, 0)
            graph.launch()
            assert np.array_equal(out.as_slice().view(np.uint32), rows.view(np.uint32))
        assert not np.array_equal(in_one, rows)
        del graph
    finally:
        dev.close()


def long_sum(dev, ty, option, cut, chunks):
    """2^24 from the first 256 of k and 1 from each other one: an addition of 1 to a sum of 2^24 leaves it as it is."""
    x = np.zeros((1, 256 * chunks), np.float32)
    x[:, ::256] = 1.0
    x[:, 0] = 2.0 ** 24
    raw = np.zeros((16, chunks, 210 if ty == synth.Q6_K else 8 * 34), np.uint8)  # a 256's first weight 1, the others 0
    if ty == synth.Q6_K:
        raw[..., 128:192] = 0xAA  # code 32 for all: 0
        raw[..., 0] = 1
        raw[..., 192:208] = 1
        raw[..., 208:210] = np.array([1.0], np.float16).view(np.uint8)
    else:  # Q8_0
        raw[..., 0:2] = np.array([1.0], np.float16).view(np.uint8)
        raw[..., 2] = 1
    q = QMatrix.from_raw_bytes(dev, (16, 256 * chunks), raw.reshape(-1), ty)
    return run(dev, q, Tensor.from_slice(dev, synth.to_bf16_bits(x), dtype="bf16"), option, cut).astype(np.float64) - 2.0 ** 24


@pytest.mark.parametrize("ty", [synth.Q8_0, synth.Q6_K], ids=lambda t: synth.TYPE_NAMES[t])
def test_partial_planes_are_added_in_pairs(dev, ty):
    """16 planes of one 256 each: one pair loses its 1, the 14 others arrive.  (One after the other: all 15 are lost.)"""
    assert (long_sum(dev, ty, 16, cut_of(1, 1, 16), 16) == 14).all()


@pytest.mark.parametrize("kw,kept", [(1, 56), (4, 60)])
def test_no_sum_is_long(dev, kw, kept):
    """64 times 256, scale per 256: the ones beside 2^24 in its first eight are lost, the 56 others arrive; of four groups of 16, which add up
    in fours, all but three.  One sum along k loses all 63, four of them 15."""
    assert (long_sum(dev, synth.Q6_K, 16, cut_of(1, kw, 1), 64) == kept).all()


@pytest.mark.parametrize("chunks,kept", [(1, 0), (2, 0), (8, 4), (9, 4), (32, 16)])
def test_wide_products_in_two_halves(dev, chunks, kept):
    """Scale per 32, bf16: the ones beside 2^24 in the first half of k are lost, those of the second arrive, up to the last one
    of an odd number.  (One sum along k: none does.)"""
    assert (long_sum(dev, synth.Q8_0, 15, 0, chunks) == kept).all()


@pytest.mark.parametrize("m,n,k,parted", [
    (1040, 8192, 8192, True), (600, 24576, 2048, False),  # the fragments in two parts, in one
    (200, 49152, 2048, True), (200, 32768, 2048, False),  # 384 tiles, the last 128 of them in two parts; 256 tiles
])
def test_f32_products_that_others_part(dev, m, n, k, parted):
    """f32, scale per 32: what the fragments, or the tiles in their last round, would part takes k_qmm_reg (option 16), other products
    k_qmm_wide (15)."""
    q, xt, _, _ = operands(dev, synth.Q4_0, m, n, k, "f32")
    got = {option: run(dev, q, xt, option).view(np.uint32) for option in (0, 15, 16)}
    assert not np.array_equal(got[15], got[16])
    assert np.array_equal(got[0], got[16 if parted else 15])


@pytest.mark.parametrize("ty", [synth.Q5_0, synth.Q5_K], ids=lambda t: synth.TYPE_NAMES[t])
@pytest.mark.parametrize("m", [5, 12])
@pytest.mark.parametrize("cut", [0, cut_of(1, 1, 1), cut_of(1, 2, 2), cut_of(1, 4, 1)])
def test_small_values_beside_large_ones(dev, oracle, ty, m, cut):
    """5 to 12 rows of the 5-bit formats keep every bit of a group of 32 whatever stands in the others, as the kernel for one row
    does: each 256 has a group of values 2^30 times the others', which meet weights of zero.  (Within a row's range of f16 hi + lo the others
    would keep nothing.)  Five 256s, so that groups of wavefronts have unequal numbers of them."""
    n, k = 48, 1280
    raw = synth.random_weight(ty, n, k, seed=3, sigma=2e-3).reshape(n, k // 256, -1)
    if ty == synth.Q5_0:
        raw.reshape(n, k // 256, 8, 22)[:, :, 3, 0:2] = 0  # scale of the fourth 32
    else:
        raw[..., 4 + 3] &= 0xC0      # scale and minimum of the fourth 32: six bits of bytes 3 and 7
        raw[..., 4 + 4 + 3] &= 0xC0
    x = synth.random_activation(m, k, seed=m)
    x.reshape(m, k // 256, 8, 32)[:, :, 3] *= np.float32(2.0 ** 30)
    q = QMatrix.from_raw_bytes(dev, (n, k), raw.reshape(-1), ty)
    got = run(dev, q, Tensor.from_slice(dev, x), 16 if cut else 0, cut).astype(np.float64)
    w = oracle.dequantize(ty, raw.reshape(-1)).reshape(n, k).astype(np.float64)
    assert not w.reshape(n, k // 256, 8, 32)[:, :, 3].any()
    want = x.astype(np.float64) @ w.T
    assert np.sqrt(np.mean((got - want) ** 2)) <= 1e-6 * np.sqrt(np.mean(want ** 2))


@pytest.mark.parametrize("d_model,ffn,m,fused", [(4096, 1024, 65, False), (4096, 1024, 100, False), (1024, 1024, 65, True), (2048, 5632, 65, True)])
def test_swiglu_in_two_launches(dev, d_model, ffn, m, fused):
    """SwiGLU at the store (always with option 14) takes k in one part: only where two launches, with k in several, are not quicker."""
    from kalosm_amd.llama import Model

    cfg = dict(n_layers=1, d_model=d_model, n_heads=d_model // 128, n_kv_heads=d_model // 512, head_dim=128, ffn=ffn, vocab=320, ctx=128, eps=1e-5, theta=1e4)
    model, tokens, got = Model.random_init(dev, cfg, seed=2, sigma=2e-3), np.random.default_rng(m).integers(0, 320, m), []
    for option in (0, 14):
        dev.set_option("matmul_kernel", option)
        try:
            got.append(model.forward(tokens, want_hidden=True)[1].view(np.uint32))
        finally:
            dev.set_option("matmul_kernel", 0)
        model.reset()
    assert np.array_equal(got[0], got[1]) == fused
