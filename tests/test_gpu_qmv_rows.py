"""Products of a few rows in one launch: every cut (row tiles a wavefront, 256s a workgroup, parts of k that the last workgroup adds) at the ends of its
tiles and parts, against 64 bits; which products take it; repeats, captured ones among them, and rows that do not mix."""
import numpy as np
import pytest

from kalosm_amd import synth
from kalosm_amd.fusor import QMatrix, Tensor

pytestmark = pytest.mark.gpu
TYPES = [synth.Q4_0, synth.Q5_0, synth.Q8_0, synth.Q4_K, synth.Q5_K, synth.Q6_K]
named = pytest.mark.parametrize("ty", TYPES, ids=lambda t: synth.TYPE_NAMES[t])


class options:
    def __init__(self, dev, **kv):
        self.dev, self.kv = dev, kv

    def __enter__(self):
        for k, v in self.kv.items():
            self.dev.set_option(k, v)

    def __exit__(self, *_):
        for k in self.kv:
            self.dev.set_option(k, 0)


def matrix(dev, oracle, ty, n, k, seed=1):
    raw = synth.random_weight(ty, n, k, seed=seed)
    return QMatrix.from_raw_bytes(dev, (n, k), raw, ty), oracle.dequantize(ty, raw).reshape(n, k).astype(np.float64)


def close(got, x, w):
    """An activation keeps 22 bits, a product is exact, and a sum of f32 takes at most 16 roundings to a value's place in a 256 (two operands, eight blocks,
    scale, offset and factor) and a dozen behind it: 2^-19 of the sum of magnitudes, a hundredth of which is what random signs leave."""
    x = x.astype(np.float64)
    err = np.abs(got - x @ w.T)
    assert np.isfinite(got).all() and (err <= 2.0 ** -19 * (np.abs(x) @ np.abs(w).T)).all()
    assert np.sqrt((err ** 2).mean()) <= 3e-7 * np.sqrt(((x * x) @ (w * w).T).mean())


@named
@pytest.mark.parametrize("cut", [1, 2, 3, 4, 9, 10, 11, 12])
@pytest.mark.parametrize("m,n,k", [(16, 272, 256 * 9), (5, 33, 256 * 4), (2, 600, 256 * 8), (13, 130, 256), (7, 1040, 256 * 21)])
def test_every_cut(dev, oracle, ty, cut, m, n, k):
    q, w = matrix(dev, oracle, ty, n, k)
    x = synth.random_activation(m, k, seed=2) * np.exp(np.random.default_rng(3).standard_normal((m, 1))).astype(np.float32)
    with options(dev, matvec_direct=3, matvec_tiles=cut):
        close(Tensor.from_slice(dev, x).q_mat_mul(q).as_slice().astype(np.float64), x, w)


@named
@pytest.mark.parametrize("m,n,k,taken", [(16, 512, 2048, True), (5, 4096, 1024, True), (4, 512, 2048, False), (6, 40000, 2048, False)])
def test_rule(dev, oracle, ty, m, n, k, taken):
    """Either side of its lines: the bits of one launch, or of others."""
    if ty == synth.Q6_K and m == 4:
        taken = True
    q, _ = matrix(dev, oracle, ty, n, k)
    xt = Tensor.from_slice(dev, synth.random_activation(m, k, seed=2))
    auto = xt.q_mat_mul(q).as_slice()
    with options(dev, matvec_direct=3):
        one = xt.q_mat_mul(q).as_slice()
    assert np.array_equal(auto, one) == taken


@pytest.mark.parametrize("ty,m,n,k,cut", [(synth.Q4_K, 16, 512, 1536, 0), (synth.Q6_K, 5, 22528, 256, 0), (synth.Q8_0, 5, 22528, 256, 0),
                                          (synth.Q4_0, 5, 14336, 2560, 0), (synth.Q5_K, 16, 8192, 5376, 0), (synth.Q4_K, 16, 4096, 11008, 8 + 4),
                                          (synth.Q4_0, 16, 1408, 16384, 8 + 2), (synth.Q6_K, 16, 512, 1024, 1)])
def test_level_or_slower(dev, ty, m, n, k, cut):
    """Products that stay with the kernels they had, for which one launch is level or slower (cut 0), and cuts that keep it quicker: many 256s in parts of
    eight rather than in more parts of four, few of them four to a workgroup."""
    q = QMatrix.from_raw_bytes(dev, (n, k), synth.random_weight(ty, n, k, seed=1), ty)
    xt = Tensor.from_slice(dev, synth.random_activation(m, k, seed=2))
    auto = xt.q_mat_mul(q).as_slice()
    with options(dev, **(dict(matvec_direct=3, matvec_tiles=cut) if cut else dict(matvec_rows=1))):  # (any option of matvecs keeps it off the one launch)
        assert np.array_equal(auto, xt.q_mat_mul(q).as_slice())


@named
def test_small_groups_beside_a_large_one(dev, oracle, ty):
    """Weights that are zero where the activations are large, in 32 of a 256: hi + lo keeps an activation to 2^-22 of itself or to 2^-39 of the largest with which
    it shares a power of two.  The 5-bit formats have one per 32 and lose nothing of the small ones beside 2^28 times as much (with one per 256 an output is
    off by 2^-15 of the sum of magnitudes, where 2^-19 is allowed); the others have one per 256 and 2^14."""
    n, k, m, own = 64, 2048, 6, ty in (synth.Q5_0, synth.Q5_K)
    size = synth.BLOCK_ELEMS[ty]
    blocks = synth.random_weight(ty, n, k, seed=4).reshape(n, k // size, -1).copy()
    if size == 32:
        blocks[:, 0] = 0  # a block of zeros: scale zero
    elif ty == synth.Q6_K:
        blocks[:, 0, 192:194] = 0  # scales of the first two sixteens
    else:
        blocks[:, 0, [4, 8]] &= 0xC0  # scale and offset of the first 32
    raw = np.ascontiguousarray(blocks).reshape(-1)
    w = oracle.dequantize(ty, raw).reshape(n, k).astype(np.float64)
    assert not w[:, :32].any() and w[:, 32:256].any()
    x = synth.random_activation(m, k, seed=5)
    x[:, :32] *= np.float32(2.0 ** (28 if own else 14))
    q = QMatrix.from_raw_bytes(dev, (n, k), raw, ty)
    with options(dev, matvec_direct=3):
        got = Tensor.from_slice(dev, x).q_mat_mul(q).as_slice().astype(np.float64)
    x = x.astype(np.float64)
    tol = 2.0 ** -19 * (np.abs(x) @ np.abs(w).T)
    if not own:
        tol += 2.0 ** -38 * np.abs(x).max(1)[:, None] * np.abs(w[:, :256]).sum(1)
    assert (np.abs(got - x @ w.T) <= tol).all()


@named
def test_repeats_and_rows(dev, oracle, ty):
    """The same bits every time, in a captured launch too (the counters of the parts are zero again behind each); an infinity or a NaN stays in
    its row."""
    n, k, m = 528, 256 * 13, 9
    q, _ = matrix(dev, oracle, ty, n, k)
    x = synth.random_activation(m, k, seed=6)
    xt, y = Tensor.from_slice(dev, x), Tensor(dev, (m, n), "f32")
    with options(dev, matvec_direct=3):
        base = xt.q_mat_mul(q).as_slice()
        dev.graph_begin()
        xt.q_mat_mul(q, out=y)
        graph = dev.graph_end()
        for _ in range(5):
            graph.launch()
            dev.sync()
            assert np.array_equal(y.as_slice(), base)
            assert np.array_equal(xt.q_mat_mul(q).as_slice(), base)
        x[2] = 0.0
        x[3, 7], x[4, 9] = np.inf, np.nan
        got = Tensor.from_slice(dev, x).q_mat_mul(q).as_slice()
    assert not got[2].any() and not np.isfinite(got[3]).any() and np.isnan(got[4]).all()
    rest = [r for r in range(m) if r not in (2, 3, 4)]
    assert np.array_equal(got[rest], base[rest])


@named
@pytest.mark.parametrize("m,n,k,cut", [(5, 528, 256 * 13, 0), (12, 512, 2048, 0), (16, 130, 256, 9), (9, 272, 256 * 9, 2)])
def test_infinities(dev, oracle, ty, m, n, k, cut):
    """An infinite activation gives infinities of the sign of its weight, as f32 arithmetic does, and moves no other row."""
    q, w = matrix(dev, oracle, ty, n, k)
    x = synth.random_activation(m, k, seed=8)
    at = {1: (7, np.inf), 3: (k - 1, -np.inf), 4: (k // 2 + 33, np.inf)}
    with options(dev, matvec_direct=3 if cut else 0, matvec_tiles=cut):
        base = Tensor.from_slice(dev, x).q_mat_mul(q).as_slice()
        for row, (col, value) in at.items():
            x[row, col] = value
        got = Tensor.from_slice(dev, x).q_mat_mul(q).as_slice()
    for row, (col, value) in at.items():
        some = w[:, col] != 0  # (a weight of zero gives NaN)
        assert some.any() and np.array_equal(got[row][some], np.sign(w[some, col]).astype(np.float32) * np.float32(value)), (row, got[row][:4])
    rest = [r for r in range(m) if r not in at]
    assert np.array_equal(got[rest], base[rest])


@named
@pytest.mark.parametrize("m,n,k", [(5, 528, 256 * 13), (16, 512, 2048)])
@pytest.mark.parametrize("size", [1e-30, 1e-34, 1e-36])
def test_tiny_rows(dev, oracle, ty, m, n, k, size):
    """Rows of tiny activations keep their bits: a power of two per 256 reaches 2^126.  Per 32 of k it ends at 2^100, where half of the second operand's last
    place is 2^-125 of an activation."""
    q, w = matrix(dev, oracle, ty, n, k)
    x = synth.random_activation(m, k, seed=9) * np.float32(size)
    with options(dev, matvec_direct=3):
        got = Tensor.from_slice(dev, x).q_mat_mul(q).as_slice().astype(np.float64)
    if ty not in (synth.Q5_0, synth.Q5_K):
        close(got, x, w)
    x = x.astype(np.float64)
    assert (np.abs(got - x @ w.T) <= 2.0 ** -19 * (np.abs(x) @ np.abs(w).T) + 2.0 ** -125 * np.abs(w).sum(1)).all()
