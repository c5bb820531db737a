"""GPU parity: one f32 row times bf16 weights (csrc/fh_dense.hip: k_matvec_mix, k_matvec_rows) against float64, over every way
the input takes to the LDS and past the requests that go out ahead.

Bound: f32 products and sums of k terms, a lane's chain of k / 64 of them: rounding errors of 2^-24 of either sign, 1e-6 of the
result's root mean square for k up to 30720, and ten times that for the largest single difference."""
import numpy as np
import pytest

import hybridgen as G
from kalosm_amd import synth
from kalosm_amd.fusor import Device, QMatrix, Tensor
from oracle import hybrid_ref as R
from test_gpu_hybrid import TOL, close, run_portions

pytestmark = pytest.mark.gpu


def near(got, want):
    rms = np.sqrt(np.mean(want * want))
    assert np.sqrt(np.mean((got - want) ** 2)) <= 1e-6 * rms
    assert np.abs(got - want).max() <= 1e-5 * rms


@pytest.mark.parametrize("n,ks", [
    (37, (60, 1024, 1025, 2048, 2112, 4096, 4160, 8195, 14336, 16384, 16452, 30720)),  # a row a wavefront
    (2051, (1000, 1028, 4096, 4102, 4160, 14336, 16448)),                            # two
    (8193, (64, 513, 1024, 1600, 4160)),                                             # four
])
def test_products(dev, n, ks):
    rng = np.random.default_rng(n)
    for k in ks:
        w = synth.to_bf16_bits(rng.standard_normal(n * k, dtype=np.float32))
        x = rng.standard_normal((1, k), dtype=np.float32)
        out = Tensor.filled_bytes(dev, (1, n), 0xFF)
        got = Tensor.from_slice(dev, x).q_mat_mul(QMatrix.from_raw_bytes(dev, (n, k), w, synth.W_BF16), out=out).as_slice()
        near(got[0].astype(np.float64), synth.from_bf16_bits(w).reshape(n, k).astype(np.float64) @ x[0].astype(np.float64))


@pytest.mark.parametrize("width,vocab", [(1000, 40), (2050, 40), (4100, 40), (4160, 2100), (1030, 2100), (520, 8200)])
def test_normed(dev, width, vocab):
    """The output matrix behind the final norm: the normed row that is given back, and its product."""
    cfg = G.config([G.with_mlp(G.delta(1, 1, 16, 16, 4), None)], width, vocab)
    w = G.weights(cfg)
    m = G.build(dev, cfg, w)
    m.keep_layers()
    logits, hidden = m.forward([3, 1, 2], want_hidden=True)
    x = m.layer_output(0, 3)[2].astype(np.float64)
    near(hidden, x / np.sqrt(np.mean(x * x) + 1e-5) * (1.0 + w["final.norm"].astype(np.float64)))
    near(logits, w["head"].astype(np.float64) @ hidden.astype(np.float64))


@pytest.mark.parametrize("width,ff", [(64, 16640), (4160, 48), (16400, 48), (16402, 40)])
def test_decode_step(dev, width, ff):
    """Inputs of a step's products that no thread holds whole: a long feed-forward, a wide stream."""
    cfg = G.config_apart([G.with_mlp(G.pair(), G.dense(ff)), G.with_mlp(G.retention(), G.dense(ff))], width=width, vocab=50)
    w = G.weights(cfg)
    toks = np.random.default_rng(ff).integers(0, 50, 12)
    close(run_portions(G.build(dev, cfg, w), toks, [1]), R.forward(cfg, w, toks)[0], TOL["float32"])


@pytest.mark.parametrize("k", [64, 2112, 11008])
@pytest.mark.parametrize("n", [9, 5000])
def test_infinite_weights(dev, n, k):
    """An infinity among the last stored weights of a row that does not fill whole pieces of 512 gives an infinity: lanes past the row multiply nothing."""
    rng = np.random.default_rng(k)
    w = synth.to_bf16_bits(rng.standard_normal(n * k, dtype=np.float32)).reshape(n, k)
    w[2, k - 1], w[3, k - 8], w[4, 0] = 0x7F80, 0xFF80, 0x7F80
    x = np.abs(rng.standard_normal((1, k), dtype=np.float32))
    got = Tensor.from_slice(dev, x).q_mat_mul(QMatrix.from_raw_bytes(dev, (n, k), w, synth.W_BF16)).as_slice()[0]
    assert got[2] == np.inf and got[3] == -np.inf and got[4] == np.inf
    rest = [i for i in range(n) if i not in (2, 3, 4)]
    near(got[rest].astype(np.float64), synth.from_bf16_bits(w[rest]).astype(np.float64) @ x[0].astype(np.float64))


@pytest.mark.parametrize("n,k", [(37, 500), (1024, 4100), (1025, 4100), (1000, 20000), (5000, 1500), (2048, 2048), (6144, 3072), (8192, 2048), (8200, 1024), (3000, 1002)])
@pytest.mark.parametrize("offset", [0, 4])
def test_the_same_sums_dealt_out_or_not(dev, n, k, offset):
    """Either side of the lines between the two ways rows are handed to wavefronts, one of which is whether the device's matrices are more than its last
    cache; the input may begin at any value."""
    rng = np.random.default_rng(n + k)
    w = synth.to_bf16_bits(rng.standard_normal(n * k, dtype=np.float32))
    x = rng.standard_normal((1, k), dtype=np.float32)
    own = Device.gpu(0)
    try:
        q = QMatrix.from_raw_bytes(own, (n, k), w, synth.W_BF16)
        base = Tensor.from_slice(own, np.concatenate([np.zeros(offset // 4, np.float32), x[0]]))
        xt = Tensor(own, (1, k), ptr=base.ptr + offset)
        alone = xt.q_mat_mul(q).as_slice()
        near(alone[0].astype(np.float64), synth.from_bf16_bits(w).reshape(n, k).astype(np.float64) @ x[0].astype(np.float64))
        others = QMatrix.from_raw_bytes(own, (65536, 2056), np.zeros(65536 * 2056, np.uint16), synth.W_BF16)
        assert np.array_equal(xt.q_mat_mul(q).as_slice(), alone)
        del others
    finally:
        own.close()
