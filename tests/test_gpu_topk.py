"""GPU parity: the two-launch top-k (csrc/fh_elementwise.hip: k_topk_keys, k_topk_pick) on the layouts where its threshold, its
gather and its chunks can go wrong, against the oracle.  Bit-equal pairs."""
import numpy as np
import pytest

from kalosm_amd.fusor import Tensor

pytestmark = pytest.mark.gpu


def _logits(layout, n, rng):
    x = rng.standard_normal(n).astype(np.float32)
    if layout == "rising":                      # the k largest maxima are the last lists, every key of them above the threshold
        return np.sort(x)
    if layout == "one_list":                    # the candidates in one list of 64
        x[n // 2 // 64 * 64:][:64] += 100
    elif layout == "spread":                    # one large value per list: more lists than candidates above any other value
        x[::64] += 100
    elif layout == "equal":                     # the order is that of the ids
        x[:] = -0.25
    elif layout == "few":                       # fewer finite values than candidates, in different lists
        x[:] = np.nan
        x[rng.choice(n, 7, replace=False)] = [1, 2, 2, -3, 0.0, -0.0, 1e-42]
    elif layout == "none":
        x[:] = -np.inf
    elif layout == "close":                     # differences in the last bits only
        x = (np.float32(3.0).view(np.uint32) + rng.integers(0, 40, n).astype(np.uint32)).view(np.float32)
    return x


@pytest.mark.parametrize("n", [1025, 4097, 8192, 16385, 20000, 32768, 131073, 1 << 20, (1 << 20) + 1])
@pytest.mark.parametrize("layout", ["rising", "one_list", "spread", "equal", "few", "none", "close"])
def test_layouts(dev, oracle, n, layout):
    """Up to 256 candidates of 32 lists or more: fewer lists than candidates, as many, a few more, far more."""
    x = _logits(layout, n, np.random.default_rng(n))
    t = Tensor.from_slice(dev, x)
    for k in (1, 2, 63, 200, 256):
        got, want = t.top_k_pairs(k), oracle.top_k(x, k)
        assert [g[0] for g in got] == [w[0] for w in want], (k, len(got), len(want))
        assert np.array_equal(np.float32([g[1] for g in got]).view(np.uint32), np.float32([w[1] for w in want]).view(np.uint32))


@pytest.mark.parametrize("kind", ["standard", "mirostat2"])
def test_continuation(dev, oracle, kind):
    """64 draws in a row on given logits, the state and a window of 20 previous ids (which moves on three times) carried over: the
    oracle's token at each step whose deciding comparison is not closer than exp and log2 of the two sides differ."""
    from kalosm_amd.fusor import GpuMirostat2Sampler, GpuMirostat2SamplerParams, GpuStandardSamplerParams

    rng, n = np.random.default_rng(64), 32768
    sampler, mu, history, near = GpuMirostat2Sampler(dev, 10.0), 10.0, rng.integers(0, n, 20).tolist(), 0
    for _ in range(64):
        x = (2.0 * rng.standard_normal(n)).astype(np.float32)
        x[history[-30:]] += 8.0  # (so that the ids of the window, and some that left it, are candidates)
        t, u, prev = Tensor.from_slice(dev, x), float(rng.random(dtype=np.float32)), np.array(history[-20:])
        if kind == "standard":
            got = t.sample_standard_token(prev, GpuStandardSamplerParams(64, 0.8, 1.3, 0.95, 0.01, u))
            want = oracle.sample_token(x, 0, 64, 0.8, 1.3, 0.95, 0.01, random=u, previous=prev)
        else:
            got = t.sample_mirostat2_token(sampler, prev, GpuMirostat2SamplerParams(64, 0.8, 1.3, 5.0, 0.1, u))
            want = oracle.sample_token(x, 1, 64, 0.8, 1.3, tau=5.0, eta=0.1, random=u, previous=prev, mu=mu)
        if want["margin"] > 1e-4:
            assert got == want["token"]
        near += want["margin"] <= 1e-4
        if kind == "mirostat2":
            if got == want["token"]:
                assert sampler.mu == pytest.approx(want["mu"], rel=1e-5, abs=1e-5)
            mu = sampler.mu
        history.append(got)
    assert near <= 6


def test_graphs_outlive_a_larger_vocabulary():
    """The keys of 151936 logits lie in memory that never moves, and so do the rows of an output matrix of width 12288: a graph
    that was captured before them is still launched."""
    import hybridgen as G
    from kalosm_amd import synth
    from kalosm_amd.fusor import Device, QMatrix

    dev = Device.gpu(0)
    try:
        rng = np.random.default_rng(3)
        q = QMatrix.from_raw_bytes(dev, (64, 512), synth.random_weight(synth.Q8_0, 64, 512, 1), synth.Q8_0)
        x, y = Tensor.from_slice(dev, synth.random_activation(16, 512, 2)), Tensor.zeros(dev, (16, 64))
        cfg = G.config([G.with_mlp(G.delta(1, 1, 16, 16, 4), None)], 12288, 40)
        model = G.build(dev, cfg, G.weights(cfg))
        alone = model.forward([3, 1, 2])
        Tensor.from_slice(dev, rng.standard_normal((1 << 20) + 1).astype(np.float32)).top_k_pairs(1)  # the passes' scratch: 1 MB
        x.q_mat_mul(q, out=y)
        want = y.as_slice()
        dev.graph_begin()
        x.q_mat_mul(q, out=y)
        graph = dev.graph_end()
        logits = rng.standard_normal(151936).astype(np.float32)
        assert [p[0] for p in Tensor.from_slice(dev, logits).top_k_pairs(64)] == np.argsort(-logits, kind="stable")[:64].tolist()
        model.reset()
        several = model.forward([3, 1, 2], want=[0, 1, 2] * 3)
        assert np.sqrt(np.mean((several[-1] - alone) ** 2)) <= 2e-6 * np.sqrt(np.mean(alone ** 2))
        for _ in range(2):
            graph.launch()
            assert np.array_equal(y.as_slice(), want)
        del graph
    finally:
        dev.close()
