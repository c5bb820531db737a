"""GPU parity: the inputs of the recurrences for one token a workgroup and for four (csrc/fh_recurrent.hip: k_rec_prep<T>; four for portions of
1024 tokens and more on 256 compute units, with four taps and many channels), against the numpy restatement: every number of
taps, portions that end inside a group of four, rows from the ring."""
import numpy as np
import pytest

import hybridgen as G
from oracle import hybrid_ref as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("taps", [1, 2, 3, 4, 5])
def test_portions(dev, taps):
    check(dev, G.config([G.with_mlp(G.delta(2, 1, 16, 16, taps), None), G.with_mlp(G.mamba2(4, 8, 16, 2, 2, taps), None)], 64, 50), taps)


@pytest.mark.parametrize("layer", [G.delta(8, 4, 128, 128, 4), G.delta(16, 4, 128, 60, 4), G.mamba2(16, 64, 128, 1, 1, 4), G.mamba2(19, 64, 30, 1, 1, 4)],
                         ids=["2048", "1984", "1280", "1276"])
def test_channels(dev, layer):
    """As many channels as the form for four tokens takes, and fewer."""
    check(dev, G.config([G.with_mlp(layer, None)], 64, 50), 7)


def check(dev, cfg, seed):
    w = G.weights(cfg)
    toks = np.random.default_rng(seed).integers(0, 50, 2080)
    want, _ = R.forward(cfg, w, toks)
    m = G.build(dev, cfg, w)
    for sizes in ([2080 - 1029, 1029], [2, 1030, 1048]):
        m.reset()
        at = 0
        for n in sizes:
            places = sorted({0, 1, 2, 3, 4, n // 2, n - 2, n - 1} & set(range(n)))
            got = m.forward(toks[at:at + n], want=places)
            assert G.rel_err(got, want[at + np.array(places)]).max() <= 3e-5, (sizes, at)
            at += n


@pytest.mark.parametrize("layer", [G.mamba2(4, 64, 16, 1, 1, 2), G.mamba2(3, 85, 16, 1, 1, 2), G.mamba2(5, 104, 16, 1, 2, 2), G.mamba2(2, 129, 16, 1, 1, 2),
                                   G.delta(2, 1, 16, 256, 2), G.delta(2, 1, 16, 252, 2)], ids=["256", "255", "2x260", "258", "2x256", "2x252"])
def test_normed_groups(dev, layer):
    """The gated norm of the outputs, four channels a thread for groups of 256 and more in fours: gate ahead of the norm and behind it, lanes
    that stand idle at a group's end."""
    cfg = G.config([G.with_mlp(layer, None)], 64, 50)
    w = G.weights(cfg)
    toks = np.random.default_rng(8).integers(0, 50, 70)
    want, _ = R.forward(cfg, w, toks)
    for dtype, tol in (("float32", 3e-5), ("bfloat16", 4e-2)):
        got = G.build(dev, cfg, w, dtype).forward(toks, want=range(70))
        assert G.rel_err(got, want).max() <= tol
