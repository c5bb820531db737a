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
