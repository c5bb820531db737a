"""GPU parity: the inputs of the recurrences for four tokens a workgroup (csrc/fh_recurrent.hip: k_rec_prep<4>), which takes portions
of 1024 tokens and more on 256 compute units, against the numpy restatement: every number of taps up to one that keeps the form for
one token, portions that end inside a group of four, rows from the ring."""
import numpy as np
import pytest

import hybridgen as G
from oracle import hybrid_ref as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("taps", [1, 2, 3, 4, 5])
def test_portions(dev, taps):
    cfg = G.config([G.with_mlp(G.delta(2, 1, 16, 16, taps), None), G.with_mlp(G.mamba2(4, 8, 16, 2, 2, taps), None)], 64, 50)
    w = G.weights(cfg)
    toks = np.random.default_rng(taps).integers(0, 50, 2080)
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
