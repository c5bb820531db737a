"""GPU parity: prefill attention over windows longer than a key tile (csrc/fh_window_attn.hip) against the numpy restatement: tiles
that all queries see whole, tiles cut by the diagonal, the window's start, the kept tokens and the end of the rows."""
import numpy as np
import pytest

import hybridgen as G
from oracle import hybrid_ref as R

pytestmark = pytest.mark.gpu

TOL = {"float32": 3e-5, "bfloat16": 4e-2}  # root mean square of a position over the logits' standard deviation


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("window", [64, 65, 200, 333, 1000])
@pytest.mark.parametrize("layer", ["latent", "grouped"])
def test_windows(dev, dtype, window, layer):
    if layer == "latent":  # 128 + 64 of a key in two parts, values of 128; 24 + 8 of the padded 64, values of 40
        cfg = G.config([G.with_mlp(G.latent(heads=2, dim=192, rot_dim=64, vdim=128, kv_rank=64, window=window), None),
                        G.with_mlp(G.latent(heads=3, dim=32, rot_dim=8, vdim=40, kv_rank=72, window=window), None)], 128, 64)
    else:
        cfg = G.config_apart([G.with_mlp(G.pair(G.attention(heads=4, kv_heads=2, dim=64, vdim=64, window=window, keep=5, dims=32)), None)], 128, 64)
    w = G.weights(cfg)
    toks = np.random.default_rng(window).integers(0, 64, 470)
    want, _ = R.forward(cfg, w, toks)
    m = G.build(dev, cfg, w, dtype)
    for sizes in ([470], [129, 70, 271]):
        m.reset()
        at, got = 0, []
        for n in sizes:
            got.append(m.forward(toks[at:at + n], want=range(n)))
            at += n
        assert G.rel_err(np.concatenate(got), want).max() <= TOL[dtype], sizes
