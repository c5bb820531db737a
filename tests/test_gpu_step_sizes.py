"""GPU parity: the decode steps of layer-list decoders (csrc/fh_step.hip) against the numpy restatement at the sizes where the output launch
holds another number of values in registers (512, 1024, 2048 and 4096 of the mixer, 2048, 4096 and 8192 of the experts, and
past those) and the middle launch another number of pieces of the experts' rows on their way (rows past 1024, more and fewer
workgroups than four a compute unit)."""
import numpy as np
import pytest

import hybridgen as G
from oracle import hybrid_ref as R
from test_gpu_hybrid import TOL, close, run_portions

pytestmark = pytest.mark.gpu


def state_space(heads):
    return G.mamba2(heads, 64, 24, 1, 1, 3)


def latent(heads):
    return G.latent(heads, 16, 8, 64, 40, 5)


@pytest.mark.parametrize("width,mixer,mlp", [
    (64, state_space(8), G.moe(3, 2, 1024, 0)),    # 512 and 2048
    (64, state_space(9), None),                    # 576
    (64, latent(8), G.moe(3, 2, 1025, 40)),        # 512 and 2176
    (64, latent(16), G.moe(3, 2, 1000, 0)),        # 1024 and 2048
    (64, G.delta(17, 1, 20, 64, 4), G.moe(4, 4, 1024, 0)),  # 1088 and 4096
    (64, latent(32), G.moe(4, 4, 1026, 0)),        # 2048 and 4352
    (64, state_space(33), G.moe(8, 8, 1024, 16)),  # 2112 and 8192
    (64, state_space(64), G.moe(8, 8, 1030, 0)),   # 4096 and 8704
    (64, latent(65), G.moe(2, 1, 40, 0)),          # 4160
    (1030, state_space(2), G.moe(3, 2, 60, 0)),    # four pieces on their way
    (1030, latent(2), G.moe(3, 2, 60, 0)),
    (1030, state_space(2), G.moe(8, 8, 1024, 0)),  # two
    (1030, latent(2), G.moe(8, 8, 1024, 0)),
])
def test_sizes(dev, width, mixer, mlp):
    cfg = G.config([G.with_mlp(mixer, mlp)], width, 50)
    w = G.weights(cfg)
    toks = np.random.default_rng(width).integers(0, 50, 8)
    close(run_portions(G.build(dev, cfg, w), toks, [1]), R.forward(cfg, w, toks)[0], TOL["float32"])


def test_more_chosen_experts_than_threads(dev):
    """520 experts a token: a workgroup of the output launch has 512 threads, and its table of the chosen ones is read whole."""
    cfg = G.config([G.with_mlp(latent(2), G.moe(530, 520, 16, 0))], 64, 50)
    w = G.weights(cfg)
    toks = np.random.default_rng(1).integers(0, 50, 4)
    close(run_portions(G.build(dev, cfg, w), toks, [1]), R.forward(cfg, w, toks)[0], TOL["float32"])
