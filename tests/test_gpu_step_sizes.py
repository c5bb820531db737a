"""GPU parity: the decode steps of layer-list decoders (csrc/fh_step.hip) against the numpy restatement at the sizes where the output launch
holds another number of values in registers (1536, 2048, 4096 and 8192 of the mixer, 2048, 4096 and 8192 of the experts, 2048 of the always-on one, and past
those), asks for weights of the output projection ahead of the experts' numbers (four pieces of 512 and more) or gives a wavefront several rows (widths
beyond eight a compute unit), where the middle launch's wavefronts have several activations or none, and where the router's logits take another number of
registers (64 and 256 experts)."""
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
    (1030, state_space(2), G.moe(3, 2, 60, 0)),    # fewer activations than wavefronts
    (1030, latent(2), G.moe(3, 2, 60, 0)),
    (1030, state_space(2), G.moe(8, 8, 1024, 0)),  # several a wavefront
    (1030, latent(2), G.moe(8, 8, 1024, 0)),
    (64, state_space(25), G.moe(4, 4, 1000, 0)),   # 1600 and 4096: the first requests reach into the experts' rows
    (64, latent(32), G.moe(4, 4, 1024, 30)),       # 2048 and 4096: exactly to their end
    (64, latent(8), G.moe(2, 1, 40, 2100)),        # an always-on one of 2112
    (2060, state_space(24), G.moe(3, 2, 60, 40)),  # rows of 1536, two experts and the always-on one: some wavefronts have two
    (4100, state_space(25), G.moe(3, 2, 60, 40)),  # two and three, the first requests ahead of the experts
    (4100, state_space(33), G.moe(3, 2, 600, 0)),
    (4100, latent(33), None),                      # rows of the output projection alone
    (4100, latent(65), G.moe(3, 3, 50, 2100)),     # read as they are staged
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


@pytest.mark.parametrize("experts,distinct", [(64, 30), (65, 30), (256, 100), (257, 100), (1024, 400)])
def test_ties_of_many_experts(dev, experts, distinct):
    """Experts whose logits are exactly the same, every `distinct`-th, among them ones of other registers and of the last few: the first ones are taken."""
    cfg = G.config([G.with_mlp(latent(2), G.moe(experts, 5, 16, 0))], 512, 50)
    w = G.weights(cfg)
    router = w["l0.mlp.router"]
    router[:] = 0.0
    router[np.arange(experts), np.arange(experts) % distinct] = 1.0  # a logit is one value of the normed row
    toks = np.random.default_rng(experts).integers(0, 50, 8)
    close(run_portions(G.build(dev, cfg, w), toks, [1]), R.forward(cfg, w, toks)[0], TOL["float32"])
