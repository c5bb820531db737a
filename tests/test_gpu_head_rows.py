"""GPU parity: the output matrix for several rows in one pass (csrc/fh_dense.hip: k_head_x, k_head_rows) against float64.

Bound: a row's three bf16 terms hold its 24 bits and multiply exactly, so what is left is the rounding of the f32 sums: k errors of
2^-24 of either sign, 1e-6 of the root mean square for k up to 2060, and ten times that for the largest single difference."""
import numpy as np
import pytest

import hybridgen as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,vocab,count", [(20, 30, 2), (64, 64, 16), (72, 65, 17), (256, 130, 33), (1000, 333, 5), (1001, 70, 3), (2060, 40, 2)])
def test_rows(dev, width, vocab, count):
    """Fewer blocks of 64 than wavefronts, k and n that fill no tile, one row more than a pass takes, places in any order and
    twice; the normed row that is given back is the last one's."""
    cfg = G.config([G.with_mlp(G.delta(1, 1, 16, 16, 4), None)], width, vocab)
    w = G.weights(cfg)
    m = G.build(dev, cfg, w)
    rng = np.random.default_rng(width)
    toks = rng.integers(0, vocab, 40)
    places = [int(p) for p in rng.integers(0, 40, count)]
    places[1] = places[0]
    got, last = m.forward(toks, want_hidden=True, want=places)
    head = G.round_bf16(w["head"]).astype(np.float64)
    for i, place in enumerate(places):
        m.reset()
        alone, hidden = m.forward(toks, want_hidden=True, want=[place])
        want = head @ hidden.astype(np.float64)
        rms = np.sqrt(np.mean(want * want))
        for y in (got[i], alone[0]):
            assert np.sqrt(np.mean((y - want) ** 2)) <= 1e-6 * rms
            assert np.abs(y - want).max() <= 1e-5 * rms
    assert np.array_equal(last.view(np.uint32), hidden.view(np.uint32))  # of one place and of several: the same bits


@pytest.mark.parametrize("width,vocab,matvecs", [(1000, 40, 2), (1024, 40, 3), (2048, 40, 3), (4100, 40, 4), (4100, 2050, 4), (100, 3500, 2), (2100, 3510, 3), (64, 6000, 2), (64, 12010, 1)])
def test_few_rows(dev, width, vocab, matvecs):
    """Up to so many places of a small matrix take a matvec each, the same bits as alone; one more and they share a pass."""
    cfg = G.config([G.with_mlp(G.delta(1, 1, 16, 16, 4), None)], width, vocab)
    m = G.build(dev, cfg, G.weights(cfg))
    toks = np.random.default_rng(width).integers(0, vocab, 8)
    alone = []
    for place in range(matvecs + 1):
        m.reset()
        alone.append(m.forward(toks, want=[place])[0])
    for count in (matvecs, matvecs + 1):
        m.reset()
        got = m.forward(toks, want=list(range(count)))
        want = np.array(alone[:count])
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)) == (count == matvecs)
        assert np.sqrt(np.mean((got - want) ** 2)) <= 2e-6 * np.sqrt(np.mean(want ** 2))


@pytest.mark.parametrize("width", [16388, 16400, 16401])
def test_wide_rows_norm_alike(dev, width):
    """Rows longer than a workgroup holds in registers, in fours and value by value: of one place and of several the same bits."""
    cfg = G.config([G.with_mlp(G.delta(1, 1, 16, 16, 4), None)], width, 30)
    m = G.build(dev, cfg, G.weights(cfg))
    toks = np.random.default_rng(width).integers(0, 30, 9)
    _, last = m.forward(toks, want_hidden=True, want=list(range(9)))
    m.reset()
    _, hidden = m.forward(toks, want_hidden=True, want=[8])
    assert np.array_equal(last.view(np.uint32), hidden.view(np.uint32))
