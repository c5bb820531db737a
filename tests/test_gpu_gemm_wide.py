"""GPU parity: the 256-row product of bf16 weights and bf16 activations (csrc/fh_dense.hip) against float64.

Bound: bf16 operands multiply exactly and are added in f32: k rounding errors of 2^-24 of either sign, so 1e-6 of the
result's root mean square for k up to 4096, and ten times that for the largest single difference."""
import numpy as np
import pytest

from kalosm_amd import synth
from kalosm_amd.fusor import QMatrix, Tensor

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("option", [4, 14])
@pytest.mark.parametrize("m,n,k", [(1, 1, 64), (128, 256, 128), (129, 257, 192), (256, 256, 64), (257, 255, 128), (300, 513, 192), (511, 272, 1024), (40, 1030, 4096),
                                   (700, 600, 1000)])
def test_wide_product(dev, m, n, k, option):
    """Tiles exactly full and one row or column past that, fewer slabs of k than buffers, k that is not a multiple of 64; options 4 and
    14 take the forms with 256 and 128 activation rows whatever the size."""
    rng = np.random.default_rng(m + n + k)
    w = synth.to_bf16_bits(rng.standard_normal((n, k)).astype(np.float32))
    x = synth.to_bf16_bits(rng.standard_normal((m, k)).astype(np.float32))
    q = QMatrix.from_raw_bytes(dev, (n, k), w, synth.W_BF16)
    out = Tensor.filled_bytes(dev, (m, n), 0xFF)
    dev.set_option("matmul_kernel", option)
    try:
        got = Tensor.from_slice(dev, x, dtype="bf16").q_mat_mul(q, out=out).as_slice().astype(np.float64)
    finally:
        dev.set_option("matmul_kernel", 0)
    want = synth.from_bf16_bits(x).astype(np.float64) @ synth.from_bf16_bits(w).astype(np.float64).T
    rms = np.sqrt(np.mean(want * want))
    assert np.sqrt(np.mean((got - want) ** 2)) <= 1e-6 * rms
    assert np.abs(got - want).max() <= 1e-5 * rms


@pytest.mark.parametrize("option", [0, 4, 14])
def test_layers_agree(dev, option):
    """Every output form (f32, operand rows, transposed, gated, squared relu, grouped by expert) inside the two layer-list
    decoders: the wide kernel, by its rule and in both forms whatever the size, and the others (option 3) differ by the order of
    f32 sums and the bf16 roundings that flips."""
    from kalosm_amd import bench_hybrid
    from kalosm_amd.hybrid import HybridModel

    small = dict(width=512, heads=4, experts=4, top=2, ff=256, window=128, groups=2)
    for cfg in (bench_hybrid.config(vocab=512, **small), bench_hybrid.zovovik_config(512, 4, 1024, 128, vocab=512)):
        m = HybridModel.random_init(dev, cfg, ctx=512)
        tokens = np.random.default_rng(3).integers(0, 512, 300)
        dev.set_option("matmul_kernel", 3)
        try:
            want = m.forward(tokens, want=range(290, 300)).astype(np.float64)
            m.reset()
            dev.set_option("matmul_kernel", option)
            got = m.forward(tokens, want=range(290, 300)).astype(np.float64)
        finally:
            dev.set_option("matmul_kernel", 0)
        assert np.sqrt(np.mean((got - want) ** 2)) <= 2.7e-2 * np.sqrt(np.mean(want * want))


@pytest.mark.parametrize("experts", [3, 5])
@pytest.mark.parametrize("tokens", [31, 65, 160, 300, 511])
def test_grouped_tiles(dev, tokens, experts):
    """Groups of a few to 320 rows a tile, past that shared out evenly (option 4), against tiles of 128 rows (option 14): an output is the
    same chain of products over k in both, so that they agree bit by bit."""
    from kalosm_amd import bench_hybrid
    from kalosm_amd.hybrid import HybridModel

    small = dict(width=512, heads=4, experts=experts, top=2, ff=192, window=128, groups=2)
    for cfg in (bench_hybrid.config(vocab=512, **small), bench_hybrid.zovovik_config(512, 4, 1024, 128, vocab=512)):
        m = HybridModel.random_init(dev, cfg, ctx=512)
        ids, got = np.random.default_rng(tokens).integers(0, 512, tokens), {}
        try:
            for option in (14, 4):
                m.reset()
                dev.set_option("matmul_kernel", option)
                got[option] = m.forward(ids, want=range(tokens - 20, tokens))
        finally:
            dev.set_option("matmul_kernel", 0)
        np.testing.assert_array_equal(got[4], got[14])


@pytest.mark.parametrize("tokens", [1025, 1100, 2047])
def test_grouped_tiles_more_than_eight(dev, tokens):
    """Two experts of two take every token: as tiles of 128 rows (option 14) they are nine or sixteen each, eight neighbours and what is left, of up to 320 (option 4)
    no more than seven."""
    from kalosm_amd import bench_hybrid
    from kalosm_amd.hybrid import HybridModel

    m = HybridModel.random_init(dev, bench_hybrid.config(vocab=512, width=512, heads=4, experts=2, top=2, ff=192, window=128, groups=2), ctx=2048)
    ids, got = np.random.default_rng(tokens).integers(0, 512, tokens), {}
    try:
        for option in (14, 4):
            m.reset()
            dev.set_option("matmul_kernel", option)
            got[option] = m.forward(ids, want=range(tokens - 200, tokens))
    finally:
        dev.set_option("matmul_kernel", 0)
    np.testing.assert_array_equal(got[4], got[14])
