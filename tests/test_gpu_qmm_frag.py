"""GPU parity: the prompt matmul on fragment-ordered operands (csrc/fh_qmm_frag.hip) against a float64 product of the oracle's
dequantised weights.

Bound: the operands are exact up to 2^-22 of each activation and each product is added in f32, k / 16 * 3 additions in a
chain at most, whose rounding errors (2^-24 each, of either sign) grow with the root of their number: 2e-6 of the result's
root mean square covers k = 14336 with the cancellation of the offsets (a factor of about two) included.  The largest single
difference is held to ten times that (ten standard deviations)."""
import numpy as np
import pytest

from kalosm_amd import synth
from kalosm_amd.fusor import Device, FusorHipError, QMatrix, Tensor

pytestmark = pytest.mark.gpu
TYPES = [synth.Q4_0, synth.Q5_0, synth.Q8_0, synth.Q4_K, synth.Q5_K, synth.Q6_K]


def product(dev, oracle, ty, m, n, k, act, option, x=None, seed=1):
    raw = synth.random_weight(ty, n, k, seed=seed + n, sigma=2e-3)
    x = synth.random_activation(m, k, seed=seed + m) if x is None else x
    bits = synth.to_bf16_bits(x) if act == "bf16" else None
    if bits is not None:
        x = synth.from_bf16_bits(bits)
    q = QMatrix.from_raw_bytes(dev, (n, k), raw, ty)
    xt = Tensor.from_slice(dev, x) if bits is None else Tensor.from_slice(dev, bits, dtype="bf16")
    out = Tensor.filled_bytes(dev, (m, n), 0xFF)  # poisoned: unwritten elements show as NaN
    dev.set_option("matmul_kernel", option)
    try:
        got = xt.q_mat_mul(q, out=out).as_slice().astype(np.float64)
    finally:
        dev.set_option("matmul_kernel", 0)
    w = oracle.dequantize(ty, raw).reshape(n, k).astype(np.float64)
    return got, x.astype(np.float64) @ w.T


@pytest.mark.parametrize("act", ["f32", "bf16"])
@pytest.mark.parametrize("ty", TYPES, ids=lambda t: synth.TYPE_NAMES[t])
@pytest.mark.parametrize("m,n,k", [
    (1, 1, 256),        # one row, one output
    (64, 256, 512),     # exactly a tile of the small form
    (65, 257, 768),     # one past it; three scales of 256
    (127, 100, 1024),
    (129, 513, 2048),   # one past 128 activation and 512 weight rows; k split over workgroups
    (300, 40, 14336),   # long k
])
def test_product(dev, oracle, ty, act, m, n, k):
    got, want = product(dev, oracle, ty, m, n, k, act, 13)
    rms = np.sqrt(np.mean(want * want))
    assert np.isfinite(got).all()
    assert np.sqrt(np.mean((got - want) ** 2)) <= 2e-6 * rms
    assert np.abs(got - want).max() <= 2e-5 * rms


@pytest.mark.parametrize("ty", [synth.Q4_0, synth.Q8_0, synth.Q5_0], ids=lambda t: synth.TYPE_NAMES[t])
@pytest.mark.parametrize("k", [128, 384, 640])
def test_odd_multiples_of_128(dev, oracle, ty, k):
    """Formats with a scale per 32: the last 128 of k are a half round of the loop."""
    got, want = product(dev, oracle, ty, 70, 130, k, "f32", 13)
    assert np.sqrt(np.mean((got - want) ** 2)) <= 2e-6 * np.sqrt(np.mean(want * want))


@pytest.mark.parametrize("act", ["f32", "bf16"])
@pytest.mark.parametrize("ty,m,n,k", [(synth.Q4_K, 17, 272, 2048), (synth.Q6_K, 64, 300, 512), (synth.Q4_K, 1025, 512, 512),
                                      (synth.Q6_K, 513, 512, 512), (synth.Q8_0, 513, 130, 4096), (synth.Q5_K, 129, 512, 1024)])
def test_default_dispatch(dev, oracle, ty, m, n, k, act):
    """Sizes at the lines of the dispatch rule, whichever kernel they take."""
    got, want = product(dev, oracle, ty, m, n, k, act, 0)
    assert np.sqrt(np.mean((got - want) ** 2)) <= 2e-6 * np.sqrt(np.mean(want * want))


@pytest.mark.parametrize("ty,act,m,n,k,fragments", [
    (synth.Q4_K, "f32", 32, 4096, 512, True), (synth.Q4_K, "f32", 32, 32784, 512, False),        # more tiles than fit at once
    (synth.Q6_K, "bf16", 64, 18432, 512, True), (synth.Q6_K, "bf16", 64, 18448, 512, False),
    (synth.Q8_0, "f32", 17, 32768, 512, True), (synth.Q8_0, "f32", 17, 22544, 2176, False),
    (synth.Q8_0, "f32", 600, 512, 2048, False), (synth.Q8_0, "f32", 600, 2048, 512, True),       # narrow matrices
    (synth.Q8_0, "f32", 600, 130, 2048, True), (synth.Q4_0, "f32", 1100, 1024, 512, True),
    (synth.Q5_0, "f32", 200, 3072, 512, True), (synth.Q5_0, "f32", 200, 8192, 2048, False),      # few rows, tiles that fill the device
    (synth.Q4_K, "f32", 300, 2048, 512, True), (synth.Q4_K, "f32", 512, 8192, 2048, False),
    (synth.Q4_K, "bf16", 800, 1024, 512, False), (synth.Q4_K, "bf16", 800, 2048, 512, True),
    (synth.Q5_K, "bf16", 200, 2048, 512, False), (synth.Q5_K, "bf16", 200, 3072, 512, True),
])
def test_rule(dev, ty, act, m, n, k, fragments):
    """Both sides of the dispatch's lines: the bits of the fragments (option 13) or those of the tiles (11), which are different."""
    q = QMatrix.from_raw_bytes(dev, (n, k), synth.random_weight(ty, n, k, seed=n, sigma=2e-3), ty)
    x = synth.random_activation(m, k, seed=m)
    xt = Tensor.from_slice(dev, x) if act == "f32" else Tensor.from_slice(dev, synth.to_bf16_bits(x), dtype="bf16")
    got = {}
    for option in (0, 11, 13):
        dev.set_option("matmul_kernel", option)
        try:
            got[option] = xt.q_mat_mul(q).as_slice().view(np.uint32)
        finally:
            dev.set_option("matmul_kernel", 0)
    assert not np.array_equal(got[11], got[13])
    assert np.array_equal(got[0], got[13 if fragments else 11])


@pytest.mark.parametrize("ty", [synth.Q4_K, synth.Q6_K, synth.Q8_0], ids=lambda t: synth.TYPE_NAMES[t])
def test_rows_are_independent(dev, oracle, ty):
    """Zeros stay zero, a power of two passes through exactly, and an infinity or a NaN stays in its row."""
    m, n, k = 80, 96, 1024
    x = synth.random_activation(m, k, seed=5)
    base, _ = product(dev, oracle, ty, m, n, k, "f32", 13, x=x.copy(), seed=9)
    x[3] = 0.0
    x[4] *= np.float32(2.0 ** 20)
    x[5, 7] = np.inf
    x[6, 9] = np.nan
    got, _ = product(dev, oracle, ty, m, n, k, "f32", 13, x=x, seed=9)
    assert not got[3].any()
    assert np.array_equal(got[4], base[4] * 2.0 ** 20)
    assert not np.isfinite(got[5]).any() and np.isnan(got[6]).all()
    rest = [r for r in range(m) if r not in (3, 4, 5, 6)]
    assert np.array_equal(got[rest], base[rest])


@pytest.mark.parametrize("m", [17, 64, 65, 257])
@pytest.mark.parametrize("ffn,d_model", [(256, 256), (768, 256), (1280, 256), (256, 2048), (512, 4096)])
def test_swiglu_epilogue(dev, m, ffn, d_model):
    """gate | up of one launch, SwiGLU at the store, against the two halves as matrices of their own: the same sums and the same
    formula, so the logits are the same bits.  (Halves that end within a tile of 512 weight rows; with a long d_model k is in
    several parts, so SwiGLU is a launch of its own and the sums of one matrix and of two are parted differently: each within the
    2e-6 of above, in two layers, is 8e-6 between them.)"""
    from kalosm_amd.llama import Model

    cfg = dict(n_layers=2, d_model=d_model, n_heads=d_model // 128, n_kv_heads=d_model // 256, head_dim=128, ffn=ffn, vocab=320, ctx=512, eps=1e-5, theta=1e4)
    tokens = np.random.default_rng(m).integers(0, 320, m)
    got = []
    for fuse in (True, False):
        model = Model.random_init(dev, cfg, seed=2, sigma=2e-3, fuse_gate_up=fuse)
        dev.set_option("matmul_kernel", 13)
        try:
            got.append(model.forward(tokens))
        finally:
            dev.set_option("matmul_kernel", 0)
    assert np.isfinite(got[0]).all()
    if d_model == 256:
        assert np.array_equal(got[0], got[1])
    assert np.sqrt(np.mean((got[0] - got[1]) ** 2)) <= 1e-5 * np.sqrt(np.mean(got[1] ** 2))


@pytest.mark.parametrize("tokens", [17, 37, 64])
def test_short_prompts_keep_the_tile_sums(dev, tokens):
    """What a sampled answer draws follows from the last bits of the cache that its prompt left, so a decoder's short prompts stay
    on the tile kernels (option 11 takes the fragments nowhere and is the default in all else at these sizes): the same bits."""
    from kalosm_amd.llama import Model

    cfg = dict(n_layers=2, d_model=512, n_heads=4, n_kv_heads=2, head_dim=128, ffn=1024, vocab=320, ctx=128, eps=1e-5, theta=1e4)
    model = Model.random_init(dev, cfg, seed=2, sigma=2e-3)
    prompt = np.random.default_rng(tokens).integers(0, 320, tokens)
    got = []
    for option in (0, 11):
        dev.set_option("matmul_kernel", option)
        try:
            got.append(model.forward(prompt, want_hidden=True)[1])
        finally:
            dev.set_option("matmul_kernel", 0)
        model.reset()
    assert np.isfinite(got[0]).all() and np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32))


def bits(dev, q, x, option):
    dev.set_option("matmul_kernel", option)
    try:
        return x.q_mat_mul(q).as_slice().view(np.uint32)
    finally:
        dev.set_option("matmul_kernel", 0)


@pytest.mark.parametrize("ty", [synth.Q8_0, synth.Q4_K, synth.Q6_K], ids=lambda t: synth.TYPE_NAMES[t])
def test_weights_in_several_launches(oracle, ty):
    """Scratch of 3.5 MB holds the fragments of 768 to 1536 of the 3000 rows."""
    dev = Device.gpu(0)
    dev.set_option("scratch_limit", 3500000)
    try:
        got, want = product(dev, oracle, ty, 70, 3000, 1024, "f32", 13)
        tiles, _ = product(dev, oracle, ty, 70, 3000, 1024, "f32", 11)
    finally:
        dev.close()
    assert np.sqrt(np.mean((got - want) ** 2)) <= 2e-6 * np.sqrt(np.mean(want * want))
    assert not np.array_equal(got, tiles)


def test_without_memory_for_the_fragments():
    """The tile kernels, which need less, take the product."""
    dev = Device.gpu(0)
    try:
        q = QMatrix.from_raw_bytes(dev, (512, 512), synth.random_weight(synth.Q4_K, 512, 512, seed=1, sigma=2e-3), synth.Q4_K)
        x = Tensor.from_slice(dev, synth.random_activation(40, 512, seed=2))
        dev.set_option("scratch_limit", 300000)
        refused = bits(dev, q, x, 0)
        dev.set_option("scratch_limit", 0)
        assert np.array_equal(refused, bits(dev, q, x, 11))
        assert np.array_equal(bits(dev, q, x, 0), bits(dev, q, x, 13)) and not np.array_equal(bits(dev, q, x, 0), refused)
    finally:
        dev.close()


def test_fragments_and_graphs():
    """A captured product takes the fragments if their memory is there, and the tiles if not; growth of that memory ends the graphs
    that use it and no others; an allocation that fails has asked for it first."""
    dev = Device.gpu(0)
    try:
        x = Tensor.from_slice(dev, synth.random_activation(40, 512, seed=2))
        q = {n: QMatrix.from_raw_bytes(dev, (n, 512), synth.random_weight(synth.Q8_0, n, 512, seed=n, sigma=2e-3), synth.Q8_0)
             for n in (64, 2048, 8192)}
        out = Tensor(dev, (40, 2048))

        def capture():
            dev.graph_begin()
            x.q_mat_mul(q[2048], out=out)
            return dev.graph_end()

        def replay(graph):
            graph.launch()
            return out.as_slice().view(np.uint32)

        bits(dev, q[64], x, 13)                       # 1 MB of each buffer
        tiles = bits(dev, q[2048], x, 11)
        on_tiles = capture()                          # 2 MB of fragments
        assert np.array_equal(replay(on_tiles), tiles)
        fragments = bits(dev, q[2048], x, 0)
        assert not np.array_equal(fragments, tiles)
        on_fragments = capture()
        for _ in range(3):
            assert np.array_equal(replay(on_fragments), fragments)
            assert np.array_equal(replay(on_tiles), tiles)
        bits(dev, q[8192], x, 0)
        with pytest.raises(FusorHipError, match="capture it again"):
            on_fragments.launch()
        assert np.array_equal(replay(on_tiles), tiles)
        with pytest.raises(FusorHipError):
            dev.alloc(1 << 42)
        assert np.array_equal(replay(capture()), tiles)
        assert np.array_equal(bits(dev, q[2048], x, 0), fragments)
        del on_tiles, on_fragments
    finally:
        dev.close()


def test_fragments_in_a_captured_step():
    """Option 13 takes a decoder's one-row products there as well: a step that was captured with them is captured again when a
    larger product moves their memory."""
    from kalosm_amd.llama import Model

    dev = Device.gpu(0)
    dev.set_option("matmul_kernel", 13)
    try:
        cfg = dict(n_layers=1, d_model=512, n_heads=4, n_kv_heads=2, head_dim=128, ffn=1024, vocab=320, ctx=64, eps=1e-5, theta=1e4)
        model = Model.random_init(dev, cfg, seed=2, sigma=2e-3, fuse_qkv=False)
        want = model.decode_greedy(5, 8)[0].tolist()
        x = Tensor.from_slice(dev, synth.random_activation(40, 512, seed=2))
        large = QMatrix.from_raw_bytes(dev, (16384, 512), synth.random_weight(synth.Q8_0, 16384, 512, seed=3, sigma=2e-3), synth.Q8_0)
        for _ in range(2):
            x.q_mat_mul(large).as_slice()
            model.reset()
            assert model.decode_greedy(5, 8)[0].tolist() == want
    finally:
        dev.close()


def test_graphs_of_other_calls_outlive_fragments():
    """A product on fragments takes more memory than on the tiles (activations for whole tiles, here 2.2 MB for 0.3), all of it its
    own: a graph that was captured on the tiles is still launched after it, and one that holds fragments until they move."""
    dev = Device.gpu(0)
    try:
        q = QMatrix.from_raw_bytes(dev, (1024, 2048), synth.random_weight(synth.Q4_K, 1024, 2048, seed=1, sigma=2e-3), synth.Q4_K)
        x = Tensor.from_slice(dev, synth.random_activation(32, 2048, seed=2))
        few, out = Tensor.from_slice(dev, synth.random_activation(8, 2048, seed=3)), Tensor(dev, (8, 1024))
        tiles = bits(dev, q, x, 11)
        want = few.q_mat_mul(q, out=out).as_slice()
        dev.graph_begin()
        few.q_mat_mul(q, out=out)
        graph = dev.graph_end()
        fragments = bits(dev, q, x, 0)
        assert not np.array_equal(fragments, tiles)
        graph.launch()
        assert np.array_equal(out.as_slice(), want)
        result = Tensor(dev, (32, 1024))
        dev.graph_begin()
        x.q_mat_mul(q, out=result)
        on_fragments = dev.graph_end()
        on_fragments.launch()
        assert np.array_equal(result.as_slice().view(np.uint32), fragments)
        many = Tensor.from_slice(dev, synth.random_activation(2000, 2048, seed=4))
        many.q_mat_mul(q).as_slice()
        with pytest.raises(FusorHipError, match="capture it again"):
            on_fragments.launch()
        assert np.array_equal(bits(dev, q, x, 0), fragments)
        del graph, on_fragments
    finally:
        dev.close()
