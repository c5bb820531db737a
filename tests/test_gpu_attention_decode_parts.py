"""Matrix-core decode attention where the number of parts changes: one workgroup a compute unit, two, fewer parts than that for few keys."""
import numpy as np
import pytest

from kalosm_amd.fusor import Device, Tensor

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hq,hkv,L", [
    (64, 64, 1536),    # four parts of twelve chunks: three a wavefront
    (64, 64, 1537),    # one key more: eight parts
    (64, 64, 255),     # fewer chunks than wavefronts
    (300, 300, 130),   # more heads than compute units: one part
    (16, 2, 4100),     # as many parts as there are pairs of chunks
])
def test_parts_of_the_keys_match_oracle(dev, oracle, hq, hkv, L):
    rng = np.random.default_rng(hq + L)
    q = rng.standard_normal((1, hq, 1, 128)).astype(np.float16)
    k = rng.standard_normal((1, hkv, L, 128)).astype(np.float16)
    v = rng.standard_normal((1, hkv, L, 128)).astype(np.float16)
    scale = 1 / np.sqrt(128)
    ref = oracle.flash_attention(*(a.astype(np.float32) for a in (q, k, v)), scale)
    dev.set_option("attn_kernel", 5)
    try:
        got = Tensor.from_slice(dev, q, "f16").flash_attention(*(Tensor.from_slice(dev, a, "f16") for a in (k, v)), scale).as_slice().astype(np.float32)
    finally:
        dev.set_option("attn_kernel", 0)
    # weights and outputs are rounded to f16: 2^-11 of each weight, in all at most 2^-11 of the largest |v|, and 2^-11 of an output
    assert (np.abs(got - ref) <= 2.0 ** -11 * (np.abs(v.astype(np.float32)).max() + np.abs(ref)) + 1e-6).all()


def test_long_caches_captured_after_a_short_one():
    """The room for parts that a call of 100 keys leaves behind is enough for a captured one of 4096, of twice as many parts as before, and of 16384."""
    dev = Device.gpu(0)
    try:
        rng = np.random.default_rng(5)
        q = Tensor.from_slice(dev, rng.standard_normal((1, 32, 1, 128)).astype(np.float16), "f16")
        for L in (100, 4096, 16384):
            k, v = (Tensor.from_slice(dev, rng.standard_normal((1, 8, L, 128)).astype(np.float16), "f16") for _ in range(2))
            out = Tensor(dev, (1, 32, 1, 128), "f16")
            if L > 100:
                dev.graph_begin()
            q.flash_attention(k, v, 0.1, out=out)
            if L > 100:
                graph = dev.graph_end()
                got = []
                for _ in range(3):
                    graph.launch()
                    got.append(out.as_slice().view(np.uint16).copy())
                q.flash_attention(k, v, 0.1, out=out)
                assert all(np.array_equal(g, out.as_slice().view(np.uint16)) for g in got)
                del graph
    finally:
        dev.close()


def test_captured_beside_calls_of_other_heads(oracle):
    """The room belongs to the device: calls of eight heads leave it so that one of 32 heads and few keys fits and one of 4096 keys has fewer parts than it would take."""
    dev = Device.gpu(0)
    try:
        rng = np.random.default_rng(6)

        def inputs(hq, L):
            return [rng.standard_normal((1, h, n, 128)).astype(np.float16) for h, n in ((hq, 1), (8, L), (8, L))]

        def put(a):
            return [Tensor.from_slice(dev, t, "f16") for t in a]

        for hq, L in ((8, 4096), (32, 100), (32, 3000)):
            q, k, v = put(inputs(hq, L))
            q.flash_attention(k, v, 0.1)
        for L in (4096, 16384):
            a = inputs(32, L)
            q, k, v = put(a)
            out = Tensor(dev, (1, 32, 1, 128), "f16")
            dev.graph_begin()
            q.flash_attention(k, v, 0.1, out=out)
            graph = dev.graph_end()
            got = []
            for _ in range(3):
                graph.launch()
                got.append(out.as_slice())
            a = [t.astype(np.float32) for t in a]
            want = oracle.flash_attention(*a, 0.1)
            # (weights and outputs are rounded to f16, as above)
            assert (np.abs(got[0].astype(np.float32) - want) <= 2.0 ** -11 * (np.abs(a[2]).max() + np.abs(want)) + 1e-6).all()
            assert all(np.array_equal(g.view(np.uint16), got[0].view(np.uint16)) for g in got)
            del graph
    finally:
        dev.close()


@pytest.mark.parametrize("dtype,L", [("f16", 100), ("f32", 100), ("f16", 4096)])
def test_scratch_limit_that_the_call_keeps(oracle, dtype, L):
    """A call whose own parts fit the limit does not fail because those of longer caches would not."""
    dev = Device.gpu(0)
    try:
        dev.set_option("scratch_limit", 32 * 32 * 132 * 4)  # the 32 parts of 4096 keys; a cache of any length may take 64
        rng = np.random.default_rng(7)
        a = [rng.standard_normal((1, h, n, 128)).astype(np.float16) for h, n in ((32, 1), (8, L), (8, L))]
        got = Tensor.from_slice(dev, a[0], dtype).flash_attention(*(Tensor.from_slice(dev, t, dtype) for t in a[1:]), 0.1).as_slice().astype(np.float32)
        a = [t.astype(np.float32) for t in a]
        want = oracle.flash_attention(*a, 0.1)
        assert (np.abs(got - want) <= 2.0 ** -11 * (np.abs(a[2]).max() + np.abs(want)) + 1e-6).all()
    finally:
        dev.close()
