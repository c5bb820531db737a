"""Decode attention where the number of parts changes: on the matrix cores one workgroup a compute unit, two, fewer parts than that for few keys; without them
8 or 16, and one or two heads a workgroup, of up to 64 heads."""
import numpy as np
import pytest

from kalosm_amd.fusor import Device, Tensor

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hq,hkv,L", [
    (64, 64, 1536),    # four parts of twelve chunks: three a wavefront
    (64, 64, 1537),    # one key more: eight parts
    (64, 64, 255),     # fewer chunks than wavefronts
    (300, 300, 130),   # more than 64 heads: the kernel of any number of them
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


@pytest.mark.parametrize("dtype,hq,hkv,L,parts", [
    ("f16", 64, 8, 300, 8),     # two heads a workgroup of short caches, one chunk of a part and its end
    ("f16", 64, 8, 2048, 8),
    ("f16", 34, 17, 2047, 8),
    ("f32", 64, 8, 1024, 8),
    ("f32", 64, 8, 1025, 8),    # one head again
    ("f32", 40, 40, 2049, 16),  # more workgroups than compute units, but fewer than half as many again
    ("f32", 48, 16, 2049, 8),   # not fewer
    ("f32", 40, 8, 4000, 16),
    ("f32", 36, 12, 4095, 16),  # twelve KV heads
    ("f32", 36, 12, 4096, 8),
    ("f32", 64, 8, 4000, 8),    # two heads a workgroup
    ("f32", 36, 6, 3072, 8),    # of few KV heads, while the keys are few
    ("f32", 36, 6, 3073, 16),
    ("f16", 33, 11, 4095, 8),
    ("f16", 33, 33, 4095, 16),
    ("f32", 32, 8, 2049, 16),
])
def test_heads_and_parts_without_matrix_cores(dev, oracle, dtype, hq, hkv, L, parts):
    rng = np.random.default_rng(L)
    a = [rng.standard_normal((1, h, n, 128)).astype(np.float16 if dtype == "f16" else np.float32) for h, n in ((hq, 1), (hkv, L), (hkv, L))]
    q, k, v = (Tensor.from_slice(dev, t, dtype) for t in a)
    auto = q.flash_attention(k, v, 0.1).as_slice()
    same = []
    for forced in (8, 16):  # another number of parts rounds the sums elsewhere
        dev.set_option("attn_splits", forced)
        try:
            same.append(np.array_equal(q.flash_attention(k, v, 0.1).as_slice(), auto))
        finally:
            dev.set_option("attn_splits", 0)
    assert same[parts == 16] and (dtype == "f16" or not same[parts != 16])
    a = [t.astype(np.float32) for t in a]
    want = oracle.flash_attention(*a, 0.1)
    # f32 sums of the weighted values, a lane's chain of a few hundred; of f16 the outputs are rounded
    bound = 2.0 ** -17 * np.abs(a[2]).max() + (2.0 ** -11 * np.abs(want) if dtype == "f16" else 0)
    assert (np.abs(auto.astype(np.float32) - want) <= bound).all()


@pytest.mark.parametrize("hq,hkv,L,parts", [
    (16, 16, 8192, 32),    # heads 2 MB apart: two chunks a wavefront
    (16, 16, 8100, 32),    # nearly (the number in sixteens)
    (16, 16, 7600, 32),    # not: two workgroups a compute unit
    (48, 48, 4096, 16),    # 1 MB
    (48, 48, 4400, 10),    # a little more
    (8, 8, 32768, 128),    # eight heads, from so many keys on
    (8, 8, 16384, 64),
    (40, 40, 8192, 32),
    (24, 12, 4096, 16),    # KV heads that do not share the compute units out
    (24, 12, 8200, 16),
    (10, 10, 8192, 16),
    (10, 10, 8224, 25),
    (8, 8, 32832, 64),
    (12, 3, 8224, 64),
])
def test_parts_on_the_matrix_cores(dev, oracle, hq, hkv, L, parts):
    rng = np.random.default_rng(L)
    a = [rng.standard_normal((1, h, n, 128), dtype=np.float32).astype(np.float16) for h, n in ((hq, 1), (hkv, L), (hkv, L))]
    q, k, v = (Tensor.from_slice(dev, t, "f16") for t in a)
    auto = q.flash_attention(k, v, 0.1).as_slice()
    same = []
    for forced in (parts, parts - 3):  # another number of parts rounds the sums elsewhere
        dev.set_option("attn_splits", forced)
        try:
            same.append(np.array_equal(q.flash_attention(k, v, 0.1).as_slice(), auto))
        finally:
            dev.set_option("attn_splits", 0)
    assert same == [True, False]
    a = [t.astype(np.float32) for t in a]
    want = oracle.flash_attention(*a, 0.1)
    # (weights and outputs are rounded to f16, as above)
    assert (np.abs(auto.astype(np.float32) - want) <= 2.0 ** -11 * (np.abs(a[2]).max() + np.abs(want)) + 1e-6).all()
