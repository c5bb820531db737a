"""Matrix-core decode attention where the number of parts changes: one workgroup a compute unit, two, fewer parts than that for few keys."""
import numpy as np
import pytest

from kalosm_amd.fusor import Tensor

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
