"""GPU: the matmul of a decoder's short prompt (csrc/fh_qmm_tile.hip, k_qmm_short; option 11 takes it at these sizes) against the
tile kernel that it stands in for (option 5): the same sums in the same order, so the same bits."""
import numpy as np
import pytest

from kalosm_amd import synth
from kalosm_amd.fusor import QMatrix, Tensor

pytestmark = pytest.mark.gpu
TYPES = [synth.Q4_0, synth.Q5_0, synth.Q8_0, synth.Q4_K, synth.Q5_K, synth.Q6_K]


@pytest.mark.parametrize("act", ["f32", "bf16"])
@pytest.mark.parametrize("ty", TYPES, ids=lambda t: synth.TYPE_NAMES[t])
@pytest.mark.parametrize("m,n,k", [
    (17, 1, 256),     # one output, one 256
    (32, 33, 512),    # exactly one group of rows; one weight row past a workgroup's 32, in a tile of its own
    (33, 130, 768),   # one row past; n no multiple of four
    (64, 100, 2304),  # nine 256s
])
def test_bits_of_the_tiles(dev, ty, act, m, n, k):
    q = QMatrix.from_raw_bytes(dev, (n, k), synth.random_weight(ty, n, k, seed=n + k, sigma=2e-3), ty)
    x = synth.random_activation(m, k, seed=m)
    x[3] = 0.0
    x[5, 7] = np.inf
    x[6, 9] = np.nan
    xt = Tensor.from_slice(dev, x) if act == "f32" else Tensor.from_slice(dev, synth.to_bf16_bits(x), dtype="bf16")
    got = {}
    for option in (5, 11):
        out = Tensor.filled_bytes(dev, (m, n), 0xFF)
        dev.set_option("matmul_kernel", option)
        try:
            got[option] = xt.q_mat_mul(q, out=out).as_slice()
        finally:
            dev.set_option("matmul_kernel", 0)
    rest = [r for r in range(m) if r not in (5, 6)]
    assert np.isfinite(got[11][rest]).all() and not got[11][3].any()
    assert np.array_equal(got[5].view(np.uint32)[rest + [5]], got[11].view(np.uint32)[rest + [5]])
    assert np.isnan(got[11][6]).all() and np.isnan(got[5][6]).all()
