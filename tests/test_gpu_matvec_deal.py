"""GPU parity: rows dealt out over the compute units (csrc/fh_dense.h: FhRowDeal) against float64, where a wavefront has no row, one, several, and where
a row is less than one piece of 512, whole pieces, or ends within one.

Bound: f32 products and sums of k terms of unit variance, a lane's chain of k / 64 of them: rounding errors of 2^-24 of either sign, 1e-6 of
sqrt(k), the results' deviation (a single result may be small beside its terms), and ten times that for the largest difference."""
import numpy as np
import pytest

from kalosm_amd import synth
from kalosm_amd.fusor import QMatrix, Tensor

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 7, 257, 1024, 1025, 4096, 4097, 10881])
@pytest.mark.parametrize("k", [8, 512, 520, 2048, 2060, 4108])
def test_products(dev, n, k):
    rng = np.random.default_rng(n * 8192 + k)
    w = synth.to_bf16_bits(rng.standard_normal(n * k, dtype=np.float32))
    x = rng.standard_normal((1, k), dtype=np.float32)
    out = Tensor.filled_bytes(dev, (1, n), 0xFF)
    got = Tensor.from_slice(dev, x).q_mat_mul(QMatrix.from_raw_bytes(dev, (n, k), w, synth.W_BF16), out=out).as_slice()
    off = got[0].astype(np.float64) - synth.from_bf16_bits(w).reshape(n, k).astype(np.float64) @ x[0].astype(np.float64)
    assert np.sqrt(np.mean(off * off)) <= 1e-6 * np.sqrt(k) and np.abs(off).max() <= 1e-5 * np.sqrt(k)
