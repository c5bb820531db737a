"""GPU parity: one row of k whose 256s no number of up to 16 wavefronts shares out evenly (43 of 11008 columns), and 3 and 4 rows of 5-bit matrices in one
launch, against 64 bits.

Bound: as of products of a few rows, but that the kernels of one row multiply f16 subnormals, which lose up to 1.3e-6 of a product."""
import numpy as np
import pytest

from kalosm_amd import synth
from kalosm_amd.fusor import Tensor
from test_gpu_qmv_rows import close, matrix, named

pytestmark = pytest.mark.gpu


@named
@pytest.mark.parametrize("n,blocks", [(16, 17), (33, 19), (70, 31), (50, 34), (48, 43), (20, 61)])
def test_one_row(dev, oracle, ty, n, blocks):
    q, w = matrix(dev, oracle, ty, n, 256 * blocks)
    x = synth.random_activation(1, 256 * blocks, seed=2)
    out = Tensor.filled_bytes(dev, (1, n), 0xFF)
    got = Tensor.from_slice(dev, x).q_mat_mul(q, out=out).as_slice().astype(np.float64)
    err, mag = np.abs(got - x.astype(np.float64) @ w.T), np.abs(x).astype(np.float64) @ np.abs(w).T
    assert np.isfinite(got).all() and (err <= (2.0 ** -19 + 1.3e-6) * mag).all()
    add = [Tensor.from_slice(dev, synth.random_activation(1, n, seed=s)) for s in (3, 4)]  # the other epilogue
    both = Tensor.from_slice(dev, x).q_mat_mul_add2(q, *add).as_slice()
    assert np.array_equal(both, (got.astype(np.float32) + add[0].as_slice()) + add[1].as_slice())


@pytest.mark.parametrize("ty", [synth.Q5_0, synth.Q5_K], ids=lambda t: synth.TYPE_NAMES[t])
@pytest.mark.parametrize("m", [3, 4])
@pytest.mark.parametrize("n,k", [(1030, 2048), (520, 11008)])
def test_few_rows_of_five_bits(dev, oracle, ty, m, n, k):
    q, w = matrix(dev, oracle, ty, n, k)
    x = synth.random_activation(m, k, seed=2) * np.exp(np.random.default_rng(3).standard_normal((m, 1))).astype(np.float32)
    close(Tensor.from_slice(dev, x).q_mat_mul(q).as_slice().astype(np.float64), x, w)
