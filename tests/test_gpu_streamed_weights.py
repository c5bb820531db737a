"""Products of one to sixteen rows of matrices on both sides of the size from which weights are read as a stream where there are more of them than the last
cache holds, and of the same matrix with and without others beside it: the same weights, the same sums."""
import numpy as np
import pytest

from kalosm_amd import synth
from kalosm_amd.fusor import Device, QMatrix, Tensor

pytestmark = pytest.mark.gpu

TYPES = [synth.Q4_0, 6, synth.Q8_0, synth.Q4_K, 13, synth.Q6_K]  # 6: Q5_0, 13: Q5_K


@pytest.mark.parametrize("rows", [1, 2, 3, 16])
@pytest.mark.parametrize("ty", TYPES)
def test_rows_do_not_depend_on_how_weights_are_read(ty, rows):
    """The upper rows of a matrix of 16 MB and more have the bits, up to the order of the sums, of the same rows as a small matrix."""
    dev, n, k, few = Device.gpu(0), 16384, 4096, 512
    part = synth.random_weight(ty, few, k, seed=ty)
    raw = np.tile(part, n // few)
    assert raw.nbytes >= 16 << 20
    x = synth.random_activation(rows, k, seed=rows)
    t = Tensor.from_slice(dev, x)
    got = t.q_mat_mul(QMatrix.from_raw_bytes(dev, (n, k), raw, ty)).as_slice().reshape(rows, n // few, few)
    want = t.q_mat_mul(QMatrix.from_raw_bytes(dev, (few, k), part, ty)).as_slice().reshape(rows, few)
    # every part of the large matrix is the same product in the same launch
    assert np.array_equal(got, np.broadcast_to(got[:, :1], got.shape))
    # 4096 products summed in another order in f32: 4096 * 2^-24 of the sum of their sizes at the very most; that sum is at most |x| . |w| over a row
    w = np.abs(QMatrix.from_raw_bytes(dev, (few, k), part, ty).dequantize().as_slice().astype(np.float64).reshape(few, k))
    bound = np.abs(x.astype(np.float64)).reshape(rows, k) @ w.T * 4096 * 2.0 ** -24
    assert (np.abs(got[:, 0].astype(np.float64) - want) <= bound).all()


@pytest.mark.parametrize("ty", TYPES)
def test_bits_do_not_depend_on_other_matrices(ty):
    """A matrix of 16 MB by itself is read plainly, beside 256 MB of others as a stream, and plainly again when they are gone."""
    dev, n, k = Device.gpu(0), 16384, 4096
    q = QMatrix.from_raw_bytes(dev, (n, k), np.tile(synth.random_weight(ty, 512, k, seed=ty), n // 512), ty)
    xs = [Tensor.from_slice(dev, synth.random_activation(rows, k, seed=rows)) for rows in (1, 2, 4, 16)]
    alone = [x.q_mat_mul(q).as_slice() for x in xs]
    others = QMatrix.from_raw_bytes(dev, (65536, 4096), np.zeros(65536 * 4096 // 32 * 34, np.uint8), synth.Q8_0)
    for x, want in zip(xs, alone):
        assert np.array_equal(x.q_mat_mul(q).as_slice(), want)
    del others
    for x, want in zip(xs, alone):
        assert np.array_equal(x.q_mat_mul(q).as_slice(), want)
