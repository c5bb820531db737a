"""GPU parity: one row of k whose 256s no number of up to 16 wavefronts shares out evenly (43 of 11008 columns), and 3 and 4 rows of 5-bit matrices, in one
launch (2048 columns) and element by element (11008), against 64 bits.

Bound: as of products of a few rows, but that the kernels of one row multiply f16 subnormals, which lose up to 1.3e-6 of a product."""
import numpy as np
import pytest

from kalosm_amd import synth
from kalosm_amd.fusor import QMatrix, Tensor
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


def alternating(ty, raw, n, k, row, bits):
    """`raw` with scale `bits` and its largest and smallest codes in turn (scales of one, offsets of none) in the last block of a row."""
    per, size = k // synth.BLOCK_ELEMS[ty], synth.BLOCK_BYTES[ty]
    out = raw.copy().reshape(n, per, size)
    block = out[row, -1]
    codes = np.tile(np.array([0xFF, 0], np.uint8), 100)
    if ty == synth.Q6_K:
        block[0:192], block[192:208] = codes[:192], 1
        block[208:210] = np.array([bits], np.uint16).view(np.uint8)
    else:
        block[0:2] = np.array([bits], np.uint16).view(np.uint8)
        if ty == synth.Q4_K:
            block[2:4], block[4:16] = 0, synth.pack_k4_scales(np.ones(8), np.zeros(8))
        block[size - (16 if ty == synth.Q4_0 else 128):] = codes[:16 if ty == synth.Q4_0 else 128]
    return out.reshape(-1)


@pytest.mark.parametrize("ty", [synth.Q4_0, synth.Q4_K, synth.Q6_K], ids=lambda t: synth.TYPE_NAMES[t])
@pytest.mark.parametrize("blocks", [17, 31, 43])
def test_infinite_scale_of_the_last_block(dev, ty, blocks):
    """A wavefront with fewer blocks than others multiplies the last one again by nothing: an infinite scale there gives the infinity that it stands for."""
    n, k = 48, 256 * blocks
    raw = synth.random_weight(ty, n, k, seed=1)
    x = synth.random_activation(1, k, seed=2)
    x[0, -256:] = np.tile(np.array([-1.0, 1.5], np.float32), 128)  # large codes meet the negative ones, the sum is positive
    t = Tensor.from_slice(dev, x)
    got, want = (t.q_mat_mul(QMatrix.from_raw_bytes(dev, (n, k), alternating(ty, raw, n, k, 5, bits), ty)).as_slice()[0] for bits in (0x7C00, 0x3C00))
    assert got[5] == -np.inf
    got[5] = want[5]
    assert np.array_equal(got, want)


@pytest.mark.parametrize("ty", [synth.Q4_0, synth.Q4_K], ids=lambda t: synth.TYPE_NAMES[t])
def test_tiny_activations_of_one_row(dev, ty):
    """Down to 2^-113 a power of two more or less in the activations changes nothing but the results' exponents: 22 bits of each are there."""
    n, k = 48, 256 * 43
    q = QMatrix.from_raw_bytes(dev, (n, k), synth.random_weight(ty, n, k, seed=1), ty)
    x = synth.random_activation(1, k, seed=2)
    want = Tensor.from_slice(dev, x).q_mat_mul(q).as_slice().astype(np.float64)
    rms = np.sqrt((want ** 2).mean())
    for e in (-60, -90, -113):
        got = Tensor.from_slice(dev, np.ldexp(x, e)).q_mat_mul(q).as_slice().astype(np.float64)
        # the products are exact and the sums the same; a bit that leaves a low term is 2^-22 of an activation
        assert np.sqrt(((np.ldexp(got, -e) - want) ** 2).mean()) <= 2.0 ** -22 * rms, e


@pytest.mark.parametrize("ty", [synth.Q5_0, synth.Q8_0, synth.Q5_K], ids=lambda t: synth.TYPE_NAMES[t])
@pytest.mark.parametrize("rows", [1, 2])
def test_formats_that_would_lose_bits(dev, oracle, ty, rows):
    """Ragged rows of the formats whose single-row kernel is further from 64 bits (Q8_0 1.9e-6 of the results' size, Q5_0 9e-7, Q5_K 4e-7) stay with the
    kernels that sum them to 3.1e-7; those of the 5-bit formats take f32 values as they are, whatever their exponents, infinities among them."""
    n, k = 512, 256 * 43
    q, w = matrix(dev, oracle, ty, n, k)
    x = synth.random_activation(rows, k, seed=2)
    got = Tensor.from_slice(dev, x).q_mat_mul(q).as_slice()
    want = x.astype(np.float64) @ w.T
    assert np.sqrt(((got - want) ** 2).mean()) <= 3.5e-7 * np.sqrt((want ** 2).mean())
    if ty == synth.Q8_0:
        return
    assert np.array_equal(np.ldexp(Tensor.from_slice(dev, np.ldexp(x, -100)).q_mat_mul(q).as_slice(), 100), got)
    x[0, 5] = np.inf
    got = Tensor.from_slice(dev, x).q_mat_mul(q).as_slice()
    assert np.array_equal(got[0], np.where(w[:, 5] == 0, np.nan, np.copysign(np.inf, w[:, 5])).astype(np.float32), equal_nan=True)
    assert np.isfinite(got[1:]).all()


@pytest.mark.parametrize("ty", [synth.Q5_0, synth.Q5_K], ids=lambda t: synth.TYPE_NAMES[t])
@pytest.mark.parametrize("m", [3, 4])
@pytest.mark.parametrize("blocks", [17, 43, 61, 112])
def test_few_ragged_rows_of_five_bits(dev, ty, m, blocks):
    """3 and 4 rows of what the single-row kernel does not share out: f32 values as they are, so powers of two come through."""
    n, k = 512, 256 * blocks
    q = QMatrix.from_raw_bytes(dev, (n, k), synth.random_weight(ty, n, k, seed=1), ty)
    x = synth.random_activation(m, k, seed=2)
    got = [Tensor.from_slice(dev, np.ldexp(x, e)).q_mat_mul(q).as_slice() for e in (0, -100)]
    assert np.array_equal(np.ldexp(got[1], 100), got[0])
