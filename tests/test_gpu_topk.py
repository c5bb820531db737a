"""GPU parity: the two-launch top-k (csrc/fh_elementwise.hip: k_topk_keys, k_topk_pick) on the layouts where its threshold, its
gather and its chunks can go wrong, against the oracle.  Bit-equal pairs."""
import numpy as np
import pytest

from kalosm_amd.fusor import Tensor

pytestmark = pytest.mark.gpu


def _logits(layout, n, rng):
    x = rng.standard_normal(n).astype(np.float32)
    if layout == "rising":                      # the k largest maxima are the last lists, every key of them above the threshold
        return np.sort(x)
    if layout == "one_list":                    # the candidates in one list of 64
        x[n // 2 // 64 * 64:][:64] += 100
    elif layout == "spread":                    # one large value per list: more lists than candidates above any other value
        x[::64] += 100
    elif layout == "equal":                     # the order is that of the ids
        x[:] = -0.25
    elif layout == "few":                       # fewer finite values than candidates, in different lists
        x[:] = np.nan
        x[rng.choice(n, 7, replace=False)] = [1, 2, 2, -3, 0.0, -0.0, 1e-42]
    elif layout == "none":
        x[:] = -np.inf
    elif layout == "close":                     # differences in the last bits only
        x = (np.float32(3.0).view(np.uint32) + rng.integers(0, 40, n).astype(np.uint32)).view(np.float32)
    return x


@pytest.mark.parametrize("n", [1025, 4097, 32768, 131073, 1 << 20, (1 << 20) + 1])
@pytest.mark.parametrize("layout", ["rising", "one_list", "spread", "equal", "few", "none", "close"])
def test_layouts(dev, oracle, n, layout):
    x = _logits(layout, n, np.random.default_rng(n))
    t = Tensor.from_slice(dev, x)
    for k in (1, 2, 63, 200, 256):
        got, want = t.top_k_pairs(k), oracle.top_k(x, k)
        assert [g[0] for g in got] == [w[0] for w in want], (k, len(got), len(want))
        assert np.array_equal(np.float32([g[1] for g in got]).view(np.uint32), np.float32([w[1] for w in want]).view(np.uint32))
