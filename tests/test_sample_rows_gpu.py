"""The sort-free draw of tpr_sample (k > 1024): rows on both sides of every
register-part size, rows that start at any element, k = cols and k < cols, lists
that overflow (flat rows, top_p = 1) and rows whose sums are not finite."""
import numpy as np
import pytest

from oracle import oracle as O
from tensorplay_amd import _capi
from test_sample_gpu import check_large_k

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

V = 4 * 512  # elements of one vector per thread


def logits(rng, rows, cols, scale=2.0):
    x = (rng.standard_normal((rows, cols)) * scale).astype(np.float32)
    x[:, rng.integers(0, cols, 4)] += np.float32(6.0)
    return x


@pytest.mark.parametrize("cols", [1025, 2047, 6 * V - 1, 6 * V, 14 * V + 1, 24 * V, 36 * V + 3, 54 * V, 54 * V + 4 * V + 2,
                                  62 * V - 1, 62 * V, 62 * V + 5, 71 * V + 3])
@pytest.mark.parametrize("T,top_p", [(0.8, 0.9), (1.0, 1.0), (0.0, 0.5)])
def test_row_lengths(cols, T, top_p):
    rng = np.random.default_rng(cols)
    x = logits(rng, 3, cols)
    u = rng.random(3).astype(np.float32)
    check_large_k(x, u, cols, T, top_p)
    if cols > 1100:
        check_large_k(x, u, 1100, T, top_p)


@pytest.mark.parametrize("offset", [1, 2, 3])
def test_rows_at_any_element(offset):
    rng = np.random.default_rng(offset)
    cols, stride = 30001, 30007
    buf = logits(rng, 5, stride)
    x = np.ascontiguousarray(buf[:, offset:offset + cols])
    u = rng.random(5).astype(np.float32)
    t = torch.from_numpy(buf).cuda()[:, offset:offset + cols]
    print(f"case sample_rows offset={offset}", flush=True)
    got = _capi.sample(t, torch.from_numpy(u).cuda(), cols, 0.7, 0.9).cpu().numpy()
    exp, margin = O.sample(x, u, cols, 0.7, 0.9)
    np.testing.assert_array_equal(got[margin > 1e-5], exp[margin > 1e-5])


@pytest.mark.parametrize("k", [1500, 20000])
def test_flat_rows_overflow_the_list(k):
    rng = np.random.default_rng(k)
    x = (rng.standard_normal((4, 20000)) * 0.01).astype(np.float32)
    x[2] = 1.5                                         # all equal: ties by index
    x[3] = rng.integers(0, 3, 20000).astype(np.float32)  # heavy ties
    u = np.array([0.1, 0.6, 0.35, 0.9], np.float32)
    for top_p in (0.3, 0.95, 1.0):
        check_large_k(x, u, k, 1.0, top_p)


def test_rows_without_finite_sums():
    rng = np.random.default_rng(9)
    x = (rng.standard_normal((5, 3000)) * 2).astype(np.float32)
    x[0, 7] = np.nan
    x[1, 8] = np.inf
    x[2] = -np.inf
    x[3, ::2] = -np.inf  # masked logits: weight 0
    u = np.full(5, 0.5, np.float32)
    print("case sample_rows non-finite", flush=True)
    for k in (3000, 1300):
        got = _capi.sample(torch.from_numpy(x).cuda(), torch.from_numpy(u).cuda(), k, 1.0, 0.9).cpu().numpy()
        with np.errstate(invalid="ignore"):
            exp, margin = O.sample(x, u, k, 1.0, 0.9)
        np.testing.assert_array_equal(got[:3], exp[:3])
        sure = margin[3:] > 1e-5
        np.testing.assert_array_equal(got[3:][sure], exp[3:][sure])
