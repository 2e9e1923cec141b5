"""Integer and float64 reductions over short rows: lengths on both sides of a
vector, of 16 lanes and of 16 lanes of vectors, at any alignment, with ties and
the type's extremes, against numpy (exact: sums of integers, and of whole
numbers held in float64)."""
import numpy as np
import pytest

from tensorplay_amd import _capi

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

ROWS = 1003


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("n", [1, 2, 3, 7, 8, 9, 15, 16, 17, 24, 31, 32, 33, 47, 48, 49, 63, 64, 65, 100, 129, 255, 257])
@pytest.mark.parametrize("dt", ["int8", "uint8", "int16", "int32", "int64", "float64"])
def test_rows(dt, n, off):
    rng = np.random.default_rng(n * 2 + off)
    np_dt = np.dtype(dt)
    if dt == "float64":
        x = rng.integers(-1000, 1000, (ROWS, n)).astype(np_dt)
    else:
        i = np.iinfo(np_dt)
        lo, hi = max(i.min, -(1 << 40)), min(i.max, 1 << 40)
        x = rng.integers(lo, hi, (ROWS, n), endpoint=True, dtype=np_dt)
        x[::3, rng.integers(0, n)] = hi  # ties and extremes
        x[1::3, rng.integers(0, n)] = lo
    print(f"case short rows {dt} n={n} offset={off}", flush=True)
    buf = torch.empty(x.size + off, dtype=getattr(torch, dt), device="cuda")
    t = buf[off:].view(ROWS, n)
    t.copy_(torch.from_numpy(x))
    wide = np.float64 if dt == "float64" else np.int64
    np.testing.assert_array_equal(_capi.reduce(t, "sum", [1]).cpu().numpy(), x.sum(1, dtype=wide))
    np.testing.assert_array_equal(_capi.reduce(t, "amin", [1]).cpu().numpy(), x.min(1))
    np.testing.assert_array_equal(_capi.reduce(t, "argmax", [1]).cpu().numpy(), x.argmax(1))
    np.testing.assert_array_equal(_capi.reduce(t, "argmin", [1]).cpu().numpy(), x.argmin(1))
