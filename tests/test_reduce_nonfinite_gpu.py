"""Infinities, NaN and a far first element (the shift of the shared-shift
variance) in every layout that float32 reductions have kernels for, against
numpy in float64 and the oracle: a special value changes its own output only."""
import numpy as np
import pytest

from oracle import oracle as O
from tensorplay_amd import _capi
from tests.gpu_util import assert_bits_equal

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

# shape, reduced dims: full and partial register rows, other rows, split rows, a full
# reduction, columns (16-byte and odd), few columns, runs (one vector per lane, chunks)
LAYOUTS = [((3000, 1024), [1]), ((3000, 1000), [1]), ((40, 77), [1]), ((3, 70001), [1]), ((500000,), [0]),
           ((300, 512), [0]), ((5, 70, 131), [1]), ((4, 9000, 3), [1]), ((6, 5, 14, 14), [0, 2, 3]),
           ((8, 3, 9001), [0, 2])]


def run(x, op, dims):
    return _capi.reduce(torch.from_numpy(x).cuda(), op, dims).cpu().numpy()


def reference(x, op, dims):
    d, ax = x.astype(np.float64), tuple(dims)
    with np.errstate(all="ignore"):
        if op in ("var", "std"):
            return getattr(d, op)(axis=ax, ddof=1)
        return getattr(d, op)(axis=ax)


def first_of(x, dims, out):
    """The index of the first element of output `out` (a multi-index over the kept dims)."""
    kept = iter(out)
    return tuple(0 if i in dims else next(kept) for i in range(x.ndim))


@pytest.mark.parametrize("shape,dims", LAYOUTS)
@pytest.mark.parametrize("special", ["inf", "-inf", "nan", "both"])
@pytest.mark.parametrize("at", ["first", "last"])
def test_special_values(shape, dims, special, at):
    rng = np.random.default_rng(len(shape) + shape[0])
    x = rng.standard_normal(shape).astype(np.float32)
    clean = {op: run(x, op, dims) for op in ("sum", "mean", "var", "std")}
    outs = clean["sum"].shape
    out = tuple(s // 2 for s in outs)
    first = first_of(x, dims, out)
    last = tuple(x.shape[i] - 1 if i in dims else first[i] for i in range(x.ndim))
    y = x.copy()
    if special == "both":
        y[first], y[last] = np.inf, -np.inf
    else:
        y[first if at == "first" else last] = float(special)
    print(f"case non-finite {special} {at} shape={shape} dims={dims}", flush=True)
    rest = np.ones(outs, bool)
    rest[out] = False
    for op in ("sum", "mean", "var", "std"):
        got = run(y, op, dims)
        np.testing.assert_array_equal(got[rest], clean[op][rest])
        np.testing.assert_array_equal(got[out], reference(y, op, dims)[out])  # an infinity or NaN
    # the oracle reduces one dim, so a slice laid out alike stands for several
    moved = np.moveaxis(y, dims, range(y.ndim - len(dims), y.ndim)).reshape(-1, int(np.prod([shape[d] for d in dims])))
    assert_bits_equal(run(y, "amax", dims).reshape(-1), O.amax(np.ascontiguousarray(moved), [1]))
    assert_bits_equal(run(y, "amin", dims).reshape(-1), O.amin(np.ascontiguousarray(moved), [1]))
    if len(dims) == 1:
        np.testing.assert_array_equal(run(y, "argmax", dims).reshape(-1), O.argmax(np.ascontiguousarray(moved), 1))


@pytest.mark.parametrize("shape,dims", LAYOUTS + [((1 << 24,), [0]), ((16, 1 << 20), [1]), ((1 << 22, 4), [0])])
@pytest.mark.parametrize("first", [0.0, 1e4, -3e18])
def test_variance_around_a_far_first_element(shape, dims, first):
    """The shared shift is the output's first element K; its own term bounds what
    the shifted sums lose: n 2^-53 of the sum of squares (2e-9 at 2^24
    elements), below half an ulp of the float32 result (6e-8)."""
    rng = np.random.default_rng(shape[0])
    x = rng.standard_normal(shape).astype(np.float32) + np.float32(5)
    if first:
        idx = tuple(slice(0, 1) if i in dims else slice(None) for i in range(len(shape)))
        x[idx] = first
    print(f"case far first element {first} shape={shape} dims={dims}", flush=True)
    for op in ("var", "std"):
        got = run(x, op, dims).astype(np.float64)
        ref = reference(x, op, dims)
        assert np.abs(got / ref - 1).max() <= 2.0 ** -23  # rounding to float32, and std's square root
