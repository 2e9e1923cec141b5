"""The run kernel of tpr_reduce (several reduced dims, or kept dims that do not
merge, over contiguous runs) and the views whose dims are visited in memory
order, against the general kernel (forced by the test build's `general` knob),
which walks any view element by element.  Both accumulate in 64 bits, so float
results differ by the final rounding at most; indices, extrema and integers
are equal."""
import numpy as np
import pytest

from tensorplay_amd import _capi

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

OPS = ["sum", "mean", "prod", "amax", "amin", "var", "std", "norm", "all", "any"]


@pytest.fixture(autouse=True)
def _no_knob():
    yield
    _capi.debug_set("general", 0)


def both(x, op, dims, **kw):
    print(f"case runs {op} dims={dims} shape={list(x.shape)} strides={list(x.stride())} {x.dtype}", flush=True)
    got = _capi.reduce(x, op, dims, **kw)
    again = _capi.reduce(x, op, dims, **kw)
    _capi.debug_set("general", 1)
    exp = _capi.reduce(x, op, dims, **kw)
    _capi.debug_set("general", 0)
    assert torch.equal(torch.nan_to_num(got.float()), torch.nan_to_num(again.float()))
    got, exp = got.cpu().numpy(), exp.cpu().numpy()
    if got.dtype.kind == "f" and op not in ("amax", "amin"):
        # two orders of a 64-bit sum, then one rounding to the output type
        tol = 2.0 ** -22 if got.dtype == np.float32 else 1e-12
        np.testing.assert_allclose(got, exp, rtol=tol, atol=1e-11 if op in ("sum", "mean") else 0)
    else:
        np.testing.assert_array_equal(got, exp)
        if got.dtype == np.float32:
            np.testing.assert_array_equal(np.signbit(got), np.signbit(exp))


@pytest.mark.parametrize("L", [4, 5, 15, 16, 17, 63, 64, 255, 257, 1025, 4100, 17000])
def test_run_lengths(L):
    rng = np.random.default_rng(L)
    n = max(2, min(40, 40000 // L))
    x = torch.from_numpy((rng.standard_normal((n, 5, L)) + 0.5).astype(np.float32)).cuda()
    for op in OPS:
        y = x * 0.01 + 1 if op == "prod" else x.round() if op in ("amax", "amin", "any", "all") else x
        both(y, op, [0, 2])


@pytest.mark.parametrize("dtype", [torch.float64, torch.int64, torch.int32, torch.int16, torch.int8, torch.uint8, torch.bool])
@pytest.mark.parametrize("L", [7, 49, 4099])
def test_element_types(dtype, L):
    g = torch.Generator().manual_seed(L)
    x = torch.randint(0, 100, (9, 3, L), generator=g)
    x = (x > 2) if dtype == torch.bool else x.to(dtype)
    for off in (0, 1):
        v = x.cuda()[:, :, off:]
        for op in ["sum", "mean", "amax", "amin", "all", "any"] + (["var", "norm"] if dtype == torch.float64 else []):
            both(v, op, [0, 2])


def test_several_outer_dims_and_kept_dims():
    rng = np.random.default_rng(5)
    x = torch.from_numpy(rng.standard_normal((3, 4, 5, 6, 37)).astype(np.float32).round(1)).cuda()
    for dims in ([0, 2, 4], [1, 4], [0, 1, 3, 4], [2, 4], [1, 2, 4]):
        for op in OPS:
            both(x, op, dims)
    v = x[:, 1:3, :, ::2, 1:]  # kept dims that do not merge, rows at odd elements
    for dims in ([4], [0, 4], [1, 2, 4]):
        for op in ("sum", "amax", "std", "any"):
            both(v, op, dims)
    both(v, "argmax", [4])
    both(v, "argmin", [4])


def test_memory_order_views():
    rng = np.random.default_rng(6)
    x = torch.from_numpy(rng.standard_normal((17, 33, 65)).astype(np.float32).round(1)).cuda()
    for perm in ([1, 2, 0], [2, 1, 0], [0, 2, 1], [2, 0, 1]):
        v = x.permute(perm)
        for dims in ([0], [1], [2], [0, 1], [0, 2], [1, 2], None):
            for op in OPS + (["argmax", "argmin"] if dims is None or len(dims) == 1 else []):
                both(v, op, dims)
    # the sign of a zero maximum is the first one's in the view's order
    z = torch.zeros(2, 3, 8, device="cuda")
    z[0, 0, 1:] = -0.0
    z[1] = -0.0
    for perm in ([0, 1, 2], [2, 1, 0], [1, 2, 0]):
        both(z.permute(perm), "amax", None)
        both(-z.permute(perm), "amin", [0, 2])
    both(x.expand(17, 33, 65)[:, :1].expand(17, 9, 65), "sum", [0, 1, 2])  # a broadcast dim


def test_long_kept_extent_and_split_count():
    g = torch.Generator().manual_seed(3)
    for shape, dims in (((5, 3000, 12), [0, 2]), ((300, 1, 3000), [0, 2]), ((64, 2, 3136), [0, 2])):
        x = torch.randn(shape, generator=g).cuda()
        for op in ("sum", "var", "amin"):
            both(x, op, dims)
    x = torch.randn((4, 3, 5000), generator=g).cuda()
    for splits in (1, 2, 7, 40):
        _capi.debug_set("splits", splits)
        try:
            both(x, "mean", [0, 2])
            both(x, "amax", [0, 2])
        finally:
            _capi.debug_set("splits", 0)
