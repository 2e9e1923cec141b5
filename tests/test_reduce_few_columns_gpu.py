"""Reductions over the rows of dense [.., R, few columns] views: every thread
count and remainder of the few-columns kernel against the general kernel (as
test_reduce_runs_gpu.py)."""
import pytest

from tensorplay_amd import _capi
from tests.test_reduce_runs_gpu import _no_knob, both  # noqa: F401

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("c", [1, 2, 3, 4, 5, 7, 16, 31, 64, 77, 100, 127, 128, 129])
@pytest.mark.parametrize("r", [64, 65, 701, 9000])
def test_float_columns(c, r):
    g = torch.Generator().manual_seed(c * r)
    x = torch.randn((3, r, c), generator=g).cuda()
    for op in ("sum", "mean", "amax", "var", "std", "norm", "any"):
        both(x, op, [1])
    both(x.round(), "argmax", [1])
    both(x[1], "argmin", [0])


@pytest.mark.parametrize("dtype", [torch.float64, torch.int64, torch.int32, torch.int16, torch.int8, torch.uint8, torch.bool])
@pytest.mark.parametrize("c", [1, 3, 5, 24, 128])
def test_other_types(dtype, c):
    g = torch.Generator().manual_seed(c)
    x = torch.randint(0, 120, (5, 1333, c), generator=g)
    x = (x > 60 if dtype == torch.bool else x.to(dtype)).cuda()
    for op in ("sum", "mean", "amax", "amin", "argmax", "all"):
        both(x, op, [1])
        both(x[1:, 1:], op, [1])  # rows that start at any element


def test_splits():
    x = torch.randn((2, 50000, 3), generator=torch.Generator().manual_seed(1)).cuda()
    for splits in (1, 2, 5, 70):
        _capi.debug_set("splits", splits)
        try:
            for op in ("sum", "var", "argmin"):
                both(x, op, [1])
        finally:
            _capi.debug_set("splits", 0)
