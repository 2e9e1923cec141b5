"""Reduced runs that come near 2^31 elements are cut into chunks of 2^30 as
longer ones are (the kernels count a run's elements in int and look past its
end for their next element): the workspace holds the partial states of every
chunk.  The planner runs on the host, no GPU needed."""
import ctypes

import pytest

from tensorplay_amd import _capi

CHUNK = 1 << 30
LAST = (1 << 31) - 1 - (1 << 24)  # the longest run that one launch takes


def ws(op, sizes, strides, dims, dtype):
    out = _capi.default_out_dtype(op, dtype)
    d = _capi.make_desc(op, sizes, strides, dims, out, 1, in_dtype=dtype)
    return _capi.lib().tpr_reduce_workspace_bytes(ctypes.byref(d))


@pytest.mark.parametrize("op,dtype", [("sum", _capi.INT8), ("argmax", _capi.UINT8), ("sum", _capi.FLOAT32),
                                      ("norm", _capi.FLOAT32), ("sum", _capi.FLOAT64), ("var", _capi.FLOAT32)])
@pytest.mark.parametrize("n", [LAST + 1, (1 << 31) - 100000, (1 << 31) - 2, (1 << 31) - 1])
def test_runs_near_2_31_are_cut(op, dtype, n):
    one = ws(op, [CHUNK], [1], [0], dtype)
    assert one > 0 and ws(op, [n], [1], [0], dtype) == 2 * one
    # unsplit rows need no workspace in one launch; here two partial states of 8 bytes or more per row
    assert ws(op, [300, n], [n, 1], [1], dtype) >= 2 * 300 * 8
    cols = ws(op, [CHUNK, 200], [200, 1], [0], dtype)
    assert cols > 0 and ws(op, [n, 200], [200, 1], [0], dtype) == 2 * cols


@pytest.mark.parametrize("op,dtype", [("sum", _capi.INT8), ("argmax", _capi.FLOAT32)])
def test_shorter_runs_are_not(op, dtype):
    assert ws(op, [LAST], [1], [0], dtype) == ws(op, [CHUNK], [1], [0], dtype)
    assert ws(op, [LAST, 200], [200, 1], [0], dtype) == ws(op, [CHUNK, 200], [200, 1], [0], dtype)


@pytest.mark.parametrize("n", [LAST, LAST + 1, (1 << 31) - 2])
def test_run_kernel_takes_whole_runs(n):
    # two kept dims that do not merge: the run kernel, which cuts runs itself
    assert ws("sum", [2, 3, n], [8 * n, 2 * n, 1], [2], _capi.INT8) == ws("sum", [2, 3, LAST], [8 * LAST, 2 * LAST, 1],
                                                                         [2], _capi.INT8)
