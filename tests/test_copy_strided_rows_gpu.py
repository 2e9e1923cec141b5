"""Copies into dense rows from a source of any stride: row lengths at the edges of
the rule, of the 16-byte stores and of a workgroup, destinations that start at any
element, stepped, reversed and broadcast sources, bit-exact against the CPU oracle."""
import numpy as np
import pytest

from tests.copy_util import src_values
from tests.test_copy_gpu import E, check

pytestmark = pytest.mark.gpu

PAIRS = [("uint8", "float32"), ("float32", "uint8"), ("float32", "float32"), ("float64", "int16"), ("int64", "float64"),
         ("bool", "int32"), ("int32", "bool")]


@pytest.mark.parametrize("src_dtype,dst_dtype", PAIRS)
@pytest.mark.parametrize("length", [1000, 2047, 2048, 4095, 4097, 8192, 16383, 16384, 16397, 20007])
@pytest.mark.parametrize("step,off", [(3, 0), (2, 1), (-1, 3), (0, 2)])
def test_strided_rows(src_dtype, dst_dtype, length, step, off):
    s, d = np.dtype(src_dtype), np.dtype(dst_dtype)
    n = abs(step) * (length - 1) + 1
    sb = src_values(np.random.default_rng(length), s, d, (3, n + 5))
    view = np.lib.stride_tricks.as_strided(sb[:, n - 1:] if step < 0 else sb, (3, length),
                                           (sb.strides[0], step * s.itemsize))
    db = np.zeros(3 * (length + 1) + off, d)
    dv = np.lib.stride_tricks.as_strided(db[off:], (3, length), ((length + 1) * d.itemsize, d.itemsize))
    check(sb, view, d, db, dv, expect_kind=E if step else None)


def test_channels_last_images():
    sb = src_values(np.random.default_rng(0), "uint8", "float32", (5, 137, 141, 3))
    check(sb, sb.transpose(0, 3, 1, 2), np.dtype("float32"), expect_kind=E)
