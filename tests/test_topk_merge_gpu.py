"""The merge of a split row's segment winners: nseg * k around the 512 candidates
that are ranked directly, lists cut by the segments' bound (winners spread evenly,
all in one segment, all equal), and lists that the bound leaves too long."""
import numpy as np
import pytest

from tensorplay_amd import _capi

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(autouse=True)
def _no_knobs():
    yield
    _capi.debug_set("splits", 0)


def rows(kind, cols, rng):
    x = rng.standard_normal((3, cols)).astype(np.float32)
    if kind == "ascending":
        x.sort(axis=1)
    elif kind == "equal":
        x[:] = 1.5
    elif kind == "ties":
        x = np.round(x * 2).astype(np.float32)
    return x


@pytest.mark.parametrize("kind", ["random", "ascending", "equal", "ties"])
@pytest.mark.parametrize("k,splits", [(50, 5), (51, 10), (64, 8), (65, 8), (200, 9), (300, 12), (511, 9), (512, 3),
                                      (513, 4), (1024, 8)])
def test_merge(kind, k, splits):
    rng = np.random.default_rng(k)
    x = rows(kind, 200003, rng)
    _capi.debug_set("splits", splits)
    print(f"case merge {kind} k={k} splits={splits}", flush=True)
    for largest in (True, False):
        v, i = _capi.topk(torch.from_numpy(x).cuda(), k, largest)
        order = np.argsort(-x if largest else x, axis=1, kind="stable")[:, :k]
        np.testing.assert_array_equal(i.cpu().numpy(), order)
        np.testing.assert_array_equal(v.cpu().numpy(), np.take_along_axis(x, order, 1))
