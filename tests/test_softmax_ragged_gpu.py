"""Softmax and log_softmax rows, forward and gradient, that start and end at any
float: every register-row size class and the piece kernels at their edges,
against torch in float64 (the bounds of test_softmax_gpu.py), the row pieces'
exchange against the forced recompute, and rows of the piece kernels' lengths
replayed from a graph on changed inputs."""
import numpy as np
import pytest

from tensorplay_amd import _capi

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(autouse=True)
def _no_knobs():
    yield
    _capi.debug_set("smx_spin", 0)


def make(rows, n, off, seed):
    g = torch.Generator().manual_seed(seed)
    pad = (n + off + 3) // 4 * 4 + 4
    buf = torch.randn((rows, pad), generator=g) * 3
    return buf.cuda()[:, off:off + n]


def check(x, gy):
    print(f"case ragged shape={list(x.shape)} stride={x.stride(0)} offset={x.storage_offset()}", flush=True)
    xd, gd = x.double(), gy.double()
    for log in (False, True):
        y = _capi.softmax(x, -1, log=log)
        ref = (torch.log_softmax if log else torch.softmax)(xd, -1)
        lse = torch.logsumexp(xd - xd.amax(-1, keepdim=True), -1, keepdim=True)
        tol = 1e-5 * (ref.abs() + lse.abs()) + 2.0 ** -20 if log else 1e-5 * ref
        assert bool(((y.double() - ref).abs() <= tol).all())
        gx = _capi.softmax(gy, -1, log=log, grad_of=y)
        yd = y.double()
        if log:
            r = gd - yd.exp() * gd.sum(-1, keepdim=True)
            mag = gd.abs() + yd.exp() * gd.abs().sum(-1, keepdim=True)
        else:
            r = (gd - (gd * yd).sum(-1, keepdim=True)) * yd
            mag = (gd.abs() + (gd * yd).abs().sum(-1, keepdim=True)) * yd
        assert bool(((gx.double() - r).abs() <= 1e-5 * mag + 1e-12).all())


@pytest.mark.parametrize("n", [1, 3, 5, 63, 65, 77, 255, 257, 1021, 1025, 4095, 4099, 8193, 16381, 16383])
@pytest.mark.parametrize("off", [0, 1, 3])
def test_register_rows(n, off):
    check(make(37, n, off, n), make(37, n, (off + 1) % 4, n + 1))


@pytest.mark.parametrize("n", [16384, 16385, 16387, 40959, 40961, 40963, 49151, 49153, 98306, 151937])
@pytest.mark.parametrize("off", [0, 2])
def test_row_pieces(n, off):
    check(make(5, n, off, n), make(5, n, (off + 1) % 4, n + 1))


def test_many_odd_rows():
    check(make(400, 50001, 0, 7).contiguous(), make(400, 50001, 0, 8).contiguous())


@pytest.mark.parametrize("n", [50001, 81922, 98307])
def test_exchange_equals_recompute(n):
    x, g = make(40, n, 1, n), make(40, n, 0, n + 1)
    outs = []
    for spin in (0, -1):
        _capi.debug_set("smx_spin", spin)
        o = []
        for log in (False, True):
            y = _capi.softmax(x, -1, log=log)
            o += [y, _capi.softmax(g, -1, log=log, grad_of=y)]
        outs.append(o)
    for a, b in zip(*outs):
        assert torch.equal(a, b)


@pytest.mark.parametrize("n", [1023, 50003])
def test_non_finite_rows(n):
    x = make(6, n, 1, 3).clone()
    x[0, n - 1] = float("nan")
    x[1] = -float("inf")
    x[2, : n - 1] = -float("inf")
    x[3, n - 2] = float("inf")
    for log in (False, True):
        y = _capi.softmax(x, -1, log=log).cpu().numpy()
        ref = (torch.log_softmax if log else torch.softmax)(x[[2, 4, 5]].double(), -1).cpu().numpy()
        assert np.isnan(y[0]).all() and np.isnan(y[1]).all()
        assert y[2, n - 1] == (0.0 if log else 1.0)
        assert np.isnan(y[3, n - 2])
        fin = np.isfinite(ref[1:])
        np.testing.assert_allclose(y[4:][fin], ref[1:][fin], rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("shape", [(300, 50001), (300, 65536), (6, 1024, 256)])
def test_graph_replays_follow_the_inputs(shape):
    dim = -1 if len(shape) == 2 else 1
    x, g = torch.randn(shape, device="cuda"), torch.randn(shape, device="cuda")
    y0 = _capi.softmax(x, dim)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        y = _capi.softmax(x, dim)
        gx = _capi.softmax(g, dim, grad_of=y)
    for k in range(3):
        x.normal_(0, 1 + k)
        g.normal_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        ye = _capi.softmax(x, dim)
        ge = _capi.softmax(g, dim, grad_of=ye)
        torch.cuda.synchronize()
        # other kernels than the eager calls take, other orders of float32 sums
        torch.testing.assert_close(y, ye, rtol=1e-5, atol=1e-9)
        torch.testing.assert_close(gx, ge, rtol=1e-4, atol=1e-6)
    del y0
