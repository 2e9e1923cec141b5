"""Softmax along a strided dim with rows at any float: forward and gradient at
the edges of the row pieces (256 rows each) and of the 64-column groups, against
torch in float64 (the bounds of test_softmax_gpu.py), the pieces' exchange
against the forced recompute, and outer extents that take several launches."""
import pytest

from tensorplay_amd import _capi

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(autouse=True)
def _no_knobs():
    yield
    _capi.debug_set("smx_spin", 0)


def make(outer, n, inner, off, seed):
    g = torch.Generator().manual_seed(seed)
    buf = torch.randn(outer * n * inner + off, generator=g) * 3
    return buf.cuda()[off:].view(outer, n, inner)


def check(x, gy):
    print(f"case columns shape={list(x.shape)} offsets={x.storage_offset()},{gy.storage_offset()}", flush=True)
    xd, gd = x.double(), gy.double()
    for log in (False, True):
        y = _capi.softmax(x, 1, log=log)
        ref = (torch.log_softmax if log else torch.softmax)(xd, 1)
        lse = torch.logsumexp(xd - xd.amax(1, keepdim=True), 1, keepdim=True)
        tol = 1e-5 * (ref.abs() + lse.abs()) + 2.0 ** -20 if log else 1e-5 * ref
        assert bool(((y.double() - ref).abs() <= tol).all())
        gx = _capi.softmax(gy, 1, log=log, grad_of=y)
        yd = y.double()
        if log:
            r = gd - yd.exp() * gd.sum(1, keepdim=True)
            mag = gd.abs() + yd.exp() * gd.abs().sum(1, keepdim=True)
        else:
            r = (gd - (gd * yd).sum(1, keepdim=True)) * yd
            mag = (gd.abs() + (gd * yd).abs().sum(1, keepdim=True)) * yd
        assert bool(((gx.double() - r).abs() <= 1e-5 * mag + 1e-12).all())


@pytest.mark.parametrize("n", [2, 63, 65, 255, 256, 257, 511, 513, 768, 769, 1023, 1024, 1025, 3001])
@pytest.mark.parametrize("inner,off", [(16, 0), (16, 1), (17, 0), (63, 2), (64, 3), (65, 0), (67, 1), (130, 0)])
def test_edges(n, inner, off):
    check(make(3, n, inner, off, n), make(3, n, inner, (off + 1) % 4, n + 1))


@pytest.mark.parametrize("outer,n,inner", [(1500, 300, 65), (40, 1024, 2049)])
def test_more_pieces_than_exchange_slots(outer, n, inner):
    check(make(outer, n, inner, 0, 5), make(outer, n, inner, 0, 6))


@pytest.mark.parametrize("n", [257, 700, 1024])
@pytest.mark.parametrize("inner", [64, 77])
def test_exchange_equals_recompute(n, inner):
    x, g = make(9, n, inner, 0, n), make(9, n, inner, 0, n + 1)
    outs = []
    for spin in (0, -1):
        _capi.debug_set("smx_spin", spin)
        o = []
        for log in (False, True):
            y = _capi.softmax(x, 1, log=log)
            o += [y, _capi.softmax(g, 1, log=log, grad_of=y)]
        outs.append(o)
    for a, b in zip(*outs):
        assert torch.equal(a, b)


@pytest.mark.parametrize("n", [200, 600])
@pytest.mark.parametrize("inner", [64, 67])
def test_non_finite_stays_in_its_column(n, inner):
    x, g = make(2, n, inner, 0, 1), make(2, n, inner, 0, 2)
    g2 = g.clone()
    g2[1, n - 1, inner - 2] = float("nan")
    x2 = x.clone()
    x2[0, 3, inner - 1] = float("inf")
    y, y2 = _capi.softmax(x, 1), _capi.softmax(x2, 1)
    gx, gx2 = _capi.softmax(g, 1, grad_of=y), _capi.softmax(g2, 1, grad_of=y)
    bad = torch.zeros_like(x, dtype=torch.bool)
    bad[0, :, inner - 1] = True
    assert torch.equal(y2[~bad], y[~bad]) and bool(y2[0, 3, inner - 1].isnan())
    bad.zero_()
    bad[1, :, inner - 2] = True
    assert torch.equal(gx2[~bad], gx[~bad]) and bool(gx2[bad].isnan().all())
