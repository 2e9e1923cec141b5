"""tpr_softmax with its output over one of its inputs: rows and strided dims
that a call with its own output cuts into pieces, with the wait for the other
pieces cut short (smx_spin = -1: a piece then reads the others' input again),
against torch in float64 with the bounds of test_softmax_gpu.py."""
import ctypes

import pytest

from tensorplay_amd import _capi

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(autouse=True, params=[0, -1], ids=["wait", "no_wait"])
def _spin(request):
    _capi.debug_set("smx_spin", request.param)
    yield
    _capi.debug_set("smx_spin", 0)


def call(mode, shape, a, b, out):
    d = _capi.SoftmaxDesc()
    d.mode, d.dtype = mode, _capi.FLOAT32
    d.outer, d.n, d.inner = shape
    for s in (d.a_strides, d.b_strides):
        s[0], s[1], s[2] = shape[1] * shape[2], shape[2], 1
    L = _capi.lib()
    n = L.tpr_softmax_workspace_bytes(ctypes.byref(d))
    ws = torch.empty(max(n, 1), dtype=torch.uint8, device="cuda")
    ptr = lambda t: ctypes.c_void_p(t.data_ptr() if t is not None else 0)
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert L.tpr_softmax(ctypes.byref(d), ptr(a), ptr(b), ptr(out), ptr(ws), n, st) == _capi.OK
    return out


def inputs(shape, off):
    g = torch.Generator(device="cuda").manual_seed(shape[1] + off)
    n = shape[0] * shape[1] * shape[2]
    x = (torch.randn(n + off, generator=g, device="cuda") * 3)[off:].view(shape)
    return x, torch.randn(n + off, generator=g, device="cuda")[off:].view(shape)


def own(t, off):
    """A copy of t at the same offset from a 16-byte address."""
    buf = torch.empty(t.numel() + off, device="cuda")
    return buf[off:].view(t.shape).copy_(t)


# rows of one CU and more, of whole vectors and not; 300 rows: more than CUs
ROWS = [(3, 16388, 0), (3, 16387, 0), (300, 45000, 0), (300, 45001, 0), (5, 45000, 1), (3, 163840, 0), (3, 163841, 0),
        (300, 50260, 0)]
COLS = [(4, n, inner, 0) for n in (300, 700, 1024) for inner in (64, 67)] + [(40, 700, 64, 1), (40, 1000, 1024, 0)]
CASES = [((r, n, 1), off) for r, n, off in ROWS] + [((o, n, i), off) for o, n, i, off in COLS]


@pytest.mark.parametrize("shape,off", CASES)
@pytest.mark.parametrize("log", [False, True])
def test_forward_over_its_input(shape, off, log):
    print(f"case softmax in place shape={shape} offset={off} log={log}", flush=True)
    x, _ = inputs(shape, off)
    xd = x.double()
    ref = (torch.log_softmax if log else torch.softmax)(xd, 1)
    tol = 1e-5 * ref
    if log:
        lse = torch.logsumexp(xd - xd.amax(1, keepdim=True), 1, keepdim=True)
        tol = 1e-5 * (ref.abs() + lse.abs()) + 2.0 ** -20
    y = call(_capi.LOG_SOFTMAX_FWD if log else _capi.SOFTMAX_FWD, shape, x, None, x)
    assert bool(((y.double() - ref).abs() <= tol).all())


@pytest.mark.parametrize("shape,off", CASES)
@pytest.mark.parametrize("log", [False, True])
@pytest.mark.parametrize("over", ["g", "y"])
def test_gradient_over_an_input(shape, off, log, over):
    print(f"case softmax gradient over {over} shape={shape} offset={off} log={log}", flush=True)
    x, g = inputs(shape, off)
    y = own((torch.log_softmax if log else torch.softmax)(x, 1), off)
    gd, yd = g.double(), y.double()
    if log:
        ref = gd - yd.exp() * gd.sum(1, keepdim=True)
        mag = gd.abs() + yd.exp() * gd.abs().sum(1, keepdim=True)
    else:
        ref = (gd - (gd * yd).sum(1, keepdim=True)) * yd
        mag = (gd.abs() + (gd * yd).abs().sum(1, keepdim=True)) * yd
    out = g if over == "g" else y
    r = call(_capi.LOG_SOFTMAX_BWD if log else _capi.SOFTMAX_BWD, shape, g, y, out)
    assert bool(((r.double() - ref).abs() <= 1e-5 * mag + 1e-12).all())
