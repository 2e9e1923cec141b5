"""nll_loss at the edges of its kernels: class counts that are no multiple of a
vector, sample counts on both sides of the single-workgroup forward."""
import pytest

from tensorplay_amd import _capi

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("c", [1, 2, 3, 5, 10, 77, 1000, 1023, 1024, 1025, 4099])
@pytest.mark.parametrize("n", [1, 63, 4096, 4097])
@pytest.mark.parametrize("reduction", [0, 1, 2])
def test_values_and_gradient(n, c, reduction):
    g = torch.Generator().manual_seed(n * 7 + c)
    x = torch.randn((n, c), generator=g).cuda()
    t = torch.randint(0, c, (n,), generator=g)
    t[::5] = -100  # ignored
    t = t.cuda()
    w = (torch.rand((c,), generator=g) + 0.5).cuda()
    print(f"case nll n={n} c={c} reduction={reduction}", flush=True)
    out, tw, status = _capi.nll_loss(x, t, w, reduction)
    keep = t >= 0
    at = t.clamp(min=0)
    wt = torch.where(keep, w[at], 0.0)
    li = -x.gather(1, at[:, None])[:, 0] * wt  # float32, as the kernel
    assert int(status) == 0
    torch.testing.assert_close(tw[0].double(), wt.double().sum(), rtol=1e-6, atol=0)
    if reduction == 0:
        assert torch.equal(out, torch.where(keep, li, 0.0))
    else:
        s = li.double().sum() / (tw[0].double() if reduction == 1 and float(tw) > 0 else 1.0)
        torch.testing.assert_close(out.double(), s, rtol=1e-6, atol=1e-9)
    go = torch.randn((n,) if reduction == 0 else (1,), generator=g).cuda()
    gi = _capi.nll_loss_backward(go, t, n, c, w, reduction, -100, tw)
    gv = go if reduction == 0 else go.expand(n)
    if reduction == 1 and float(tw) > 0:
        gv = (gv.double() / tw[0].double()).float()
    ref = torch.zeros((n, c), device="cuda").scatter_(1, at[:, None], torch.where(keep, -w[at] * gv, 0.0)[:, None])
    assert torch.equal(gi, ref)


def test_targets_out_of_range_set_the_flag():
    for n in (5, 5000):
        x = torch.zeros((n, 7), device="cuda")
        t = torch.zeros((n,), dtype=torch.int64, device="cuda")
        t[n - 1] = 7
        assert int(_capi.nll_loss(x, t)[2]) == 1
        gi = _capi.nll_loss_backward(torch.ones(1, device="cuda"), t, n, 7, None, 2)
        assert float(gi[n - 1].abs().sum()) == 0 and float(gi.sum()) == -(n - 1)


@pytest.mark.parametrize("n", [1, 2, 3, 5])
@pytest.mark.parametrize("past", [0, 1, 2, 3])
def test_weighted_target_past_the_last_class(n, past):
    """The last sample's target c .. c + 3 has no column: its row is all zeros
    (n * 7 leaves remainders of 1, 2 and 3 to the last vector)."""
    c = 7
    print(f"case nll weighted last target c+{past} n={n}", flush=True)
    w = (torch.arange(c, dtype=torch.float32) + 1).cuda()
    t = torch.arange(n, dtype=torch.int64) % c
    t[n - 1] = c + past
    go = torch.full((1,), 2.0, device="cuda")
    gi = _capi.nll_loss_backward(go, t.cuda(), n, c, w, 2).cpu()
    ref = torch.zeros((n, c))
    for i in range(n - 1):
        ref[i, t[i]] = -2.0 * float(t[i] + 1)
    assert torch.equal(gi, ref)
