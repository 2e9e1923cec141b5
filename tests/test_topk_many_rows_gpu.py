"""Top-k and draws of more rows than the threads of one launch allow (2^32; a
larger launch runs the rest modulo 2^32 and reports nothing)."""
import pytest

from tensorplay_amd import _capi

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(autouse=True)
def _free():
    torch.cuda.empty_cache()
    yield
    torch.cuda.empty_cache()


def named(n):
    return torch.arange(n, device="cuda", dtype=torch.int32) % 97


def test_register_select():
    n = 17_000_000  # 256 threads a row
    print(f"case topk int8 [{n}, 5] k=2", flush=True)
    v = named(n)
    x = torch.zeros((n, 5), dtype=torch.int8, device="cuda")
    x.scatter_(1, (v % 5).long()[:, None], 9)
    x.scatter_(1, ((v + 2) % 5).long()[:, None], 5)
    vals, idx = _capi.topk(x, 2)
    assert bool((vals[:, 0] == 9).all()) and bool((vals[:, 1] == 5).all())
    assert torch.equal(idx[:, 0], (v % 5).long()) and torch.equal(idx[:, 1], ((v + 2) % 5).long())


def test_lane_groups():
    n, c, k = 70_000_000, 18, 17  # 64 lanes a row
    print(f"case topk float32 [{n}, {c}] k={k}", flush=True)
    v = named(n)
    x = v.float()[:, None] + torch.arange(c, device="cuda")
    vals, idx = _capi.topk(x, k)
    assert torch.equal(vals[:, 0], v.float() + (c - 1)) and torch.equal(vals[:, k - 1], v.float() + 1)
    del vals
    want = torch.arange(c - 1, 0, -1, device="cuda")
    for a in range(0, n, 1 << 24):
        assert bool((idx[a:a + (1 << 24)] == want).all())


def test_draws():
    n, c = 70_000_000, 18
    print(f"case sample [{n}, {c}] k=2", flush=True)
    v = (named(n) % c).long()
    x = torch.zeros((n, c), device="cuda")
    x.scatter_(1, v[:, None], 2.0)
    x.scatter_(1, ((v + 1) % c)[:, None], 1.9)
    u = torch.zeros(n, device="cuda")
    u[1::2] = 0.99
    ids = _capi.sample(x, u, 2, 1.0, 1.0)
    odd = torch.arange(n, device="cuda") % 2
    assert torch.equal(ids, (v + odd) % c)
