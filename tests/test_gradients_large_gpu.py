"""Gradients that would take more threads than a launch counts (2^32; a larger
one runs the rest modulo 2^32 and reports nothing)."""
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
    return (torch.arange(n, device="cuda", dtype=torch.int32) % 97).float()


def test_variance_of_many_short_rows():
    n = 68_000_000  # a wave each
    print(f"case var gradient [{n}, 4]", flush=True)
    v = named(n)
    x = v[:, None].repeat(1, 4)
    x[:, 0] += 4  # mean v + 1, deviations 3, -1, -1, -1
    g = _capi.reduce_backward(v, x, "var", [1])  # 2 v (x - mean) / 3
    assert torch.equal(g[:, 0], v * 2) and torch.equal(g[:, 3], (v * -2.0).double().div(3).float())


def test_variance_of_many_columns():
    n = 8_500_000
    print(f"case var gradient [{n}, 3, 16] over 1", flush=True)
    v = named(n)
    x = v[:, None, None].repeat(1, 3, 16)
    x[:, 0] += 3  # mean v + 1, deviations 2, -1, -1
    g = _capi.reduce_backward(v[:, None].expand(n, 16), x, "var", [1])
    assert torch.equal(g[:, 0], (v * 2)[:, None].expand(n, 16))
    assert torch.equal(g[:, 2], -v[:, None].expand(n, 16))


def test_sum_rows_off_16_bytes():
    n = 4_200_000  # 1025 floats a row, one element per thread
    print(f"case sum gradient [{n}, 1025]", flush=True)
    v = named(n)
    x = torch.empty(1, device="cuda").as_strided((n, 1025), (0, 0))
    g = _capi.reduce_backward(v, x, "sum", [1])
    for c in (0, 512, 1024):
        assert torch.equal(g[:, c], v)


def test_nll():
    n, c = 17_000_000, 1024
    print(f"case nll gradient [{n}, {c}]", flush=True)
    t = (torch.arange(n, device="cuda") * 7) % c
    g = _capi.nll_loss_backward(torch.full((1,), 2.0, device="cuda"), t, n, c, None, 2)
    assert bool((g.gather(1, t[:, None]) == -2).all())
    for a in range(0, n, 1 << 21):
        assert int(torch.count_nonzero(g[a:a + (1 << 21)])) == min(1 << 21, n - a)
