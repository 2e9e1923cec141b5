"""Softmax over more rows or columns than the threads of one launch allow (2^32;
a larger launch runs the rest modulo 2^32 and reports nothing).  Pairs (0, v):
their softmax is a sigmoid, their gradient a product, and v names the row."""
import pytest

from tensorplay_amd import _capi

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(autouse=True)
def _free():
    torch.cuda.empty_cache()
    yield
    torch.cuda.empty_cache()


def named(n, dtype):
    return (torch.arange(n, device="cuda", dtype=torch.int32) % 97).to(dtype) / 16 - 3


def close(got, want, eps):
    return bool(((got - want).abs_() <= eps * want.abs()).all())


@pytest.mark.parametrize("dtype,n,eps", [(torch.float32, 270_000_000, 1e-5), (torch.float64, 17_000_000, 1e-12)])
def test_rows(dtype, n, eps):
    print(f"case softmax rows [{n}, 2] {dtype}", flush=True)
    v = named(n, dtype)
    x = torch.stack([torch.zeros_like(v), v], 1)
    s = torch.sigmoid(v)
    y = _capi.softmax(x, 1)
    assert close(y[:, 1], s, eps) and close(y[:, 0], 1 - s, eps)
    # g = (0, 1): (g - sum(g y)) y
    g = torch.zeros_like(x)
    g[:, 1] = 1
    x = _capi.softmax(g, 1, grad_of=y)
    assert close(x[:, 1], s * (1 - s), eps) and close(x[:, 0], -s * (1 - s), eps)


@pytest.mark.parametrize("outer,inner", [(68_000_000, 16), (360_000_000, 3)])
def test_columns(outer, inner):
    print(f"case softmax columns [{outer}, 2, {inner}]", flush=True)
    v = named(outer, torch.float32)
    x = torch.zeros((outer, 2, inner), device="cuda")
    x[:, 1, :] = v[:, None]
    y = _capi.softmax(x, 1)
    del x
    s = torch.sigmoid(v)
    for c in (0, inner // 2, inner - 1):
        assert close(y[:, 1, c], s, 1e-5) and close(y[:, 0, c], 1 - s, 1e-5)
