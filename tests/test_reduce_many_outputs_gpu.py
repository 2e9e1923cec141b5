"""Reductions with more outputs than the threads of one launch allow (2^32
threads; a larger launch silently ran the rest modulo 2^32): every layout, with
values that name their output, built on the device."""
import pytest

from tensorplay_amd import _capi

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(autouse=True)
def _free():
    torch.cuda.empty_cache()
    yield
    torch.cuda.empty_cache()


def named(n, dtype=torch.int8):
    """0 .. 96, again and again (a prime period, so that no power of two repeats it)."""
    return (torch.arange(n, device="cuda", dtype=torch.int32) % 97).to(dtype)


def test_short_rows():
    n = 300_000_000
    print(f"case int8 rows [{n}, 4]", flush=True)
    v = named(n)
    x = v[:, None].repeat(1, 4)
    x[:, 2] += 1
    assert torch.equal(_capi.reduce(x, "argmax", [1]), torch.full((n,), 2, device="cuda"))
    assert torch.equal(_capi.reduce(x, "sum", [1]), v.long() * 4 + 1)


def test_float_rows():
    n = 280_000_000
    print(f"case float32 rows [{n}, 5]", flush=True)
    v = named(n, torch.float32)
    x = v[:, None].repeat(1, 5)
    assert torch.equal(_capi.reduce(x, "sum", [1]), v * 5)


def test_register_rows():
    n = 68_000_000  # rows of 257..512 floats take a wave each; an expanded view, so the input is small
    base = torch.arange(600, dtype=torch.float32, device="cuda").view(2, 300)
    x = base.as_strided((2, n // 2, 300), (300, 0, 1))
    print(f"case float32 register rows {list(x.shape)} {list(x.stride())}", flush=True)
    want = base.sum(1)
    y = base[0].as_strided((n, 300), (0, 1))
    assert bool((_capi.reduce(y, "sum", [1]) == want[0]).all())
    got = _capi.reduce(x, "sum", [2])
    assert bool((got == want[:, None]).all())


def test_columns():
    n = 20_000_000
    print(f"case float32 [{n}, 10, 3] over 1", flush=True)
    v = named(n, torch.float32)
    x = v[:, None, None].repeat(1, 10, 3)
    x[:, :, 1] += 1
    got = _capi.reduce(x, "sum", [1])
    assert torch.equal(got, torch.stack([v * 10, v * 10 + 10, v * 10], 1))


def test_few_columns():
    n = 17_000_000
    print(f"case int8 [{n}, 64, 2] over 1", flush=True)
    v = named(n)
    x = v[:, None, None].repeat(1, 64, 2)
    x[:, :, 1] += 1
    got = _capi.reduce(x, "sum", [1])
    assert torch.equal(got, torch.stack([v.long() * 64, v.long() * 64 + 64], 1))


@pytest.mark.parametrize("lead", [1, 3])
def test_general(lead):
    n = 18_000_000 // lead
    print(f"case int8 strided [{lead}, {n}, 2]", flush=True)
    v = named(lead * n)
    buf = v[:, None].repeat(1, 8)
    x = buf.view(lead, n, 8)[:, 1:, ::4]  # kept dims that do not merge, stride 4 inside
    got = _capi.reduce(x, "sum", [2])
    assert torch.equal(got, v.view(lead, n)[:, 1:].long() * 2)


def test_runs():
    g = torch.Generator().manual_seed(3)
    base = torch.randint(-100, 100, (3, 4200), generator=g, dtype=torch.int8)
    m = 2_800_000  # 8.4 M outputs of 2100 elements, 512 threads each
    x = base.cuda().as_strided((3, m, 2100), (4200, 0, 1))
    print(f"case int8 runs {list(x.shape)} {list(x.stride())}", flush=True)
    got = _capi.reduce(x, "sum", [2])
    want = base[:, :2100].sum(1, dtype=torch.int64).cuda()
    assert torch.equal(got, want[:, None].expand(3, m))
