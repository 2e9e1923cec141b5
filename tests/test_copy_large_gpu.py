"""Copies that would take more threads than a launch counts (2^32; it runs the
rest modulo 2^32 and reports nothing): strided rows, dense data, many short rows,
many small transposes."""
import pytest

from tensorplay_amd import _capi

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def test_strided_rows_beyond_the_threads_of_a_launch():
    rows, n = (1 << 20) + 1, 65536  # rows * n / 16 stores: just above 2^32
    torch.cuda.empty_cache()
    print(f"case copy int8 [{rows}, {n}] from an expanded view of step 2", flush=True)
    base = torch.randint(-128, 128, (2 * n,), dtype=torch.int8, device="cuda")
    out = torch.empty((rows, n), dtype=torch.int8, device="cuda")
    out[-1].zero_()
    _capi.copy_(out, base[::2].expand(rows, n))
    want = base[::2]
    for r in (0, 1, 65535, 65536, rows // 2, rows - 2, rows - 1):
        assert torch.equal(out[r], want), r
    assert torch.equal(out[::4099, ::4096], want[::4096].expand(len(range(0, rows, 4099)), n // 4096))
    del out
    torch.cuda.empty_cache()


def test_dense_copy_beyond_the_threads_of_a_launch():
    n = (1 << 36) + 4099  # 64 GiB and a ragged end
    torch.cuda.empty_cache()
    print(f"case copy int8 dense n={n}", flush=True)
    x = torch.empty(n, dtype=torch.int8, device="cuda")
    x.random_(-128, 128)
    y = torch.zeros(n, dtype=torch.int8, device="cuda")
    _capi.copy_(y, x)
    for a in range(0, n, 1 << 33):
        assert torch.equal(x[a:a + (1 << 33)], y[a:a + (1 << 33)]), a
    del x, y
    torch.cuda.empty_cache()


@pytest.mark.parametrize("off", [0, 1])
def test_many_short_rows(off):
    rows, n = 17_000_000, 256  # one workgroup a row
    torch.cuda.empty_cache()
    print(f"case copy int8 rows [{rows}, {n}] of 300, offset {off}", flush=True)
    x = torch.empty(rows * 300 + 1, dtype=torch.int8, device="cuda")
    x.random_(-128, 128)
    v = x[off:off + rows * 300].view(rows, 300)[:, :n]
    y = torch.zeros((rows, n), dtype=torch.int8, device="cuda")
    _capi.copy_(y, v)
    assert torch.equal(y, v)
    del x, y, v
    torch.cuda.empty_cache()


def test_many_small_transposes():
    b = 16_900_000  # one tile each: more than 2^24 workgroups
    torch.cuda.empty_cache()
    print(f"case copy int8 [{b}, 16, 16] transposed", flush=True)
    x = torch.empty((b, 16, 16), dtype=torch.int8, device="cuda")
    x.random_(-128, 128)
    y = torch.zeros((b, 16, 16), dtype=torch.int8, device="cuda")
    _capi.copy_(y, x.transpose(1, 2))
    assert torch.equal(y.transpose(1, 2), x)
    del x, y
    torch.cuda.empty_cache()
