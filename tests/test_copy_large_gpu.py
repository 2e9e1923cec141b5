"""A copy into more than 64 GiB of long rows from a stepped, expanded source:
one 16-byte store per thread would take more threads than a launch counts."""
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
