"""Top-k of rows of almost 2^31 elements: the last segment of the wave kernel,
which would end at 2^31, and the streaming kernel on both sides of its loads in
flight.  Rows of zeros with a few placed values, so no host copy is needed."""
import pytest

from tensorplay_amd import _capi

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

LONGEST = (1 << 31) - 1 - (1 << 20)


@pytest.mark.parametrize("n,k", [(LONGEST, 5), (LONGEST, 2000), (LONGEST + 1, 5), ((1 << 31) - 1, 5),
                                 ((1 << 31) - 1, 2000), ((1 << 31) - 5000, 300)])
def test_int8(n, k):
    print(f"case topk int8 [1, {n}] k={k}", flush=True)
    x = torch.zeros((1, n), dtype=torch.int8, device="cuda")
    at = [n - 1, 3, n - 2, n // 2, n - 9000]
    for j, e in enumerate(at):
        x[0, e] = 100 - j
    v, i = _capi.topk(x, k)
    assert v[0, :5].tolist() == [100, 99, 98, 97, 96] and i[0, :5].tolist() == at
    if k > 5:  # zeros, lowest index first
        rest = [e for e in range(k) if e != 3][:k - 5]
        assert int(v[0, 5:].abs().max()) == 0 and i[0, 5:].tolist() == rest
    v, i = _capi.topk(x, 2, largest=False)
    assert v[0].tolist() == [0, 0] and i[0].tolist() == [0, 1]
    del x
    torch.cuda.empty_cache()
