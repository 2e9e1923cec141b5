"""Draws in which one token outweighs millions of equal ones whose weights only
count together: the position must be the definition's, from float64 sums.  The
float32 exponential may be off by 2^-22, which moves the position by as much of
the 2^23 tokens it lies among; 8 positions are allowed."""
import math

import pytest

from tensorplay_amd import _capi

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def expected(n, k, logit, temperature, top_p, u):
    """Rank drawn: c_0 = 1 and c_j = 1 + j w for the k - 1 equal ones."""
    w = math.exp(logit / temperature)
    total = 1.0 + (k - 1) * w
    m = min(k - 1, max(0, math.ceil((top_p * total - 1.0) / w)))
    cm = 1.0 + m * w
    return min(m, max(0, math.floor((u * cm - 1.0) / w) + 1))


@pytest.mark.parametrize("bits,exponent", [(22, 37), (24, 39)])
@pytest.mark.parametrize("less", [0, 5])
@pytest.mark.parametrize("top_p", [1.0, 1 - 2.0 ** -17])
def test_many_small_weights(bits, exponent, less, top_p):
    n, head, temperature, u = 1 << bits, 12345, 0.75, 1 - 2.0 ** -16
    logit = float(torch.tensor(-exponent * math.log(2.0) * temperature, dtype=torch.float32))
    print(f"case sample [1, 2^{bits}] weights 2^-{exponent} k=cols-{less} top_p={top_p}", flush=True)
    x = torch.full((1, n), logit, device="cuda")
    x[0, head] = 0.0
    got = int(_capi.sample(x, torch.tensor([u], device="cuda"), n - less, temperature, top_p)[0])
    rank = 0 if got == head else got + 1 if got < head else got
    want = expected(n, n - less, logit, temperature, top_p, u)
    assert want > n // 8 and abs(rank - want) <= 8, (rank, want)
