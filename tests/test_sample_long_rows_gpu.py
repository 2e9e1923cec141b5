"""Draws from one row of 2^31 - 1 logits: the kernel's steps past the row's end
pass 2^31.  Two likely tokens, the last and an early one, over a flat rest that
weighs nothing beside them, so no host copy is needed."""
import pytest

from tensorplay_amd import _capi

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

N = (1 << 31) - 1


def test_two_tokens():
    x = torch.full((1, N), -30.0, device="cuda")
    x[0, N - 1], x[0, 3] = 10.0, 9.5
    # weights 1 and exp(-0.5) = 0.607: the nucleus of 0.9 holds both
    for k, temperature, top_p, u, want in [(1500, 0.0, 1.0, 0.5, N - 1), (N, 1.0, 0.9, 0.1, N - 1),
                                           (N, 1.0, 0.9, 0.99, 3), (N, 1.0, 1.0, 0.99, 3), (1500, 1.0, 0.9, 0.99, 3)]:
        print(f"case sample [1, {N}] k={k} T={temperature} top_p={top_p} u={u}", flush=True)
        assert int(_capi.sample(x, torch.tensor([u], device="cuda"), k, temperature, top_p)[0]) == want
    del x
    torch.cuda.empty_cache()
