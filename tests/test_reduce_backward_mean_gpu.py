"""Gradient of mean over a contiguous innermost run of 1024 elements or more: each
element is float32(g / count) with the division in float64, bit for bit, for one
and several rows per workgroup, rows cut in chunks and the two layouts beside it."""
import pytest

from tensorplay_amd import _capi

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("shape,dims", [((5, 1024), (1,)), ((3, 1027), (1,)), ((7, 2048), (1,)), ((2, 3, 4100), (0, 2)),
                                        ((4, 3, 10001), (0, 2)), ((1, 70000), (1,)), ((8, 16, 56, 56), (0, 2, 3)),
                                        ((3, 5, 1023), (2,)), ((4, 6, 2048), (1,))])
def test_mean_gradient(shape, dims):
    print(f"case mean gradient {shape} {dims}", flush=True)
    x = torch.zeros(shape, device="cuda")
    kept = [s for i, s in enumerate(shape) if i not in dims]
    g = torch.randn(kept, generator=torch.Generator().manual_seed(1)).cuda()
    count = x.numel() // max(1, g.numel())
    got = _capi.reduce_backward(g, x, "mean", list(dims))
    q = (g.double() / count).float()
    for d in sorted(dims):
        q = q.unsqueeze(d)
    assert torch.equal(got, q.expand(shape))
