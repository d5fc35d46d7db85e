"""Results that the merge stores into host memory: the device's, in memory of the caller's own."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("nq,k", [(1, 1), (1, 64), (3, 7), (16384, 1), (16385, 1), (1639, 10)])
def test_host_results_are_the_devices(native, nq, k):
    g = torch.Generator(device=DEV).manual_seed(nq + k)
    xt, q = torch.randn(32, 512, device=DEV, generator=g), torch.randn(nq, 32, device=DEV, generator=g)
    d, i = native.l2_search(xt, 512, 300, q, k)
    dist, ids = native.l2_search(xt, 512, 300, q, k, host=True)
    keep = dist.clone(), ids.clone()
    assert not dist.is_cuda and not dist.is_pinned() and torch.equal(dist, d.cpu()) and torch.equal(ids, i.cpu())
    native.l2_search(xt, 512, 300, -q, k, host=True)
    assert torch.equal(dist, keep[0]) and torch.equal(ids, keep[1])
