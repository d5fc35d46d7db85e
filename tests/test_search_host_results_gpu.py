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


def test_searches_allocate_no_host_memory(native):
    """The first search of an index as every later one, of whatever size: the index has put a block into the pool."""
    from rag_llm_k8s_amd.index.flat import FlatL2Index
    from rag_llm_k8s_amd.index.ivf import IVFFlatIndex

    g = torch.Generator(device=DEV).manual_seed(1)
    x = torch.randn(4000, 64, device=DEV, generator=g)
    flat, ivf = FlatL2Index(64, device=DEV, capacity=4000), IVFFlatIndex(64, device=DEV, nlist=16, nprobe=4)
    flat.add(x)
    ivf.train(x)
    ivf.add(x)
    made = torch.cuda.host_memory_stats()["num_host_alloc"]
    for nq, k in ((1, 1), (1, 10), (3, 64), (100, 7), (1000, 10), (2048, 8)):
        for index in (flat, ivf):
            index.search(x[:nq], k)
    assert torch.cuda.host_memory_stats()["num_host_alloc"] == made
