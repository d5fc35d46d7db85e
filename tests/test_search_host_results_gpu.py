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


def test_results_later_than_the_watch(native):
    """A stream that is busy for longer than results are watched for: the stream is waited for instead."""
    g = torch.Generator(device=DEV).manual_seed(2)
    xt, q = torch.randn(32, 512, device=DEV, generator=g), torch.randn(5, 32, device=DEV, generator=g)
    want = native.l2_search(xt, 512, 500, q, 3)
    torch.cuda._sleep(60_000_000)  # some 25 ms
    dist, ids = native.l2_search(xt, 512, 500, q, 3, host=True)
    assert torch.equal(dist, want[0].cpu()) and torch.equal(ids, want[1].cpu())


def test_searches_beside_each_other(native):
    """Threads with streams of their own, and two on one stream: each gets its own query's results."""
    from concurrent.futures import ThreadPoolExecutor

    g = torch.Generator(device=DEV).manual_seed(3)
    xt, q = torch.randn(32, 4096, device=DEV, generator=g), torch.randn(64, 32, device=DEV, generator=g)
    want = [[t.cpu() for t in native.l2_search(xt, 4096, 4000, q[j:j + 1], 4)] for j in range(64)]
    streams = [torch.cuda.Stream() for _ in range(3)]
    torch.cuda.synchronize()

    def run(t):
        with torch.cuda.stream(streams[t % 3]):
            for j in range(t, 64, 4):
                dist, ids = native.l2_search(xt, 4096, 4000, q[j:j + 1], 4, host=True)
                if not (torch.equal(dist, want[j][0]) and torch.equal(ids, want[j][1])):
                    return j
        return None

    with ThreadPoolExecutor(4) as ex:
        assert list(ex.map(run, range(4))) == [None] * 4


def test_host_results_are_refused_under_capture(native):
    xt, q = torch.randn(32, 512, device=DEV), torch.randn(1, 32, device=DEV)
    native.l2_search(xt, 512, 500, q, 3, host=True)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        native.l2_search(xt, 512, 500, q, 3, host=True)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            with pytest.raises(RuntimeError):
                native.l2_search(xt, 512, 500, q, 3, host=True)
            got = native.l2_search(xt, 512, 500, q, 3)
        graph.replay()
        want = native.l2_search(xt, 512, 500, q, 3)
    s.synchronize()
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
