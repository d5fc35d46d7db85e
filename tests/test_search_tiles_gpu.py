"""Exact search at the edges of its row tiles, query groups and dimension chunks."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("d", [32, 100, 384, 1024])
@pytest.mark.parametrize("n,begin,cap", [(7, 0, 7), (15, 0, 15), (65, 3, 66), (1025, 17, 1031), (16387, 3, 16390),
                                         (49153, 1, 49153), (70001, 5, 70001),
                                         (200003, 17, 200004)])
def test_search_tiles(native, n, begin, cap, d):
    """Stores of less than a tile, tiles cut by the end of the store or begun at an odd row; queries on both sides of every
    padded count and of the change of form; lists longer than the store."""
    g = torch.Generator(device=DEV).manual_seed(n + d)
    xt = torch.randn(d, cap, device=DEV, generator=g)
    qs = torch.randn(33, d, device=DEV, generator=g)
    x64 = xt[:, begin:n].t().double()
    exact = torch.cat([((x64 - q.double()) ** 2).sum(1)[None] for q in qs])
    # d roundings of each of the three sums that the batched form adds, each within ||x||^2 + ||q||^2 <= 2 (d + 6 sqrt(2 d))
    # at these draws; the direct form is within that too
    tol = 3 * d * 2.0 ** -24 * 2 * (d + 6 * (2 * d) ** 0.5)
    for nq, k in ((1, 1), (2, 10), (3, 5), (5, 8), (9, 10), (15, 5), (16, 8), (17, 1), (32, 10), (33, 5)):
        D, I = native.l2_search(xt, cap, n, qs[:nq], k, row_begin=begin)
        kk = min(k, n - begin)
        best = exact[:nq].topk(kk, dim=1, largest=False).values
        assert I[:, kk:].eq(-1).all() and D[:, kk:].eq(torch.finfo(torch.float32).max).all()
        D, I = D[:, :kk].double(), I[:, :kk]
        assert I.ge(begin).all() and I.lt(n).all() and all(len(set(r)) == kk for r in I.tolist())
        assert (D - exact[:nq].gather(1, I - begin)).abs().max().item() <= tol  # the distance of the row it names
        assert (D - best).abs().max().item() <= tol  # and no nearer row left out
        assert D.diff(dim=1).ge(0).all()
