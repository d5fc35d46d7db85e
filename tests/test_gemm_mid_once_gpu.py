"""Large weights under one row of tiles, streamed past the caches: the bits of the same rows under more tiles."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("epi,rows,K", [("silu_mul", 16384, 2048), ("glu_clip", 16384, 2048), ("none", 16392, 2048)])
@pytest.mark.parametrize("mi", [3, 5, 8, 21])
def test_one_row_of_tiles(native, epi, rows, K, mi):
    """One tile's rows (the streaming policy) against a tile and three rows: a K order of its own is what no tile has."""
    g = torch.Generator(device=DEV).manual_seed(mi)
    top = 160 if mi == 21 else 32 * mi
    x = torch.randn(top + 3, K, device=DEV, generator=g).bfloat16()
    w = (torch.randn(rows, K, device=DEV, generator=g) * K ** -0.5).bfloat16()
    b = torch.tensor([1.0, 1.7, 1.0], device=DEV) if epi == "glu_clip" else None
    N = rows if epi == "none" else rows // 2
    both = torch.empty(top + 3, N, device=DEV, dtype=torch.bfloat16)
    native.gemm_mid(x, w, bias=b, epi=epi, out=both, mi=mi)
    for M in (1, 17, top):
        out = torch.full((M + 1, N), 7.0, device=DEV).bfloat16()
        native.gemm_mid(x[:M], w, bias=b, epi=epi, out=out[:M], mi=mi)
        assert torch.equal(out[:M], both[:M]) and bool((out[M] == 7).all())
