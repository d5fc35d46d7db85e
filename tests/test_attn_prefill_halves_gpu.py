"""Prompts' attention in 32-query blocks (few blocks) and 64-query blocks (many) gives the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def run(native, q, kc, vc, bt, lens, ctx, Hq, Hkv):
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32).to(DEV)
    kl = torch.tensor([a + b for a, b in zip(lens, ctx)], dtype=torch.int32).to(DEV)
    out = torch.full((sum(lens) + 1, Hq * 128), -3.0, device=DEV).bfloat16()
    native.attn_prefill(q, kc, vc, cu, kl, native.build_prefill_tiles(lens, Hq, Hkv).to(DEV), out, Hq, Hkv, 128, block_tables=bt)
    assert bool((out[-1] == -3.0).all())
    return out[:-1]


# rows short of a half tile, a whole half, one past it, short of and past a tile; contexts before the queries, short ones and such
# that the ring of four key tiles goes round several times and ends in each of its slots; 8 and 4 KV heads
@pytest.mark.parametrize("Hq,Hkv", [(32, 8), (16, 4)])
@pytest.mark.parametrize("rows,ctx", [(1, 0), (31, 0), (32, 65), (33, 0), (63, 3), (64, 0), (65, 130), (97, 0), (300, 0), (200, 77),
                                      (700, 0), (33, 509), (65, 640), (40, 1000), (40, 1064), (40, 1128), (40, 1192)])
def test_few_blocks_are_many(native, Hq, Hkv, rows, ctx):
    g = torch.Generator(device=DEV).manual_seed(rows + ctx)
    pages = -(-(rows + ctx) // 64)
    copies = 128 // (-(-rows // 64) * Hkv) + 1  # together past the line
    kc, vc = (torch.randn(copies * pages, Hkv, 64, 128, device=DEV, generator=g).bfloat16() for _ in range(2))
    bt = torch.randperm(copies * pages, generator=g, device=DEV).int().view(copies, pages)
    q = torch.randn(copies * rows, (Hq + 2 * Hkv) * 128, device=DEV, generator=g).bfloat16()
    many = run(native, q, kc, vc, bt, [rows] * copies, [ctx] * copies, Hq, Hkv)
    for i in (0, copies - 1):
        few = run(native, q[i * rows:(i + 1) * rows], kc, vc, bt[i:i + 1], [rows], [ctx], Hq, Hkv)
        assert torch.equal(few, many[i * rows:(i + 1) * rows])
