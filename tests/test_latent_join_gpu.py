"""The join of latent attention's partitions against 64 bits, from partials that hold NaN wherever no partition is."""
import pytest
import torch

from rag_llm_k8s_amd.ops.backend import AttnMeta
from rag_llm_k8s_amd.ops.specs import LatentSpec

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("S", [1, 3, 12])  # gate slabs: fewer and more than are asked for together
@pytest.mark.parametrize("rank", [100, 256, 384, 512, 640, 1000])  # one to eight threads of a column for one sequence
@pytest.mark.parametrize("B,max_kv", [(1, 8192), (1, 100), (2, 8192), (3, 1500), (9, 2500), (40, 700), (53, 700)])
def test_join(native, B, max_kv, rank, S):
    from rag_llm_k8s_amd.ops import seq_native as Q

    s = LatentSpec(heads=20, dim=64, vdim=64, rank=rank, scale=0.1)
    s.own = False
    g = torch.Generator(device=DEV).manual_seed(B + rank)
    parts, tt, mt = Q.latent_parts(s, max_kv, B), Q.latent_tile(s), Q.latent_min_tiles(s)
    lens = [max(1, max_kv - (i * 997) % max_kv) for i in range(B)]
    ws_o = torch.full((B, s.heads, parts, s.rp), float("nan"), device=DEV)
    ws_ml = torch.full((B, s.heads, parts, 2), float("nan"), device=DEV)
    c = torch.zeros(B, s.heads, s.rp, dtype=torch.float64, device=DEV)
    for b, L in enumerate(lens):
        tiles = (L - 1) // tt + 1
        n = -(-tiles // max(mt, -(-tiles // parts)))
        o = torch.randn(s.heads, n, s.rp, device=DEV, generator=g)
        m, l = 9 * torch.randn(s.heads, n, device=DEV, generator=g), 1 + torch.rand(s.heads, n, device=DEV, generator=g)
        ws_o[b, :, :n], ws_ml[b, :, :n, 0], ws_ml[b, :, :n, 1] = o, m, l
        w = torch.exp2(m.double() - m.double().max(1, keepdim=True).values)
        c[b] = (o.double() * w[..., None]).sum(1) / (l.double() * w).sum(1)[:, None]
    P = torch.randn(S, B, s.row, device=DEV, generator=g)
    wuv = (torch.randn(s.heads, s.dvp, s.rp, device=DEV, generator=g) * s.rp ** -0.5).bfloat16()
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    meta = AttnMeta("decode", i32(lens), i32([[0] * 128] * B), max_kv=max_kv)
    out = torch.full((B, s.out_row), 7.0, device=DEV).bfloat16()
    Q.latent_out(P, s, wuv, meta, out, (ws_o, ws_ml))
    gate = torch.sigmoid(P.double().sum(0)[:, s.off_g:s.off_g + s.heads * s.dvp].view(B, s.heads, s.dvp))
    want = torch.einsum("bhr,hdr->bhd", c, wuv.double()) * gate
    # the joined latents and the result are rounded to bf16 (2^-8 of a value at most); the join and the gate are fp32
    lim = 2.0 ** -8 * (torch.einsum("bhr,hdr->bhd", c.abs(), wuv.double().abs()) * gate + want.abs()) + 1e-5
    assert bool(((out[:, :s.heads * s.dvp].view(B, s.heads, s.dvp).double() - want).abs() <= lim).all())
