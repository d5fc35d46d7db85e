"""Products cut into two plans by columns: where the rule cuts (CPU), and that every epilogue's operands follow the cut (GPU)."""
import random

import pytest
import torch

from rag_llm_k8s_amd.ops import native as n
from rag_llm_k8s_amd.ops import reference as R


def test_rule():
    cut = n.gemm_columns(1777, 28672, 4096, 256)  # three rounds of 256 x 256 tiles and 16 more of them
    assert cut and cut % 256 == 0
    assert n.gemm_columns(1777, 28672, 128, 256) == 0  # three K-tiles at least
    assert n.gemm_columns(2048, 8192, 4096, 256) == 0  # one round exactly
    for M in (65, 300, 529, 1129, 1777, 2813, 4072, 7917, 14076):
        for rows, K in ((28672, 4096), (11264, 2048), (8512, 2048), (6144, 4096), (3072, 1024)):
            c = n.gemm_columns(M, rows, K, 256)
            assert c % 256 == 0 and 0 <= c < rows
            if c:
                whole, a, b = (n._timed_plan(M, r, K, True, 256, s)[0] for r, s in ((rows, True), (c, False), (rows - c, False)))
                assert a + b < n.COLUMNS_GAIN * whole


def test_a_cut_splits_no_sum():
    """Every launch of a cut product, and every launch that it would have without the cut, sums over K in one piece."""
    r = random.Random(4)
    cuts = 0
    for _ in range(3000):
        M, (rows, K) = int(2 ** r.uniform(6.05, 14)), r.choice(((28672, 4096), (6144, 4096), (16704, 4096), (11264, 2048), (8512, 2048)))
        c = n.gemm_columns(M, rows, K, 256)
        plans = [n.gemm_plan(M, rows, K, True, 256)]
        if c:
            cuts += 1
            plans += [n.gemm_plan(M, m, K, True, 256, False) for m in (c, rows - c)]
            assert all(S == 1 for p in plans for _, _, _, S in p), (M, rows, K, c)
    assert cuts > 20


def test_operands_of_a_cut():
    """Every piece's operands begin at its columns and hold them all, a bias of shape [N], [1, N] or [N, 1] alike."""
    M, N, K = 3, 768, 64
    w, r, out = torch.zeros(N, K).bfloat16(), torch.zeros(M, N + 8).bfloat16()[:, :N], torch.zeros(M, N)
    for shape in ((N,), (1, N), (N, 1)):
        b = torch.arange(N).bfloat16().view(shape)
        for c0, c1 in ((0, 512), (512, N)):
            wc, bc, rc, oc = n._columns(w, b, r, out, "bias_resid", c0, c1)
            for part, whole, at in ((wc, w, c0 * K), (bc, b, c0), (rc, r, c0), (oc, out, c0)):
                assert part.data_ptr() == whole.data_ptr() + at * whole.element_size()
            assert wc.shape == (c1 - c0, K) and bc.numel() == c1 - c0 and rc.shape == oc.shape == (M, c1 - c0)
    par, row = torch.zeros(3), torch.zeros(5)  # (not read as a bias; not read at all)
    wc, bc, rc, oc = n._columns(w, par, row, out[:, :N // 2], "glu_clip", 512, N)
    assert bc is par and rc is row and wc.shape[0] == 256 and oc.shape == (M, 128)
    assert oc.data_ptr() == out.data_ptr() + 256 * 4


# cut at 9216 of 11264 columns; at 4352 of 6144 (once at 5888, with the last two heads' sums split); not cut
@pytest.mark.gpu
@pytest.mark.parametrize("M,Hq,Hkv,K", [(1297, 72, 8, 2048), (2692, 32, 8, 4096), (1500, 32, 8, 4096)])
def test_rotated_projection_agrees_with_a_cut_product(native, M, Hq, Hkv, K):
    """gemm_rope_kv, whose launches are not cut, is gemm followed by rope_kv bit for bit, cached rows included."""
    N, g = (Hq + 2 * Hkv) * 128, torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn(M, K, device="cuda", generator=g).bfloat16()
    w = (torch.randn(N, K, device="cuda", generator=g) * K ** -0.5).bfloat16()
    cos, sin = (t.cuda() for t in R.rope_tables(128, 4096))
    pos = torch.arange(M, device="cuda").int()
    slots = torch.randperm((M // 64 + 2) * 64, device="cuda", generator=g)[:M].int()
    kc, vc, kc2, vc2 = torch.zeros(4, M // 64 + 2, Hkv, 64, 128, device="cuda").bfloat16()
    assert (native.gemm_columns(M, N, K, 256) > 0) == (M != 1500)
    got, ref = native.gemm_rope_kv(x, w, pos, cos, sin, slots, kc, vc, Hq, Hkv, 128), native.gemm(x, w)
    native.rope_kv(ref, pos, cos, sin, slots, kc2, vc2, Hq, Hkv, 128)
    assert torch.equal(got, ref) and torch.equal(kc, kc2) and torch.equal(vc, vc2)


@pytest.mark.gpu
@pytest.mark.parametrize("M,rows,cut", [(65, 320, 256), (200, 1152, 512), (257, 1024, 768)])
@pytest.mark.parametrize("epi", ["none", "bias", "resid", "bias_resid", "bias_gelu", "silu_mul", "glu_clip"])
def test_operands_follow_the_cut(native, monkeypatch, M, rows, cut, epi):
    K = 256
    g = torch.Generator().manual_seed(M)
    pair = epi in native.PAIR_EPI
    if pair:
        rows = -(-rows // 128) * 128
        N = rows // 2
    else:
        N = rows
    rand = lambda *s: torch.randn(*s, generator=g).cuda()  # noqa: E731
    x, w = rand(M, K).bfloat16(), (rand(rows, K) * K ** -0.5).bfloat16()
    bias = rand(N).bfloat16() if "bias" in epi else None
    if epi == "glu_clip":
        bias = torch.tensor([7.0, 1.7, 1.0], device="cuda")
    res = rand(M, N).bfloat16() if "resid" in epi else None
    for f32 in ((False,) if pair else (False, True)):
        outs = []
        for c in (cut, 0):
            monkeypatch.setattr(native, "gemm_columns", lambda *a, c=c: c)
            wide = torch.full((M, N + 64), 3.0, device="cuda", dtype=torch.float32 if f32 else torch.bfloat16)
            out = wide[:, :N]
            if res is not None and not f32:
                out.copy_(res)  # in place, as the residual stream is
            native.gemm(x, w, bias=bias, resid=out if res is not None and not f32 else res, epi=epi, out=out, out_f32=f32)
            assert bool((wide[:, N:] == 3.0).all())
            outs.append(out.double())
        # fp32 sums of 256 products in another order (a K-split may differ): 2^-16 of the values' size, and half a bf16 unit of
        # either side where the result is rounded (2^-8 each)
        d = (outs[0] - outs[1]).abs()
        assert bool((d <= (2.0 ** -16 if f32 else 2.0 ** -7) * outs[1].abs() + 2.0 ** -15).all()), (epi, f32, float(d.max()))
