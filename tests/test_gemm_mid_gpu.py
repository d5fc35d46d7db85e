"""gemm_mid.hip (ring tiles of 96 to 256 x 128, K-split) against fp32 products and gemm_w4, at the edges of its tiles."""
import math

import pytest
import torch

from rag_llm_k8s_amd.ops import reference as R

pytestmark = pytest.mark.gpu
DEV = "cuda"


def rel_err(a, b):
    a, b = a.float().cpu(), b.float().cpu()
    return ((a - b).norm() / (b.norm() + 1e-12)).item()


def operands(M, N, K):
    torch.manual_seed(M + N + K)
    x = torch.randn(M, K, device=DEV).bfloat16()
    w = (torch.randn(N, K, device=DEV) / math.sqrt(K)).bfloat16()
    return x, w, torch.randn(N, device=DEV).bfloat16(), torch.randn(M, N, device=DEV).bfloat16()


# tile edges in rows (mi x 32), columns past the last 128-wide tile, rings of fewer K-tiles than slots, uneven K-slabs,
# more work items than CUs
@pytest.mark.parametrize("mi,S,M,N,K", [(3, 1, 65, 128, 128), (3, 3, 97, 136, 640), (4, 1, 128, 264, 256), (5, 2, 161, 256, 192),
                                         (6, 5, 193, 128, 704), (8, 1, 257, 1032, 512), (8, 4, 513, 512, 256),
                                         (4, 1, 2500, 2048, 384), (3, 7, 700, 1024, 448)])
def test_gemm_mid(native, mi, S, M, N, K):
    x, w, b, r = operands(M, N, K)
    ref = x.float() @ w.float().t()
    y = native.gemm_mid(x, w, out=torch.empty_like(r), mi=mi, S=S)
    assert rel_err(y, ref) < 4e-3  # bf16 result: 2^-9 per value
    if S == 1 and K >= 192 and K % 128 == 0:
        assert torch.equal(y, native.gemm(x, w, path=6))  # one K order in both kernels
    for epi in ("bias", "resid", "bias_resid", "bias_gelu", "gelu", "bias_gelu_tanh"):
        y = native.gemm_mid(x, w, bias=b, resid=r, epi=epi, out=torch.empty_like(r), mi=mi, S=S)
        assert rel_err(y, R.linear(x, w, b, r, epi=epi)) < 4e-3, epi
    h = r.clone()
    native.gemm_mid(x, w, resid=h, epi="resid", out=h, mi=mi, S=S)  # in place
    assert torch.equal(h, native.gemm_mid(x, w, resid=r, epi="resid", out=torch.empty_like(r), mi=mi, S=S))
    f = native.gemm_mid(x, w, out=torch.empty(M, N, device=DEV), out_f32=True, mi=mi, S=S)
    assert rel_err(f, ref) < 1e-5
    if N % 256 == 0:
        wp = R.pack_gate_up(w[:N // 2], w[N // 2:])
        out = torch.empty(M, N // 2, device=DEV).bfloat16()
        assert rel_err(native.gemm_mid(x, wp, epi="silu_mul", out=out, mi=mi, S=S), R.linear(x, wp, epi="silu_mul")) < 4e-3
        par = torch.tensor([2.0, 1.702, 1.0, 0.0], device=DEV)
        g, u = ref[:, :N // 2].clamp(max=2), ref[:, N // 2:].clamp(-2, 2)
        native.gemm_mid(x, wp, bias=par, epi="glu_clip", out=out, mi=mi, S=S)
        assert rel_err(out, g * torch.sigmoid(1.702 * g) * (u + 1)) < 4e-3


def test_gemm_mid_strided_rows_stay_in_place(native):
    """Rows of a wider buffer in and out: nothing outside the output columns is written."""
    x, w, _, _ = operands(300, 264, 256)
    xs = torch.full((300, 512), 7.0, device=DEV).bfloat16()
    xs[:, 128:384] = x
    for S in (1, 2):
        buf = torch.full((304, 400), -3.0, device=DEV).bfloat16()
        native.gemm_mid(xs[:, 128:384], w, out=buf[2:302, 64:328], mi=5, S=S)
        assert rel_err(buf[2:302, 64:328], x.float() @ w.float().t()) < 4e-3
        buf[2:302, 64:328] = -3.0
        assert bool((buf == -3.0).all())


@pytest.mark.parametrize("M,Hq,Hkv", [(65, 4, 2), (90, 16, 4), (300, 32, 8), (1023, 4, 2)])
def test_gemm_rope_kv_few_rows(native, M, Hq, Hkv):
    """The rotated projection below 1024 rows, whole and K-split, is gemm followed by rope_kv bit for bit."""
    D, K = 128, 2048
    N = (Hq + 2 * Hkv) * D
    x, w, _, _ = operands(M, N, K)
    cos, sin = (t.to(DEV) for t in R.rope_tables(D, 2048))
    pos = torch.randint(0, 2048, (M,), device=DEV).int()
    slots = torch.randperm((M // 64 + 2) * 64, device=DEV)[:M].int()
    slots[::5] = -1
    kc = torch.zeros(M // 64 + 2, Hkv, 64, D, device=DEV).bfloat16()
    vc, kc2, vc2 = torch.zeros_like(kc), torch.zeros_like(kc), torch.zeros_like(kc)
    assert native.gemm_rope_kv_ok(x, w, pos, cos, sin, slots, kc, vc, Hq, Hkv, D)
    got = native.gemm_rope_kv(x, w, pos, cos, sin, slots, kc, vc, Hq, Hkv, D)
    ref = native.gemm(x, w)
    native.rope_kv(ref, pos, cos, sin, slots, kc2, vc2, Hq, Hkv, D)
    assert torch.equal(got, ref) and torch.equal(kc, kc2) and torch.equal(vc, vc2)


@pytest.mark.parametrize("M,N,K", [(66, 512, 4096), (300, 4096, 14336), (1300, 768, 640), (4200, 1024, 512)])
def test_gemm_routes_agree(native, M, N, K):
    """The default route (whatever launches its plan has) against the fp32 product and, unsplit, gemm_w4."""
    x, w, b, r = operands(M, N, K)
    plan = native.gemm_plan(M, N, K, True, native._cu_count())
    y = native.gemm(x, w, bias=b, resid=r, epi="bias_resid")
    assert rel_err(y, R.linear(x, w, b, r, epi="bias_resid")) < 4e-3
    if all(S == 1 for _, _, _, S in plan):
        assert torch.equal(y, native.gemm(x, w, bias=b, resid=r, epi="bias_resid", path=6))
    S = native.slab_count(M, N, K)
    if S > 1:
        assert rel_err(native.gemm_splitk(x, w, S).sum(0), x.float() @ w.float().t()) < 1e-5
