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


@pytest.mark.parametrize("M", [65, 70, 300, 1100])
def test_operands_between_vectors(native, M):
    """x and w with rows off 16 bytes or from a start between vectors, or megabytes apart: what their copies give, bit for bit,
    through every entry that fetches them in 16-byte pieces. Bias, residual and output lie anywhere."""
    g = torch.Generator(device=DEV).manual_seed(M)

    def odd(rows, cols, how):
        t = torch.randn(rows, cols + 16, device=DEV, generator=g).bfloat16()
        flat = torch.randn(rows * cols + 8, device=DEV, generator=g).bfloat16()
        return {"stride": torch.randn(rows, cols + 5, device=DEV, generator=g).bfloat16()[:, :cols], "start": t[:, 3:cols + 3],
                "flat": flat[1:rows * cols + 1].view(rows, cols)}[how]

    N, K = 1024, 1024
    for how in ("stride", "start", "flat"):
        x, w, wgu = odd(M, K, how), odd(N, K, how), odd(2 * N, K, how)
        cx, cw, cgu = (t.clone(memory_format=torch.contiguous_format) for t in (x, w, wgu))
        b, r = odd(1, N, how)[0], odd(M, N, how)
        out = odd(M, N, how)
        native.gemm(x, w, bias=b, resid=r, epi="bias_resid", out=out)
        assert torch.equal(out, native.gemm(cx, cw, bias=b.clone(), resid=r.contiguous(), epi="bias_resid"))
        assert torch.equal(native.gemm(x, wgu, epi="silu_mul"), native.gemm(cx, cgu, epi="silu_mul"))
        assert torch.equal(native.gemm(x, w, path=0), native.gemm(cx, cw, path=0))
        assert torch.equal(native.gemm_splitk(x, w, 2), native.gemm_splitk(cx, cw, 2))
        gain, shift = torch.randn(2, N, device=DEV, generator=g).bfloat16()
        assert torch.equal(native.gemm_layernorm(x, w, b.clone(), cx, gain, shift, 1e-5),
                           native.gemm_layernorm(cx, cw, b.clone(), cx, gain, shift, 1e-5))
        few = odd(60, K, how)
        assert torch.equal(native.gemm_layernorm(few, w, b.clone(), cx[:60], gain, shift, 1e-5),
                           native.gemm_layernorm(few.clone(memory_format=torch.contiguous_format), cw, b.clone(), cx[:60], gain, shift, 1e-5))
        cos, sin = (t.to(DEV) for t in R.rope_tables(128, M))
        pos = torch.arange(M, device=DEV).int()
        kc = torch.zeros(2, M // 64 + 1, 2, 64, 128, device=DEV).bfloat16()
        vc = torch.zeros_like(kc)
        a, c = (native.gemm_rope_kv(p, q, pos, cos, sin, pos, kc[i], vc[i], 4, 2, 128) for i, (p, q) in enumerate(((x, w), (cx, cw))))
        assert torch.equal(a, c) and torch.equal(kc[0], kc[1]) and torch.equal(vc[0], vc[1])
    if M <= 70:
        far = torch.empty_strided((M, K), (2 ** 22, 1), dtype=torch.bfloat16, device=DEV)
        far.copy_(cx)
        assert torch.equal(native.gemm_splitk(far, cw, 2), native.gemm_splitk(cx, cw, 2))


def test_library_refuses_rows_between_vectors(native):
    """The C entry itself: nothing is launched."""
    t = torch.zeros(128 * 136, dtype=torch.bfloat16, device=DEV)
    out, L = torch.zeros(80, 128, dtype=torch.bfloat16, device=DEV), native._lib.lib()
    for a, lda, b, ldb in ((0, 129, 0, 128), (2, 128, 0, 128), (0, 128, 0, 132), (0, 128, 4, 128)):
        assert L.ragk_gemm_mid(t.data_ptr() + a, lda, t.data_ptr() + b, ldb, out.data_ptr(), 128, None, None, 0, 80, 128, 128, 0, 0,
                               4, 1, None, 0) != 0
    torch.cuda.synchronize()
    assert not out.any()


# 224 x 128 and 160 x 256: edges in rows, a last tile of 8, 136 and 248 columns, rings with as many K-tiles as slots and fewer
@pytest.mark.parametrize("mi,S,M,N,K", [(7, 1, 225, 136, 192), (7, 2, 223, 384, 128), (7, 3, 449, 640, 704), (21, 1, 161, 264, 192),
                                         (21, 1, 159, 392, 128), (21, 2, 321, 504, 256), (21, 5, 320, 256, 704), (21, 1, 2000, 5120, 192)])
def test_gemm_mid_larger_tiles(native, mi, S, M, N, K):
    x, w, b, r = operands(M, N, K)
    y = native.gemm_mid(x, w, out=torch.empty_like(r), mi=mi, S=S)
    assert rel_err(y, x.float() @ w.float().t()) < 4e-3  # bf16 result: 2^-9 per value
    for epi in ("none", "bias", "bias_resid", "gelu"):
        y = native.gemm_mid(x, w, bias=b, resid=r, epi=epi, out=torch.empty_like(r), mi=mi, S=S)
        # another tile's values: the order of K is the same in all of them
        assert torch.equal(y, native.gemm_mid(x, w, bias=b, resid=r, epi=epi, out=torch.empty_like(r), mi=4, S=S)), epi
    rows = N // 128 * 128  # gate / up: also one group in the last 256-column tile
    par = torch.tensor([2.0, 1.702, 1.0, 0.0], device=DEV)
    for epi, bias in (("silu_mul", None), ("glu_clip", par)):
        y, z = (native.gemm_mid(x, w[:rows], bias=bias, epi=epi, out=torch.empty(M, rows // 2, device=DEV).bfloat16(), mi=m, S=S)
                for m in (mi, 3))
        assert torch.equal(y, z), epi
    buf = torch.full((M + 2, N + 16), -3.0, device=DEV).bfloat16()
    native.gemm_mid(x, w, out=buf[1:M + 1, 8:N + 8], mi=mi, S=S)
    buf[1:M + 1, 8:N + 8] = -3.0
    assert bool((buf == -3.0).all())


@pytest.mark.parametrize("mi", [7, 21])
@pytest.mark.parametrize("M,Hq,Hkv,S", [(161, 1, 1, 1), (300, 4, 2, 1), (225, 2, 1, 3)])
def test_rotated_projection_larger_tiles(native, mi, M, Hq, Hkv, S):
    """The C entry with a given tile against 128 x 128 (which gemm + rope_kv is compared with above); three heads leave half of the
    last 256 columns."""
    K, N, L = 640, (Hq + 2 * Hkv) * 128, native._lib.lib()
    x, w, _, _ = operands(M, N, K)
    cos, sin = (t.to(DEV) for t in R.rope_tables(128, 512))
    pos = torch.randint(0, 512, (M,), device=DEV).int()
    slots = torch.randperm((M // 64 + 2) * 64, device=DEV)[:M].int()
    slots[::5] = -1
    ws = torch.empty(S * M * N, device=DEV)
    got = []
    for m in (mi, 4):
        out = torch.zeros(M + 1, N, device=DEV).bfloat16()
        kc, vc = torch.zeros(2, M // 64 + 2, Hkv, 64, 128, device=DEV).bfloat16()
        rc = L.ragk_gemm_mid_rope_kv(x.data_ptr(), K, w.data_ptr(), K, out.data_ptr(), N, M, K, pos.data_ptr(), slots.data_ptr(),
                                     cos.data_ptr(), sin.data_ptr(), kc.data_ptr(), vc.data_ptr(), Hq, Hkv, 64, m, S, ws.data_ptr(),
                                     native.stream_ptr())
        assert rc == 0
        got.append((out, kc, vc))
    assert all(torch.equal(a, b) for a, b in zip(*got)) and bool(got[0][0][:M].any())
