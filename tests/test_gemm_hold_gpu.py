"""Decode projections of a few rows: gate/up with held activations, logits and split-K slabs of the weight ring."""
import pytest
import torch

from rag_llm_k8s_amd.ops.fp8 import quantize_weight

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _glu(x, w, act):
    z = (x.double() @ w.double().t()).view(x.shape[0], -1, 2, 64)
    return act(z[:, :, 0].reshape(x.shape[0], -1), z[:, :, 1].reshape(x.shape[0], -1))


@pytest.mark.parametrize("rows", [128, 2816, 8320, 16384])  # one tile group; less than a tile a CU; uneven shares; even ones
@pytest.mark.parametrize("K", [1024, 2048, 3072, 4096, 5120])
def test_gemm_hold(native, rows, K):
    """Row counts around the 16-row fragments and the launch's limit, both weight types, strided activations and output."""
    g = torch.Generator(device=DEV).manual_seed(rows + K)
    w = (torch.randn(rows, K, device=DEV, generator=g) * K ** -0.5).bfloat16()
    w8 = quantize_weight(w)
    par = torch.tensor([1.0, 1.7, 1.0], device=DEV)
    X = torch.randn(64, K + 8, device=DEV, generator=g).bfloat16()[:, :K]
    for M in (1, 15, 16, 17, 33, 64):
        x, out = X[:M], torch.full((M + 1, rows // 2 + 64), 7.0, device=DEV).bfloat16()
        cases = [(w8.w8, w8.scale, None, "silu_mul", w8.w8.double() * w8.scale.double()[:, None]),
                 (w, None, None, "silu_mul", w), (w, None, par, "glu_clip", w)]
        for wt, sw, p, epi, wd in cases:
            if native._lib.lib().ragk_gemm_hold_rows(K, int(sw is not None)) == 0:
                continue
            native.gemm_hold(x, wt, sw, p, epi, out=out[:M, :rows // 2])

            def act(a, b):
                if epi == "silu_mul":
                    return a * torch.sigmoid(a) * b
                a = a.clamp(max=1.0)
                return a * torch.sigmoid(1.7 * a) * (b.clamp(-1.0, 1.0) + 1.0)
            ref = _glu(x, wd, act)
            # one rounding to the 8 bits of bf16: at most 2^-8 of each value (1.6e-3 in the mean square); fp32 sums are far below
            assert (out[:M, :rows // 2].double() - ref).norm() / ref.norm() < 2.0 ** -8, (M, epi)
            assert out[M:].eq(7.0).all() and out[:, rows // 2:].eq(7.0).all()


@pytest.mark.parametrize("N,K", [(16384, 1024), (32000, 256), (32772, 2048), (50304, 384)])
def test_logits_rows(native, N, K):
    """Vocabularies of a ragged last tile, on both sides of the row count where the kernel changes."""
    w = (torch.randn(N, K, device=DEV) * K ** -0.5).bfloat16()
    for M in (1, 7, 8, 17, 64):
        x = torch.randn(M, K, device=DEV).bfloat16()
        got = native.gemm(x, w, out_f32=True)
        ref = x.double() @ w.double().t()
        # fp32 sums of K products of size K^-0.5
        assert (got.double() - ref).abs().max().item() < K * 2.0 ** -24 * 8


@pytest.mark.parametrize("N,K", [(2048, 5632), (4096, 4096), (4096, 7168), (4096, 8192), (6144, 4096)])
def test_stream_slabs(native, N, K):
    """The split-K slabs sum to the product whichever tile and split the rule takes."""
    w = (torch.randn(N, K, device=DEV) * K ** -0.5).bfloat16()
    for M in (5, 17, 64):
        x = torch.randn(M, K, device=DEV).bfloat16()
        assert (native.gemm_part(x, w).double().sum(0) - x.double() @ w.double().t()).abs().max().item() < K * 2.0 ** -24 * 8


def test_rows_of_any_stride(native):
    """Rows that start off the 16 bytes of a vector, or megabytes apart, give what their copies give."""
    w = (torch.randn(2816, 2048, device=DEV) * 2048 ** -0.5).bfloat16()
    head = (torch.randn(16384, 2048, device=DEV) * 2048 ** -0.5).bfloat16()
    w8 = quantize_weight(w)
    base = torch.randn(12, 2053, device=DEV).bfloat16()
    for x in (base[:, :2048], base[:, 3:2051]):
        c = x.contiguous()
        # both round to bf16 once from fp32 sums of another order
        for a, b in ((native.gemm(x, w, epi="silu_mul"), native.gemm(c, w, epi="silu_mul")),
                     (native.gemm_fp8(x, w8, epi="silu_mul"), native.gemm_fp8(c, w8, epi="silu_mul")),
                     (native.gemm(c, head, out_f32=True), native.gemm(c, head, out=torch.empty(12, 16392, device=DEV)[:, :16384],
                                                                      out_f32=True))):
            assert ((a.double() - b.double()).norm() / b.double().norm()).item() < 2.0 ** -7
    far = torch.empty_strided((70, 256), (2 ** 22, 1), dtype=torch.bfloat16, device=DEV)
    far.copy_(torch.randn(70, 256, device=DEV))
    assert torch.equal(native.gemm(far, w[:, :256].contiguous()), native.gemm(far.contiguous(), w[:, :256].contiguous()))


@pytest.mark.parametrize("M", [1, 12, 64, 70])
def test_gated_units_are_bf16_only(native, M):
    """fp32 rows of a gated unit are refused at every size, whichever kernel would take the product; so is another output."""
    x, w = torch.zeros(M, 2048, device=DEV).bfloat16(), torch.zeros(2816, 2048, device=DEV).bfloat16()
    out = torch.full((M, 1408), 7.0, device=DEV)
    for args in (dict(epi="silu_mul"), dict(epi="glu_clip", bias=torch.ones(3, device=DEV))):
        with pytest.raises((ValueError, native._lib.NativeLibraryError)):
            native.gemm(x, w, out=out, out_f32=True, **args)
    if M <= 64:
        for bad in (out, out.bfloat16()[:, ::2], torch.zeros(M, 1344, device=DEV).bfloat16()):
            with pytest.raises(ValueError):
                native.gemm_hold(x, w, out=bad)
    assert out.eq(7.0).all()
