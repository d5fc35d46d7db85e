"""LayerNorm and pooling at the widths where their split changes."""
import pytest
import torch

from rag_llm_k8s_amd.ops import reference as R

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("T,H", [(1, 384), (5, 512), (3, 520), (9, 1024), (4, 1032), (2, 2048), (3, 2056), (5, 8192)])
def test_layernorm_rows(native, T, H):
    """Widths around the vectors a lane holds and the change from one wave to four a row."""
    torch.manual_seed(H)
    x, r = torch.randn(T, H, device=DEV).bfloat16(), torch.randn(T, H, device=DEV).bfloat16()
    g, b = torch.randn(H, device=DEV).bfloat16(), torch.randn(H, device=DEV).bfloat16()
    for res in (None, r):
        ref = R.layernorm(x.double(), g.double(), b.double(), 1e-12, resid=None if res is None else res.double())
        assert (native.layernorm(x, g, b, 1e-12, resid=res).double() - ref).norm() / ref.norm() < 3e-3


@pytest.mark.parametrize("H", [8, 100, 384, 1000, 2048])
def test_pool_rows(native, H):
    """Column groups of eight and single columns (odd widths and strides), one row to more rows than row groups."""
    lens = [1, 3, 200, 17]
    cu = torch.tensor([0, 1, 4, 204, 221], dtype=torch.int32, device=DEV)
    h = torch.randn(sum(lens), H + 3, device=DEV).bfloat16()
    for x in (h[:, :H], h[:, :H].contiguous()):
        for mode in ("cls", "mean", "last"):
            ref = R.pool_l2norm(x.float().cpu(), cu.cpu(), mode=mode)
            assert (native.pool_l2norm(x, cu, mode=mode).cpu() - ref).abs().max().item() < 1e-5


@pytest.mark.parametrize("S", [1, 3, 4, 9])
@pytest.mark.parametrize("T,H", [(1, 384), (5, 520), (3, 1032), (2, 2056), (5, 8192)])
def test_layernorm_slabs(native, T, H, S):
    """Slab counts around the four that are loaded together, widths as above; the residual's rows are overwritten in place."""
    torch.manual_seed(H + S)
    P, r = torch.randn(S, T, H, device=DEV), torch.randn(T, H, device=DEV).bfloat16()
    bias, g, b = (torch.randn(H, device=DEV).bfloat16() for _ in range(3))
    ref = R.layernorm(P.double().sum(0) + bias.double() + r.double(), g.double(), b.double(), 1e-12)
    # one rounding to bf16 a value: at most 2^-8 of it
    assert (native.layernorm_slabs(P, bias, r, g, b, 1e-12, out=r).double() - ref).norm() / ref.norm() < 2.0 ** -8


@pytest.mark.parametrize("N,K", [(384, 384), (384, 1536), (1024, 1024), (1024, 4096), (256, 512)])
def test_gemm_layernorm(native, N, K):
    """Both forms of the pair, on either side of every line between them."""
    torch.manual_seed(N + K)
    w = (torch.randn(N, K, device=DEV) * K ** -0.5).bfloat16()
    bias, g, b = (torch.randn(N, device=DEV).bfloat16() for _ in range(3))
    for M in (1, 11, 12, 17, 18, 64, 65, 200, 1100):
        x, r = torch.randn(M, K, device=DEV).bfloat16(), torch.randn(M, N, device=DEV).bfloat16()
        ref = R.layernorm(x.double() @ w.double().t() + bias.double() + r.double(), g.double(), b.double(), 1e-12)
        # roundings to bf16, at most 2^-8 of a value each: the result and, unsplit, the sum that is normalised
        assert (native.gemm_layernorm(x, w, bias, r, g, b, 1e-12).double() - ref).norm() / ref.norm() < 2.0 ** -7


@pytest.mark.parametrize("T", [60, 300])
def test_gemm_layernorm_refuses_what_gemm_does(native, T):
    """At sizes whose product is split, as at the others."""
    x, w = torch.zeros(T, 1024, device=DEV).bfloat16(), torch.zeros(1024, 1024, device=DEV).bfloat16()
    v, r = torch.zeros(1024, device=DEV).bfloat16(), torch.zeros(T, 1024, device=DEV).bfloat16()
    assert native.ln_slabs(T, 1024, 1024)[0] > 1
    native.gemm_layernorm(x, w, v, r, v, v, 1e-5)
    for bad in ((x[:, :896], w, v, r), (x, w[:, :896], v, r), (x.float(), w, v, r), (x, w.half(), v, r), (x, w.t(), v, r),
                (x[:, :960], w[:, :960], v, r), (x, w, v.float(), r), (x, w, v[:512], r), (x, w, None, r), (x, w, v, r[:5]),
                (x, w, v, r.float()), (x, w.cpu(), v, r)):
        with pytest.raises(ValueError):
            native.gemm_layernorm(*bad, v, v, 1e-5)
