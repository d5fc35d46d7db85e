"""fp8 weights whose rows lie further apart, or start off 16 bytes."""
import pytest
import torch

from rag_llm_k8s_amd.ops import _lib

DEV = "cuda"
INVALID = 1  # hipErrorInvalidValue


def test_rows_off_16_bytes_are_not_launched():
    L = _lib.lib()
    for x, A in ((1, None), (None, 1)):
        assert L.ragk_gemm_fp8(x, 256, A, 256, None, None, 257, None, None, 256, None, None, 0, 4, 256, 256, 0, 0, None) == INVALID
    assert L.ragk_gemm_stream(None, 256, None, 257, 1, None, 256, None, None, 0, 4, 256, 256, 0, 0, 1, None, None, None) == INVALID


def _weight(N, K):
    from rag_llm_k8s_amd.ops.fp8 import quantize_weight

    g = torch.Generator(device=DEV).manual_seed(N + K)
    return quantize_weight(torch.randn(N, K, generator=g, device=DEV) * K ** -0.5)


def _at(w8, pitch, start=0):
    """The same rows, `pitch` bytes apart, `start` bytes into an allocation."""
    from rag_llm_k8s_amd.ops.fp8 import Fp8Weight

    buf = torch.zeros(start + w8.shape[0] * pitch, dtype=torch.uint8, device=DEV)
    rows = buf[start:].as_strided(w8.shape, (pitch, 1), start)
    rows.copy_(w8.view(torch.uint8))
    return rows.view(torch.float8_e4m3fn)


# decode products, streamed and in slabs of held activations, the tiles of prompts
@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 17, 64, 65])
@pytest.mark.parametrize("N,K,epi", [(512, 2048, "none"), (16384, 2048, "none"), (512, 2048, "silu_mul"), (16384, 2048, "silu_mul")])
def test_rows_of_fp8_products(M, N, K, epi):
    from rag_llm_k8s_amd.ops import native
    from rag_llm_k8s_amd.ops.fp8 import Fp8Weight

    q, x = _weight(N, K), torch.randn(M, K, device=DEV).bfloat16()
    y = native.gemm_fp8(x, q, epi=epi)
    for pitch, start in ((K + 128, 0), (K, 8), (K, 1), (K + 16, 8)):  # (a start off 16 bytes: a copy)
        assert torch.equal(native.gemm_fp8(x, Fp8Weight(_at(q.w8, pitch, start), q.scale), epi=epi), y), (pitch, start)
    for w8 in (_at(q.w8, K + 1), _at(q.w8, K + 8), q.w8.as_strided((N, K), (0, 1)),
               q.w8.view(1, N, K), q.w8.view(torch.uint8).t().contiguous().view(torch.float8_e4m3fn).t()):
        with pytest.raises(ValueError):
            native.gemm_fp8(x, Fp8Weight(w8, q.scale), epi=epi)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 17, 64])
def test_rows_16_mb_apart(M):
    """Not for the held activations, whose lanes reach a row by a 32-bit offset."""
    from rag_llm_k8s_amd.ops import native
    from rag_llm_k8s_amd.ops.fp8 import Fp8Weight

    q, x = _weight(128, 2048), torch.randn(M, 2048, device=DEV).bfloat16()
    y = native.gemm_fp8(x, Fp8Weight(_at(q.w8, 1 << 24), q.scale), epi="silu_mul")
    g, u = (x.double() @ q.dequant(torch.float64).t()).chunk(2, 1)
    ref = torch.nn.functional.silu(g) * u
    # a bf16 result is within half a unit in the last of its 8 bits, 2^-9 of the value at most (and 0.6 of that in the mean, which
    # leaves room for fp32 sums)
    assert float((y.double() - ref).norm() / ref.norm()) < 2.0 ** -9
