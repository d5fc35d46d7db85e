"""fp8 projections of 17 to 64 rows as slabs of held activations, and shares of tiles of every length."""
import pytest
import torch

from rag_llm_k8s_amd.ops.fp8 import quantize_weight

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _operands(M, N, K, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(M, K + 8, device=DEV, generator=g).bfloat16()[:, :K]
    w = quantize_weight((torch.randn(N, K, device=DEV, generator=g) * K ** -0.5).bfloat16())
    return x, w, w.w8.double() * w.scale.double()[:, None]


def _bound(x, wd):
    """fp32 sums of K terms in any order: K 2^-24 of the terms' magnitudes."""
    return x.shape[1] * 2.0 ** -24 * (x.double().abs() @ wd.abs().t())


@pytest.mark.parametrize("N,K", [(4096, 14336), (8192, 4096), (4096, 10240), (5136, 8192)])
def test_partials(native, N, K):
    """Both sides of the rule's rows, around the 16-row fragments; columns that do not divide among the blocks."""
    for M in (16, 17, 32, 33, 48, 49, 64):
        x, w, wd = _operands(M, N, K, M)
        P = native.gemm_part(x, w)
        if native.use_hold_slabs(M, N, K):
            assert P.shape == (K // 2048, M, N)
        assert bool(((P.double().sum(0) - x.double() @ wd.t()).abs() <= _bound(x, wd)).all()), M


@pytest.mark.parametrize("N,K,ld", [(32, 1 << 20, 1 << 20), (64, 1 << 19, 1 << 24)])
def test_rows_too_long_or_too_far_apart(native, N, K, ld):
    """More slabs than there are CUs, and rows past a lane's 32-bit offset, go where they went."""
    from rag_llm_k8s_amd.ops.fp8 import Fp8Weight

    g = torch.Generator(device=DEV).manual_seed(N)
    x = torch.randn(33, K, device=DEV, generator=g).bfloat16()
    q = quantize_weight((torch.randn(N, K, device=DEV, generator=g) * K ** -0.5).bfloat16())
    rows = torch.zeros((N - 1) * ld + K, dtype=torch.uint8, device=DEV).view(torch.float8_e4m3fn).as_strided((N, K), (ld, 1))
    rows.view(torch.uint8).copy_(q.w8.view(torch.uint8))
    wd = q.w8.double() * q.scale.double()[:, None]
    P = native.gemm_part(x, Fp8Weight(rows, q.scale))
    assert bool(((P.double().sum(0) - x.double() @ wd.t()).abs() <= _bound(x, wd)).all())
    if ld == K:
        w2 = Fp8Weight(torch.cat([q.w8.view(torch.uint8)] * 4).view(torch.float8_e4m3fn), q.scale.repeat(4))
        z = (x.double() @ wd.t()).repeat(1, 4).view(33, 2, 64)
        ref = torch.nn.functional.silu(z[:, 0]) * z[:, 1]
        assert float((native.gemm_fp8(x, w2, epi="silu_mul").double() - ref).norm()) < 2.0 ** -8 * float(ref.norm())


@pytest.mark.parametrize("tiles", [1, 2, 3, 4, 5, 7, 63, 64, 65, 200])
def test_shares(native, tiles):
    """Blocks with one to 64 tiles, fewer and more than are in flight, a share that needs more blocks than asked for."""
    L = native._lib.lib()
    N, K = 16 * tiles, 4096
    for M in (5, 20, 40, 64):
        x, w, wd = _operands(M, N, K, tiles)
        ref, lim = x.double() @ wd.t(), _bound(x, wd)
        for blocks in (2, 3, 8):
            P = torch.full((2 * M * N + 64,), 7.0, device=DEV)
            native.check(L.ragk_gemm_hold_slabs(x.data_ptr(), x.stride(0), w.w8.data_ptr(), K, w.scale.data_ptr(), P.data_ptr(), M,
                                                N, K, blocks, native.stream_ptr()), "slabs")
            assert bool(((P[:2 * M * N].view(2, M, N).double().sum(0) - ref).abs() <= lim).all()), (M, blocks)
            assert bool((P[2 * M * N:] == 7).all())


@pytest.mark.parametrize("N,K", [(1792, 4096), (14336, 4096), (704, 6144), (8192, 6144)])
def test_gate_up(native, N, K):
    """Rows on both sides of what a launch holds; strided rows of x and of the result."""
    for M in (16, 17, 33, 64):
        x, w, wd = _operands(M, 2 * N, K, M + N)
        out = torch.full((M + 1, N + 8), 7.0, device=DEV).bfloat16()
        native.gemm_fp8(x, w, epi="silu_mul", out=out[:M, :N])
        z = (x.double() @ wd.t()).view(M, -1, 2, 64)
        gate, up = z[:, :, 0].reshape(M, -1), z[:, :, 1].reshape(M, -1)
        # one rounding to the 8 bits of bf16: at most 2^-8 of each value
        assert float((out[:M, :N].double() - torch.nn.functional.silu(gate) * up).norm()) < 2.0 ** -8 * float(
            (torch.nn.functional.silu(gate) * up).norm()), M
        assert bool((out[M] == 7).all()) and bool((out[:, N:] == 7).all())


@pytest.mark.parametrize("fp8", [True, False])
@pytest.mark.parametrize("N", [64, 192, 256, 1088, 4160])
def test_pair_shares(native, N, fp8):
    """The paired form over few blocks: tiles that fill their rounds or leave some."""
    L = native._lib.lib()
    K = 2048
    for M in (3, 32, 50):
        x, w, wd = _operands(M, 2 * N, K, N + M)
        wt = w.w8 if fp8 else wd.bfloat16()
        z = (x.double() @ (wd if fp8 else wt.double()).t()).view(M, -1, 2, 64)
        ref = torch.nn.functional.silu(z[:, :, 0].reshape(M, -1)) * z[:, :, 1].reshape(M, -1)
        for blocks in (1, 5, 9):
            out = torch.full((M + 1, N), 7.0, device=DEV).bfloat16()
            native.check(L.ragk_gemm_hold(x.data_ptr(), x.stride(0), wt.data_ptr(), K, w.scale.data_ptr() if fp8 else None,
                                          out.data_ptr(), N, None, M, N, K, native.EPI["silu_mul"], blocks,
                                          native.stream_ptr()), "hold")
            assert float((out[:M].double() - ref).norm()) < 2.0 ** -8 * float(ref.norm()), (M, blocks)
            assert bool((out[M] == 7).all())
