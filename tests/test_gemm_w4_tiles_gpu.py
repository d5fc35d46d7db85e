"""gemm_w4's tiles of 224 and 192 rows: every value is the 256-row tile's (one order of K, one epilogue)."""
import math

import pytest
import torch

from rag_llm_k8s_amd.ops import reference as R

pytestmark = pytest.mark.gpu
DEV = "cuda"


# three K-tiles and odd counts of them, rows and columns on and past a tile's edge, and (blocks > 0) several tiles a block
@pytest.mark.parametrize("mi", [38, 39])
@pytest.mark.parametrize("M,N,K,blocks", [(65, 256, 192, 0), (223, 264, 256, 0), (224, 512, 320, 0), (225, 1032, 448, 0),
                                          (193, 768, 192, 0), (2000, 1024, 192, 8), (1345, 1288, 704, 16)])
def test_tiles_agree(native, mi, M, N, K, blocks):
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x = torch.randn(M, K, device=DEV, generator=g).bfloat16()
    w = (torch.randn(N, K, device=DEV, generator=g) / math.sqrt(K)).bfloat16()
    b, r = torch.randn(N, device=DEV, generator=g).bfloat16(), torch.randn(M, N, device=DEV, generator=g).bfloat16()
    par = torch.tensor([2.0, 1.702, 1.0, 0.0], device=DEV)
    try:
        native.set_w4_grid(blocks or -1)
        for epi in ("none", "bias", "resid", "bias_resid", "bias_gelu", "gelu", "bias_gelu_tanh", "silu_mul", "glu_clip"):
            pair = epi in native.PAIR_EPI
            if pair and N % 256:
                continue
            for f32 in (False,) if pair else (False, True):
                y, z = (torch.full((M + 1, N // 2 if pair else N), -3.0, device=DEV, dtype=torch.float32 if f32 else torch.bfloat16)
                        for _ in range(2))
                for out, m in ((y, mi), (z, 0)):
                    native._gemm_rows(x, w, par if epi == "glu_clip" else b if "bias" in epi else None, r if "resid" in epi else None,
                                      epi, out[:M], f32, 0, M, m, 1)
                assert torch.equal(y, z) and bool((y[M] == -3.0).all()), (epi, f32)
                if epi == "none" and f32:  # fp32 sums of K products of N(0, 1) / sqrt(K): far inside 1e-5
                    assert ((y[:M] - x.float() @ w.float().t()).norm() / y[:M].norm()).item() < 1e-5
    finally:
        native.set_w4_grid(-1)


@pytest.mark.parametrize("im", [6, 7])
@pytest.mark.parametrize("M,Hq,Hkv,blocks", [(300, 4, 2, 0), (1000, 2, 1, 8), (448, 12, 2, 8)])
def test_rotated_projection_tiles(native, im, M, Hq, Hkv, blocks):
    K, N, L = 256, (Hq + 2 * Hkv) * 128, native._lib.lib()
    g = torch.Generator(device=DEV).manual_seed(M)
    x = torch.randn(M, K, device=DEV, generator=g).bfloat16()
    w = (torch.randn(N, K, device=DEV, generator=g) / 16).bfloat16()
    cos, sin = (t.to(DEV) for t in R.rope_tables(128, 512))
    pos = torch.randint(0, 512, (M,), device=DEV, generator=g).int()
    slots = torch.randperm((M // 64 + 2) * 64, device=DEV, generator=g)[:M].int()
    slots[::5] = -1
    got = []
    try:
        native.set_w4_grid(blocks or -1)
        for m in (im, 8):
            out = torch.zeros(M, N, device=DEV).bfloat16()
            kc, vc = torch.zeros(2, M // 64 + 2, Hkv, 64, 128, device=DEV).bfloat16()
            rc = L.ragk_gemm_w4_rope_kv(x.data_ptr(), K, w.data_ptr(), K, out.data_ptr(), N, M, K, pos.data_ptr(), slots.data_ptr(),
                                        cos.data_ptr(), sin.data_ptr(), kc.data_ptr(), vc.data_ptr(), Hq, Hkv, 64, m,
                                        native.stream_ptr())
            assert rc == 0
            got.append((out, kc, vc))
    finally:
        native.set_w4_grid(-1)
    assert all(torch.equal(a, b) for a, b in zip(*got)) and bool(got[0][0].any())
