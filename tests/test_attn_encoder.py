"""Bidirectional attention over packed sequences: the work list, and attn_encoder_kernel at the edges of its tiles."""
import math
import random

import pytest
import torch

from rag_llm_k8s_amd.ops import native as n
from rag_llm_k8s_amd.ops import reference as R

DEV = "cuda"


def test_work_list_holds_every_tile_once():
    r = random.Random(3)
    for lens in ([], [0], [1], [128], [129, 0, 128], [4096, 5, 70], [r.randint(0, 900) for _ in range(9)], [64] * 40):
        tiles = n.build_encoder_tiles(lens, 12).tolist()
        assert sorted(map(tuple, tiles)) == [(s, q) for s, L in enumerate(lens) for q in range(0, L, 128)]
        by = [lens[s] for s, _ in tiles]
        assert by == sorted(by, reverse=True)
        assert all(a[0] != b[0] or a[1] + 128 == b[1] for a, b in zip(tiles, tiles[1:]))


def attend(native, qkv, lens, H, D, shift=0):
    """shift: elements by which the rows lie off 16 bytes (the general kernel then)."""
    T = qkv.shape[0]
    buf = torch.zeros(T * 3 * H * D + 8, device=DEV).bfloat16()
    g = buf[shift:shift + T * 3 * H * D].view(T, 3 * H * D)
    g.copy_(qkv)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32).to(DEV)
    out = torch.full((T + 1, H * D), -3.0, device=DEV).bfloat16()
    native.attn_prefill(g, g[:, H * D:], g[:, 2 * H * D:], cu, torch.tensor(lens, dtype=torch.int32).to(DEV),
                        n.build_encoder_tiles(lens, H).to(DEV), out, H, H, D, causal=False, paged=False, cu_kv=cu, kv_stride=3 * H * D)
    assert bool((out[T] == -3.0).all())
    return out[:T].float().cpu()


# one key, tiles of 64 keys and 128 queries filled exactly, by one more and by one less, several tiles, one head and many
@pytest.mark.gpu
@pytest.mark.parametrize("D,H", [(64, 2), (32, 3), (64, 16), (32, 12)])
@pytest.mark.parametrize("lens", [[1], [63, 64, 65], [127, 128, 129, 2], [14], [400, 1, 33], [17, 257]])
@pytest.mark.parametrize("spread", [1.0, 12.0])  # 12: maxima that move by hundreds from tile to tile
def test_attn_encoder_edges(native, D, H, lens, spread):
    g = torch.Generator().manual_seed(len(lens) + D + H)
    T = sum(lens)
    qkv = torch.randn(T, 3 * H * D, generator=g)
    qkv[:, :2 * H * D] *= torch.linspace(1, spread, T)[:, None]
    qkv = qkv.bfloat16()
    q, k, v = (qkv[:, i * H * D:(i + 1) * H * D].reshape(T, H, D) for i in range(3))
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32)
    ref = R.attention_varlen(q, k, v, cu, torch.tensor(lens, dtype=torch.int32), False, 1 / math.sqrt(D), cu_kv=cu).float().reshape(T, -1)
    got = attend(native, qkv, lens, H, D)
    # bf16 weights and result: two roundings of 2^-9
    assert ((got - ref).norm() / ref.norm()).item() < 2 ** -8
    general = attend(native, qkv, lens, H, D, shift=4)
    assert ((got - general).norm() / ref.norm()).item() < 2 ** -8


@pytest.mark.gpu
def test_attn_encoder_keeps_sequences_apart(native):
    """NaN and infinities in one sequence: its own rows as the general kernel gives them, its neighbours untouched."""
    D, H, lens = 64, 2, [70, 130, 65]
    qkv = torch.randn(265, 3 * H * D, generator=torch.Generator().manual_seed(5)).bfloat16()
    clean = attend(native, qkv, lens, H, D)
    qkv[100, H * D + 3] = float("nan")
    qkv[150, 2 * H * D + 70] = float("inf")
    got, general = attend(native, qkv, lens, H, D), attend(native, qkv, lens, H, D, shift=4)
    for rows in (slice(0, 70), slice(200, 265)):
        assert torch.equal(got[rows], clean[rows])
    assert torch.equal(got.isnan(), general.isnan()) and torch.equal(got.isinf(), general.isinf())


@pytest.mark.gpu
def test_rows_megabytes_apart(native):
    """Keys and values whose rows of a tile lie further apart than 32-bit offsets reach: what they give side by side."""
    D, H, lens = 64, 2, [66, 3]
    T = sum(lens)
    qkv = torch.randn(T, 3 * H * D, generator=torch.Generator().manual_seed(6)).bfloat16().to(DEV)
    cu = torch.tensor([0, 66, T], dtype=torch.int32, device=DEV)
    kl, tiles = torch.tensor(lens, dtype=torch.int32, device=DEV), n.build_encoder_tiles(lens, H).to(DEV)
    outs = []
    for ld in (2 * H * D, 2 ** 24 - 8, 2 ** 24, 2 ** 24 + 2 ** 20):
        kv = torch.empty(T * ld, dtype=torch.bfloat16, device=DEV).view(T, ld)[:, :2 * H * D]
        kv.copy_(qkv[:, H * D:])
        out = torch.empty(T, H * D, dtype=torch.bfloat16, device=DEV)
        native.attn_prefill(qkv, kv, kv[:, H * D:], cu, kl, tiles, out, H, H, D, causal=False, paged=False, cu_kv=cu, kv_stride=ld)
        outs.append(out.float())
        del kv
    assert torch.equal(outs[0], outs[1])
    for o in outs[2:]:  # the general kernel: bf16 weights and results of both, 2^-9 a rounding
        assert ((o - outs[0]).norm() / outs[0].norm()).item() < 2 ** -8
