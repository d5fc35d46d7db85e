"""The launch rule of products with more than 64 rows: every row once, splits that the kernels take."""
import random

import pytest
import torch

from rag_llm_k8s_amd.ops import _lib
from rag_llm_k8s_amd.ops import native as n


def test_plans_cover_every_row_with_legal_launches():
    r = random.Random(1)
    for _ in range(400):
        M = int(2 ** r.uniform(6.05, 15.5))
        rows, K = 8 * r.randint(1, 4000), 128 * r.randint(1, 120)
        for w4 in (False, K >= 192):
            plan = n.gemm_plan(M, rows, K, w4, 256)
            at = 0
            for r0, r1, mi, S in plan:
                assert r0 == at < r1
                at = r1
                assert (mi in n.MID_TILES or (mi in n.W4_TILES and w4 and S == 1)) and 1 <= S <= max(1, K // 256)
            assert at == M
        S, mi = n._slab_best(M, rows, K, 256)
        assert S == 1 or (K % (64 * S) == 0 and K // S >= 256 and (mi in n.MID_TILES or mi == 0))


def test_launch_model_prefers_full_rounds():
    """What the plan is for: few rows split K, one filled round of large tiles stays whole, a ragged last round of gemm_w4's
    tiles goes to the smaller ones."""
    assert n.gemm_plan(300, 4096, 14336, True, 256)[0][3] > 1
    assert n.gemm_plan(4096, 4096, 4096, True, 256) == ((0, 4096, 0, 1),)
    (a, b) = n.gemm_plan(14076, 4096, 4096, True, 256)
    assert a == (0, 12288, 0, 1) and b[2] > 0


def test_short_inner_dimension_stays_off_the_long_ring():
    """Encoders of 128 columns: gemm_w4 refuses two K-tiles, at the batch sizes too where its tiles would be cheapest."""
    for H, I in ((128, 512), (128, 1024), (128, 2048)):
        for T in (65, 300, 4096, 24576, 49152, 65536):
            for N, K in ((3 * H, H), (H, H), (I, H), (H, I)):
                assert all(mi in n.MID_TILES for _, _, mi, _ in n.gemm_plan(T, N, K, True, 256)) or K >= 192


def test_work_lists_of_prompts():
    """Every tile of every sequence once, later positions first, sequences in order among equals: short lists and long ones."""
    r = random.Random(2)
    for Hq, Hkv in ((32, 8), (12, 12), (16, 8)):
        qt = n.prefill_qtile(Hq, Hkv)
        for lens in ([], [0], [1], [qt], [qt + 1, 0, qt], [64 * qt], [64 * qt + 1], [4096, 5, 70], [r.randint(1, 900) for _ in range(9)]):
            want = sorted(((s, q) for s, L in enumerate(lens) for q in range(0, L, qt)), key=lambda t: -t[1])
            assert n.build_prefill_tiles(lens, Hq, Hkv).tolist() == [list(t) for t in want]


def test_operand_rows_that_are_copied():
    """Rows off 16 bytes or megabytes apart, whole tensors that start between vectors; nothing else."""
    a = torch.arange(80 * 264, dtype=torch.float32).bfloat16().view(80, 264)
    far = torch.empty_strided((3, 256), (2 ** 22, 1), dtype=torch.bfloat16)
    far.copy_(a[:3, :256])
    for t, copied in ((a, False), (a[:, :256], False), (a[:, 8:], False), (a[::2], False), (a[:, 4:260], True), (a[:, :132][1:], False),
                      (a.view(-1)[:79 * 263].view(79, 263)[:, :256], True), (a.view(-1)[1:1 + 70 * 256].view(70, 256), True),
                      (far, True), (far[:, :8], True)):
        (got, same), (same2, got2) = n._tile_rows(t, a), n._tile_rows(a, t)
        assert same is a and same2 is a and torch.equal(got, got2)
        assert (got.data_ptr() != t.data_ptr()) == copied and torch.equal(got, t)
        assert not copied or (got.is_contiguous() and got.data_ptr() % 16 == 0)


def test_plans_follow_their_settings(monkeypatch):
    """What was worked out under one setting is not kept for another: splits off and on, their least rows, a launch's blocks."""
    monkeypatch.setattr(n, "_cu_count", lambda: 256)
    sizes = [(300, 4096, 4096), (700, 1024, 4096), (5000, 4096, 4096)]
    on = [(n.slab_count(*s), n.ln_slabs(*s), n.prefill_nsplit(*s)) for s in sizes]
    assert all(a[0] > 1 for a in on[:2]) and all(a[1][0] > 1 for a in on[:2]) and on[2][2] > 1
    for f in (n._slab_best, n._splitk_tile, n.gemm_plan):
        f.cache_clear()
    monkeypatch.setattr(n, "PREFILL_SPLITK", False)
    assert all((n.slab_count(*s), n.ln_slabs(*s), n.prefill_nsplit(*s)) == (1, (1, 0), 1) for s in sizes)
    monkeypatch.setattr(n, "PREFILL_SPLITK", True)
    assert on == [(n.slab_count(*s), n.ln_slabs(*s), n.prefill_nsplit(*s)) for s in sizes]
    off = n._encoder_plans(700, 1024, 4096, 256, n.PREFILL_SPLITK, n.PREFILL_SPLITK_MIN_M)
    assert off[1] > 0 and off[0][3].slabs and [p.r1 for p in off[0][3].p[:1]] == [700]
    monkeypatch.setattr(n, "PREFILL_SPLITK_MIN_M", 10 ** 6)
    assert all(n.prefill_nsplit(*s) == 1 for s in sizes)
    assert n.slab_count(1700, 4096, 14336) == 1
    monkeypatch.setattr(n, "PREFILL_SPLITK_MIN_M", 1024)
    assert n.slab_count(1700, 4096, 14336) == 2


@pytest.mark.skipif(not _lib.available(), reason="kernel library not built")
def test_slices_follow_the_block_count(monkeypatch):
    a = n.gemm_part_slabs(1, 4096, 4096)
    monkeypatch.setattr(n, "PART_MIN_BLOCKS", 64)
    b = n.gemm_part_slabs(1, 4096, 4096)
    monkeypatch.setattr(n, "PART_MIN_BLOCKS", 512)
    assert a != b and n.gemm_part_slabs(1, 4096, 4096) == a


def test_smaller_tiles_only_well_ahead():
    """224 and 192 rows a tile instead of 256 from one modelled gain on for every product, also where the last round is all but
    empty (14076 x 28672 x 4096: 24 rounds and 16 tiles)."""
    r = random.Random(5)
    sizes = [(14076, 28672, 4096), (15284, 18560, 4096), (8908, 16704, 4096)]
    sizes += [(r.randint(1500, 16384), 256 * r.randint(4, 112), 64 * r.randint(16, 64)) for _ in range(500)]
    for M, rows, K in sizes:
        (_, _, mi, _), *rest = n.gemm_plan(M, rows, K, True, 256)
        t = n._tiles_us(M, rows, K, 0, 1, 256)
        if mi in (38, 39) and not rest and n._mid_best(M, rows, K, 256, n.SLAB_US, 3.0)[0] >= t:
            assert n._tiles_us(M, rows, K, mi, 1, 256) < {38: 0.95, 39: 0.97}[mi] * t, (M, rows, K)
