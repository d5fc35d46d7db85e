"""Which split-K slabs a decode step's products take (ops/native.py _deep_slabs, _part_stream, _fp8_halves)."""
import pytest
from hypothesis import given, settings
from hypothesis import strategies as st

from rag_llm_k8s_amd.ops import native


@pytest.mark.parametrize("N,K,few,S", [(18688, 4096, True, 4), (18688, 4096, False, 4), (20480, 4096, True, 4), (22528, 4096, True, 0),
                                       (16384, 4096, True, 0), (18688, 8192, True, 8), (18688, 3584, True, 4), (18688, 2048, True, 2),
                                       (9216, 4096, True, 4), (9216, 4096, False, 0), (12288, 4096, True, 0), (9344, 2048, True, 0),
                                       (10240, 8192, True, 8), (6144, 4096, True, 0), (4096, 14336, True, 0), (28672, 4096, True, 0)])
def test_where_rounds_of_short_slices_are_ahead(N, K, few, S):
    assert native._deep_slabs(N, K, 256, 0, 64, few) == S


@settings(max_examples=300, deadline=None)
@given(N=st.integers(1, 40000), steps=st.integers(1, 512), cus=st.sampled_from([64, 256, 304]), few=st.booleans())
def test_slabs_divide_the_product(N, steps, cus, few):
    rows, S = native._stream_part_cfg(N, steps * 64, cus, 0, 64)
    deep = native._deep_slabs(N, steps * 64, cus, 0, 64, few)
    assert deep == 0 or (deep > S >= 1 and deep <= 64 and steps % deep == 0 and steps // deep >= 14 and -(-N // rows) * S <= cus)


@pytest.mark.parametrize("N,K,ks,rows", [
    (10240, 8192, 32, [1, 3, 7, 16]), (5120, 16384, 32, [1, 3, 7, 16]), (9216, 8192, 32, [1, 4, 6, 16]), (8448, 8192, 32, [1, 4, 6, 16]),
    (20480, 4096, 32, [1, 4, 6, 16]), (6144, 12288, 32, [1, 4, 6, 16]), (9216, 4096, 16, [1, 4, 6, 16]), (12288, 4096, 16, []),
    (4096, 14336, 28, [])])
def test_where_fp8_slices_are_halved(N, K, ks, rows):
    tried = [1, 3, 4, 6, 7, 16, 17]
    took = [M for M in tried if native._fp8_halves(M, N, ks, K // (64 * ks))]
    assert took == [M for M in tried if rows and rows[0] <= M <= rows[-1] and (4 in rows or M not in (4, 6))]


@pytest.mark.parametrize("N,K,M,took", [
    # slices of 28 K-steps and more of a few rows, shorter ones, whole rounds of rows 16 KB apart
    (4096, 14336, 1, (128, 8, True)), (4096, 14336, 4, (128, 8, True)), (4096, 14336, 5, (128, 8, False)), (6144, 4096, 4, (0, 0, False)),
    (18688, 2048, 4, (0, 0, False)), (9728, 5120, 4, (0, 0, False)), (8192, 8192, 4, (0, 0, False)), (4096, 16384, 4, (0, 0, False)),
    (16384, 8192, 1, (0, 0, False)), (8192, 8192, 5, (128, 4, False)), (10240, 8192, 4, (64, 8, True)), (8192, 12288, 4, (128, 4, True)),
    # several rounds of short slices
    (18688, 4096, 1, (64, 4, True)), (18688, 4096, 64, (64, 4, True)), (20480, 8192, 33, (64, 8, True)), (9216, 4096, 32, (64, 4, True)),
    (9216, 4096, 33, (128, 2, False)), (18688, 2048, 5, (64, 2, True)), (18688, 6144, 5, (64, 4, True)), (4098, 14336, 5, (0, 0, False))])
def test_where_decode_products_go(N, K, M, took):
    assert native._part_stream(M, N, K, 256, 5, 0, 64, 512) == took
