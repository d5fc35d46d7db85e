"""Launches that took two before, bit for bit: embedding and first norm, norms of selected rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def native():
    from rag_llm_k8s_amd.ops import native

    return native


def _i32(v):
    return torch.tensor(v, dtype=torch.int32, device=DEV)


# one vector, a thread's one, two and four of them, a remainder
@pytest.mark.parametrize("H", [8, 384, 2048, 4104, 8192])
@pytest.mark.parametrize("carry", [False, True])
def test_embed_rmsnorm(native, H, carry):
    table, w = (torch.randn(50, H, device=DEV).bfloat16(), torch.randn(H, device=DEV).bfloat16())
    ids = _i32([0, 49, 7, 7, -3, 1000])  # (clamped)
    kw = dict(carry=_i32([-1, 2, -1, 0, -1, 1]), prev=_i32([11, 60, 13])) if carry else {}
    ids2 = ids.clone()
    h = native.embed(ids, table, **kw)
    h2, xn = native.embed_rmsnorm(ids2, table, w, 1e-5, **kw)
    assert torch.equal(h, h2) and torch.equal(ids, ids2) and torch.equal(xn, native.rmsnorm(h, w, 1e-5))


def test_embed_rmsnorm_refuses_wide_rows(native):
    with pytest.raises(ValueError):
        native.embed_rmsnorm(_i32([0]), torch.zeros(2, 8200, device=DEV).bfloat16(), torch.zeros(8200, device=DEV).bfloat16(), 1e-5)


def test_embeddings_refuse_rows_with_gaps(native):
    """Both read row id at id * H."""
    wide, w = torch.randn(50, 448, device=DEV).bfloat16(), torch.randn(384, device=DEV).bfloat16()
    for table in (wide[:, :384], wide[:, :384].t().contiguous().t()):
        with pytest.raises(ValueError):
            native.embed(_i32([0, 3]), table)
        with pytest.raises(ValueError):
            native.embed_rmsnorm(_i32([0, 3]), table, w, 1e-5)
    assert torch.equal(native.embed_rmsnorm(_i32([0, 0]), wide[7:8, :384], w, 1e-5)[0], wide[7, :384].expand(2, -1))  # one row has none


@pytest.mark.parametrize("H", [384, 4096, 8192])
@pytest.mark.parametrize("rows", [[0], [69, 3, 3, 0]])
def test_norms_of_rows(native, H, rows):
    x, w = torch.randn(70, H, device=DEV).bfloat16(), torch.randn(H, device=DEV).bfloat16()
    idx = _i32(rows)
    assert torch.equal(native.rmsnorm_rows(x, idx, w, 1e-5), native.rmsnorm(native.gather_rows(x, idx), w, 1e-5))
    for S in (1, 3, 9):
        for rounded in (True, False):
            P, h = torch.randn(S, 70, H, device=DEV), x.clone()
            part = native.add_partials_rmsnorm(P, h, w, 1e-5, rounded=rounded, rows=idx)
            assert torch.equal(h, x)
            assert torch.equal(part, native.add_partials_rmsnorm(P, h, w, 1e-5, rounded=rounded)[idx.long()])


@pytest.mark.parametrize("W", [384, 4096, 4224])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_dense_tables_may_start_anywhere(W, dtype):
    from rag_llm_k8s_amd.ops import seq_native

    t, w, ids = torch.randn(20, W, device=DEV).to(dtype), torch.randn(W, device=DEV), _i32([0, 19, 7])
    off = 8 // t.element_size()  # 8 bytes
    moved = torch.cat([t.new_zeros(off), t.flatten()])[off:].view(20, W)
    one = torch.as_strided(moved, (1, W), (4, 1), moved.storage_offset() + 7 * W)  # a single row has no distance to another
    assert moved.data_ptr() % 16 and torch.equal(seq_native.embed_residual(ids, moved), seq_native.embed_residual(ids, t))
    assert torch.equal(seq_native.embed_residual(_i32([0]), one), t[7:8].float())
    for a, b in zip(seq_native.embed_norm(ids, moved, w, 1e-5, W), seq_native.embed_norm(ids, t, w, 1e-5, W)):
        assert torch.equal(a, b)
    for table in (torch.as_strided(t, (9, W), (W + 4, 1)), torch.as_strided(t, (9, W), (8, 1)), moved[:, :W - 8]):
        with pytest.raises((ValueError, RuntimeError)):
            seq_native.embed_residual(ids, table)
        with pytest.raises((ValueError, RuntimeError)):
            seq_native.embed_norm(ids, table, w[:table.shape[1]], 1e-5, 8)


# a vector, a thread's one on 256 and 512 threads, padded columns, rows wider than one launch takes
@pytest.mark.parametrize("W,n", [(8, 8), (384, 380), (2048, 2048), (2056, 2050), (4096, 4096), (4224, 4200)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("carry", [False, True])
def test_embed_norm(W, n, dtype, carry):
    from rag_llm_k8s_amd.ops import seq_native

    table, w = torch.randn(50, W + 64, device=DEV).to(dtype)[:, :W], torch.randn(W, device=DEV)
    ids = _i32([0, 49, 7, 7, -3, 1000])
    kw = dict(carry=_i32([-1, 2, -1, 0, -1, 1]), prev=_i32([11, 60, 13])) if carry else {}
    ids2 = ids.clone()
    h = seq_native.embed_residual(ids, table, **kw)
    h2, xn = seq_native.embed_norm(ids2, table, w, 1e-5, n, **kw)
    assert torch.equal(h, h2) and torch.equal(ids, ids2)
    assert torch.equal(xn, seq_native.residual_norm(h, None, None, w, 1e-5, n, dtype))
