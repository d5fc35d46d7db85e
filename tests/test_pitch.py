"""Large weights whose rows lie 128 bytes further apart (ops/pitch.py): the same products and embeddings as from dense rows."""
import pytest
import torch

from rag_llm_k8s_amd.ops import pitch

DEV = "cuda"


@pytest.mark.parametrize("rows,row_bytes,itemsize,gap", [
    (8192, 8192, 2, True), (8191, 8192, 2, False), (28672, 12288, 2, True), (28672, 14336, 2, False), (16384, 4096, 2, True),
    (28672, 16384, 2, False), (4096, 4096, 1, True), (4095, 4096, 1, False), (28672, 8192, 1, False), (28672, 8192, 4, False)])
def test_rule(rows, row_bytes, itemsize, gap):
    assert pitch.wants_gap(rows, row_bytes, itemsize) == gap


def test_host_weights_stay_dense():
    w = torch.zeros(32768, 2048, dtype=torch.bfloat16)
    assert pitch.pitched(w) is w


def _with_gap(w):
    out = torch.zeros(w.shape[0], w.shape[1] + pitch.GAP // w.element_size(), dtype=w.dtype, device=w.device)[:, :w.shape[1]]
    return out.copy_(w)


def _randn(*shape, scale=1.0):
    g = torch.Generator(device=DEV).manual_seed(sum(shape))
    return (torch.randn(*shape, generator=g, device=DEV) * scale).bfloat16()


def test_gate_and_up_rows_packed_in_place():
    from rag_llm_k8s_amd.ops.reference import pack_gate_up

    g, u = torch.randn(192, 40), torch.randn(192, 40)
    for out in (torch.zeros(384, 40), torch.full((384, 104), 7.0)[:, :40], torch.zeros(384, 40, dtype=torch.bfloat16)):
        assert pack_gate_up(g, u, out=out) is out and torch.equal(out, pack_gate_up(g, u).to(out.dtype))
    assert pitch.empty_rows(32768, 2048, torch.bfloat16, "cpu").is_contiguous()


@pytest.mark.gpu
@pytest.mark.parametrize("source", ["cpu", DEV])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_loaded_gate_and_up_rows(source, dtype):
    """Into rows with a gap from any device and type, and nowhere else."""
    from rag_llm_k8s_amd.ops.reference import pack_gate_up

    g, u = torch.randn(8192, 2048).to(source, dtype), torch.randn(8192, 2048).to(source, dtype)
    out = pitch.empty_rows(16384, 2048, torch.bfloat16, DEV)
    whole = out.as_strided((16384, 2112), (2112, 1)).fill_(7.0)
    assert out.stride() == (2112, 1) and torch.equal(pack_gate_up(g, u, out=out), pack_gate_up(g, u).to(DEV, torch.bfloat16))
    assert bool((whole[:, 2048:] == 7.0).all())


@pytest.mark.gpu
def test_pitched_copy():
    w = _randn(16384, 2048)
    p = pitch.pitched(w)
    assert p.stride() == (2048 + 64, 1) and torch.equal(p, w) and pitch.pitched(p) is p
    small = w[:16383]
    assert pitch.pitched(small) is small and pitch.pitched(w[None]).dim() == 3


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 3, 4, 5, 16, 17, 64, 65, 200, 600])
def test_products_from_rows_with_a_gap(M):
    from rag_llm_k8s_amd.ops import native
    from rag_llm_k8s_amd.ops.fp8 import Fp8Weight, quantize_weight

    x, w = _randn(M, 2048), _randn(4096, 2048, scale=2048 ** -0.5)
    p = _with_gap(w)
    for kw in (dict(), dict(out_f32=True), dict(epi="silu_mul"), dict(epi="resid", resid=_randn(M, 4096))):
        assert torch.equal(native.gemm(x, w, **kw), native.gemm(x, p, **kw)), kw
    q = quantize_weight(w)
    qp = Fp8Weight(_with_gap(q.w8.view(torch.uint8)).view(torch.float8_e4m3fn), q.scale)
    assert torch.equal(native.gemm_fp8(x, q, epi="silu_mul"), native.gemm_fp8(x, qp, epi="silu_mul"))
    assert torch.equal(native.gemm_fp8(x, q), native.gemm_fp8(x, qp))
    if M <= 64:
        assert torch.equal(native.gemm_part(x, w), native.gemm_part(x, p))
        assert torch.equal(native.gemm_part(x, q), native.gemm_part(x, qp))


# weights from 16384 rows on (the weight stream's gate/up and wide products), each of the rule's distances
@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 5, 16, 17, 33, 64, 65, 300])
@pytest.mark.parametrize("N,K", [(16384, 2048), (16512, 4096), (16384, 6144)])
def test_wide_products_from_rows_with_a_gap(M, N, K):
    from rag_llm_k8s_amd.ops import native

    x, w = _randn(M, K), _randn(N, K, scale=K ** -0.5)
    p, par = _with_gap(w), torch.tensor([2.0, 1.2, 0.5, 0.0], device=DEV)
    assert native.use_stream(M, N // 2, K, "silu_mul") == native.use_stream(M, N // 2, K, "glu_clip") == (M <= 64)
    for kw in (dict(), dict(epi="silu_mul"), dict(epi="glu_clip", bias=par)):
        assert torch.equal(native.gemm(x, w, **kw), native.gemm(x, p, **kw)), kw
        if kw.get("epi") and M <= 64:  # (some of these go to the held activations)
            assert torch.equal(native.gemm(x, w, path=5, **kw), native.gemm(x, p, path=5, **kw)), kw
    if M <= 64:
        assert torch.equal(native.gemm_part(x, w), native.gemm_part(x, p))


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 7, 8, 64])
@pytest.mark.parametrize("N,K", [(32768, 2048), (32776, 4096)])
def test_vocabulary_with_a_gap(M, N, K):
    """fp32 logits take the weight stream at any row count then, in sums no longer than the kernel's that dense rows take below
    eight: its error against 64 bits, give or take what a mean of 32768 squares says of it (0.4 %) and x, which they share."""
    from rag_llm_k8s_amd.ops import native

    x, w = _randn(M, K), _randn(N, K, scale=K ** -0.5)
    ref = x.double() @ w.double().t()
    err = [((native.gemm(x, t, out_f32=True).double() - ref).norm() / ref.norm()).item() for t in (w, _with_gap(w))]
    assert err[1] <= 1.03 * err[0] < 1e-6


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 4, 7])
@pytest.mark.parametrize("K", [1024, 3072, 6144])
def test_vocabulary_sums_with_a_gap_are_no_longer(M, K):
    """Widths at which the weight stream would sum over more of K keep the dense weight's kernel, bit for bit."""
    from rag_llm_k8s_amd.ops import native

    x, w = _randn(M, K), _randn(32768, K, scale=K ** -0.5)
    y, z = native.gemm(x, w, out_f32=True), native.gemm(x, _with_gap(w), out_f32=True)
    if K % 2048:
        assert torch.equal(y, z)
    else:
        ref = x.double() @ w.double().t()
        err = [((t.double() - ref).norm() / ref.norm()).item() for t in (z, y)]
        assert err[0] <= err[1] < 1e-6


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_embedding_rows_with_a_gap(dtype):
    from rag_llm_k8s_amd.ops import seq_native

    t = _randn(100, 256).to(dtype)
    ids = torch.tensor([0, 99, 5, -3, 1000], dtype=torch.int32, device=DEV)
    assert torch.equal(seq_native.embed_residual(ids.clone(), t), seq_native.embed_residual(ids.clone(), _with_gap(t)))
    with pytest.raises(ValueError):
        seq_native.embed_residual(ids.clone(), t[:, 2:250])


@pytest.mark.gpu
def test_mlp_engine_with_a_gap():
    from rag_llm_k8s_amd.ops import native

    H, I = 4096, 14336
    w, d = _randn(2 * I, H, scale=H ** -0.5), _randn(H, I, scale=I ** -0.5)
    p, x, h = _with_gap(w), _randn(1, H), _randn(1, H)
    if not native.mlp_engine_ok(1, w, d):
        pytest.skip("no MLP engine on this device")
    off = lambda gap, start: torch.zeros(2 * I, H + gap, dtype=torch.bfloat16, device=DEV)[:, start:start + H]
    assert native.mlp_engine_ok(1, p, d) and native.mlp_engine_ok(1, off(8, 0), d) and native.mlp_engine_ok(1, off(8, 8), d)
    assert not native.mlp_engine_ok(1, off(8, 1), d) and not native.mlp_engine_ok(1, off(4, 0), d)  # rows off 16 bytes
    assert torch.equal(native.mlp_engine(x, w, d, h.clone()), native.mlp_engine(x, p, d, h.clone()))
