"""The native encoder forward (csrc/kernels/encoder.hip) against the layer-by-layer path."""
import numpy as np
import pytest
import torch

from rag_llm_k8s_amd.engine.encoder_engine import EmbeddingEngine
from rag_llm_k8s_amd.models import encoder as E

pytestmark = pytest.mark.gpu
DEV = "cuda"


def model(pooling, hidden=256, heads=4, inter=512, kind="bert"):
    cfg = E.EncoderConfig(model_type=kind, vocab_size=500, hidden_size=hidden, num_hidden_layers=2, num_attention_heads=heads,
                          intermediate_size=inter, max_position_embeddings=512, pooling=pooling,
                          pad_token_id=1 if kind == "xlm-roberta" else 0)
    return E.EncoderModel(cfg, E.EncoderWeights.random(cfg, DEV, seed=3), DEV)


@pytest.mark.parametrize("pooling,kind", [("cls", "xlm-roberta"), ("mean", "bert")])
@pytest.mark.parametrize("lens", [[1], [14], [63, 1], [30, 35], [129, 7, 300, 64, 1], [200] * 9])
def test_native_forward_is_the_layered_one(native, pooling, kind, lens):
    """Bit for bit, one launch plan in both: few rows (skinny products), past 64 (tiles), rows written where they belong."""
    m = model(pooling, kind=kind)
    ids = np.random.RandomState(sum(lens)).randint(0, 500, sum(lens)).astype(np.int32)
    ref = m.forward_packed(torch.from_numpy(ids).to(DEV), lens)
    out = torch.full((len(lens) + 2, 256), 9.0, device=DEV)
    rows = np.random.RandomState(1).permutation(len(lens)) + 1
    m.embed_into(ids, np.asarray(lens, dtype=np.int64), out, rows)
    assert native.encoder_forward_ok(m.cfg, m.w)
    assert torch.equal(out[torch.from_numpy(rows).to(DEV)], ref)
    assert bool((out[0] == 9.0).all()) and bool((out[-1] == 9.0).all())


def test_narrow_encoder_of_a_large_batch(native):
    """128 columns (two K-tiles a product) at the tokens of a full ingest batch."""
    m = model("mean", hidden=128)
    lens = [512] * 100
    ids = np.random.RandomState(4).randint(0, 500, sum(lens)).astype(np.int32)
    out = torch.zeros(len(lens), 128, device=DEV)
    m.embed_into(ids, np.asarray(lens, dtype=np.int64), out, np.arange(len(lens)))
    assert torch.equal(out, m.forward_packed(torch.from_numpy(ids).to(DEV), lens))


def test_engine_order_and_odd_outputs(native):
    """Batches cut by tokens, unsorted lengths; an output that the native call does not take (strided columns) still works."""
    m = model("mean")
    eng = EmbeddingEngine(m, None, max_batch_tokens=150)
    r = np.random.RandomState(0)
    lists = [r.randint(0, 500, n).tolist() for n in (5, 120, 33, 1, 64, 90)]
    got = eng.embed_ids(lists)
    for x, y in zip(lists, got):
        one = m.forward_packed(torch.tensor(x, dtype=torch.int32, device=DEV), [len(x)])[0]
        assert torch.nn.functional.cosine_similarity(one, y, dim=0).item() > 0.999
    cols = torch.zeros(256, len(lists), device=DEV).t()
    ids, lens = np.concatenate(lists).astype(np.int32), np.array([len(x) for x in lists], dtype=np.int32)
    eng.embed_flat(ids, lens, cols)
    assert torch.equal(cols, got)


def test_ids_of_another_type_are_refused(native):
    m = model("mean")
    out = torch.zeros(2, 256, device=DEV)
    with pytest.raises(ValueError):
        EmbeddingEngine(m, None).embed_flat(np.arange(20, dtype=np.int64), np.array([15, 5], dtype=np.int32), out)
    assert not out.any()


def test_edited_weights(native):
    """Weights whose addresses alone would mislead the native call: rows with gaps give what they give without, a transposed
    matrix is refused as the layered path refuses it, one on the host is not taken; no token type row is."""
    ids, lens, row = np.arange(5, 105, dtype=np.int32), np.array([100], dtype=np.int64), np.array([0])
    ref, out = torch.zeros(1, 256, device=DEV), torch.zeros(1, 256, device=DEV)
    m = model("mean")
    m.embed_into(ids, lens, ref, row)
    m.w.layers[1]["wi"] = torch.cat([m.w.layers[1]["wi"]] * 2, 1)[:, :256]
    assert not native.encoder_forward_ok(m.cfg, m.w)
    m.embed_into(ids, lens, out, row)
    assert torch.equal(out, ref)
    m.w.layers[0]["wo"] = m.w.layers[0]["wo"].t()
    with pytest.raises(ValueError):
        m.embed_into(ids, lens, out, row)
    m = model("mean")
    m.w.type_row = None
    m.embed_into(ids, lens, out, row)
    assert native.encoder_forward_ok(m.cfg, m.w) and not torch.equal(out, ref)
    assert torch.equal(out, m.forward_packed(torch.from_numpy(ids).to(DEV), [100]))
    m.w.layers[0]["ln1_g"] = m.w.layers[0]["ln1_g"].cpu()
    assert not native.encoder_forward_ok(m.cfg, m.w)


@pytest.mark.parametrize("lens", [[14], [14, 30], [300] * 4])
def test_host_ids_are_not_frozen_into_a_graph(native, lens):
    """Ids read from host memory when the call is made: a graph would repeat them whatever the caller's buffer holds by then, so
    a capture is refused (and given up by its owner); the same call afterwards works."""
    m = model("mean")
    ids, out = np.arange(5, 5 + sum(lens), dtype=np.int32) % 500, torch.zeros(len(lens), 256, device=DEV)
    args = ids, np.asarray(lens, dtype=np.int64), out, np.arange(len(lens))
    m.embed_into(*args)
    want = out.clone()
    out.zero_()
    torch.cuda.synchronize()
    with pytest.raises(RuntimeError):
        with torch.cuda.graph(torch.cuda.CUDAGraph()):
            m.embed_into(*args)
    m.embed_into(*args)
    assert torch.equal(out, want)
