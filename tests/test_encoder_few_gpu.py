"""One short sequence through csrc/kernels/encoder_few.hip against the seven launches a layer and against 64 bits."""
import numpy as np
import pytest
import torch

from rag_llm_k8s_amd.models import encoder as E

pytestmark = pytest.mark.gpu
DEV = "cuda"
F64 = torch.float64


def exact(c, w, ids, first):
    """[1, H] in 64 bits."""
    def lin(x, a, b):
        return x @ a.to(F64).t() + b.to(F64)

    def norm(x, g, b):
        m = x.mean(-1, keepdim=True)
        return (x - m) / ((x - m).pow(2).mean(-1, keepdim=True) + c.layer_norm_eps).sqrt() * g.to(F64) + b.to(F64)

    T, H, nh = len(ids), c.hidden_size, c.num_attention_heads
    x = w.word[ids].to(F64) + w.pos[first:first + T].to(F64)
    h = norm(x if w.type_row is None else x + w.type_row.to(F64), w.ln_g, w.ln_b)
    for L in w.layers:
        q, k, v = lin(h, L["wqkv"], L["bqkv"]).view(T, 3, nh, H // nh).permute(1, 2, 0, 3)
        a = torch.softmax(q @ k.transpose(1, 2).contiguous() * (H // nh) ** -0.5, -1) @ v.contiguous()
        h = norm(h + lin(a.permute(1, 0, 2).reshape(T, H), L["wo"], L["bo"]), L["ln1_g"], L["ln1_b"])
        f = torch.nn.functional.gelu(lin(h, L["wi"], L["bi"]))
        h = norm(h + lin(f, L["wo2"], L["bo2"]), L["ln2_g"], L["ln2_b"])
    p = {"cls": h[0], "mean": h.mean(0), "last": h[-1]}[c.pooling]
    return (p / p.norm() if c.normalize else p)[None]


# one row, rows below, at and past a 16-row tile, the most; one K-step a wave and sixteen (twice over); both head sizes; the
# narrowest and the widest rows
@pytest.mark.parametrize("T", [1, 2, 15, 16, 17, 31, 32])
@pytest.mark.parametrize("hidden,heads,inter,pooling,kind", [(128, 4, 128, "mean", "bert"), (384, 12, 1536, "cls", "bert"),
                                                             (512, 8, 2176, "last", "xlm-roberta"), (1024, 16, 4096, "cls", "bert"),
                                                             (640, 10, 8320, "mean", "xlm-roberta")])
def test_short_sequence(native, monkeypatch, T, hidden, heads, inter, pooling, kind):
    cfg = E.EncoderConfig(model_type=kind, vocab_size=500, hidden_size=hidden, num_hidden_layers=2, num_attention_heads=heads,
                          intermediate_size=inter, max_position_embeddings=64, pooling=pooling,
                          pad_token_id=1 if kind == "xlm-roberta" else 0)
    m = E.EncoderModel(cfg, E.EncoderWeights.random(cfg, DEV, seed=T), DEV)
    if T == 2:
        m.w.type_row = None
    monkeypatch.setattr(native, "FEW_SIZE", 10 ** 9)
    assert native.encoder_pointers(cfg, m.w) is not None  # else the call below goes layer by layer
    ids = np.random.RandomState(T).randint(0, 500, T + 1).astype(np.int32)[1:]
    assert native.encoder_few_ok(cfg, T, 1) and not native.encoder_few_ok(cfg, 33, 1) and not native.encoder_few_ok(cfg, T, 2)
    out = torch.full((3, hidden), 9.0, device=DEV)
    m.embed_into(ids, np.array([T], dtype=np.int64), out, np.array([1]))
    assert bool((out[0] == 9.0).all()) and bool((out[2] == 9.0).all())
    dev = torch.from_numpy(ids).to(DEV)
    assert torch.equal(m.forward_packed(dev, [T])[0], out[1])
    monkeypatch.setattr(native, "FEW_ROWS", 0)
    seven = m.forward_packed(dev, [T])
    ref = exact(cfg, m.w, dev.long(), m.first_position)
    err = [((y.to(F64) - ref).norm() / ref.norm()).item() for y in (out[1:2], seven)]
    # two layers of bf16 activations (2^-9 a rounding, a dozen of them in a row); sums kept in fp32 up to the norm: not further off
    assert err[0] < 0.01 and err[0] < 1.3 * err[1] + 1e-4, err


# the widths between (a kernel for each), and as many columns of a down projection as the call takes (encoder_pointers)
@pytest.mark.parametrize("T", [3, 17])
@pytest.mark.parametrize("hidden,heads,inter", [(256, 8, 256), (768, 12, 3072), (896, 14, 1152), (384, 6, 2048), (128, 2, 16256)])
def test_every_width(native, monkeypatch, T, hidden, heads, inter):
    test_short_sequence(native, monkeypatch, T, hidden, heads, inter, "mean", "bert")


@pytest.mark.parametrize("T", [3, 17])
def test_more_columns_than_the_call_takes(native, T):
    cfg = E.EncoderConfig(model_type="bert", vocab_size=500, hidden_size=128, num_hidden_layers=2, num_attention_heads=2,
                          intermediate_size=32768, max_position_embeddings=64, pooling="mean")
    m = E.EncoderModel(cfg, E.EncoderWeights.random(cfg, DEV, seed=T), DEV)
    assert native.encoder_pointers(cfg, m.w) is None
    ids = torch.from_numpy(np.random.RandomState(T).randint(0, 500, T).astype(np.int32)).to(DEV)
    ref = exact(cfg, m.w, ids.long(), m.first_position)
    assert ((m.forward_packed(ids, [T]).to(F64) - ref).norm() / ref.norm()).item() < 0.01  # (test_short_sequence)


def test_no_layers(native):
    """Embeddings, their norm and the pooling only: the launches of a layer have nothing to begin with."""
    cfg = E.EncoderConfig(model_type="bert", vocab_size=500, hidden_size=128, num_hidden_layers=0, num_attention_heads=4,
                          intermediate_size=128, max_position_embeddings=64, pooling="mean")
    m = E.EncoderModel(cfg, E.EncoderWeights.random(cfg, DEV, seed=1), DEV)
    ids, out = np.arange(5, 12, dtype=np.int32), torch.zeros(1, 128, device=DEV)
    m.embed_into(ids, np.array([7], dtype=np.int64), out, np.array([0]))
    ref = exact(cfg, m.w, torch.from_numpy(ids).to(DEV).long(), m.first_position)
    # rows rounded to bf16 (2^-8 of a value), pooled and scaled
    assert ((out.to(F64) - ref).norm() / ref.norm()).item() < 2.0 ** -8


def test_library_refuses_what_it_cannot_take(native):
    """Nothing is launched for more rows or columns than there is room for, a head size of its own, or no ids."""
    import ctypes
    L, c = native._lib.lib(), native._lib.EncoderCall()
    c.few, c.n_layers, c.B, c.T, c.H, c.I, c.heads = 1, 1, 1, 4, 256, 512, 4
    c.ids = 16
    for field, bad in (("T", 33), ("H", 1152), ("heads", 2), ("heads", 3), ("I", 100), ("B", 2), ("n_layers", 0), ("ids", None)):
        keep = getattr(c, field)
        setattr(c, field, bad)
        assert L.ragk_encoder_forward(ctypes.byref(c), 0) != 0, field
        setattr(c, field, keep)


def test_integers_as_arguments(native):
    for n in (1, 959, 960, 961, 3840):
        src = np.random.RandomState(n).randint(-2 ** 31, 2 ** 31 - 1, n).astype(np.int32)
        dst = torch.full((n + 2,), 7, dtype=torch.int32, device=DEV)
        assert native._lib.lib().ragk_put_ints(src.ctypes.data, n, dst.data_ptr() + 4, native.stream_ptr()) == 0
        assert dst[1:-1].tolist() == src.tolist() and int(dst[0]) == int(dst[-1]) == 7


# one call of layers and several, the last of one layer, two, three
@pytest.mark.parametrize("layers", [1, 3, 4, 5, 6])
def test_layers_in_several_calls(native, monkeypatch, layers):
    cfg = E.EncoderConfig(model_type="bert", vocab_size=500, hidden_size=128, num_hidden_layers=layers, num_attention_heads=4,
                          intermediate_size=256, max_position_embeddings=64, pooling="mean")
    m = E.EncoderModel(cfg, E.EncoderWeights.random(cfg, DEV, seed=layers), DEV)
    ids, row, lens = np.arange(5, 17, dtype=np.int32), np.array([0]), np.array([12], dtype=np.int64)
    out, once = torch.zeros(1, 128, device=DEV), torch.zeros(1, 128, device=DEV)
    m.embed_into(ids, lens, out, row)
    monkeypatch.setattr(native, "FEW_LAYERS", layers)
    m.embed_into(ids, lens, once, row)
    assert torch.equal(out, once) and bool(out.any())
    ref = exact(cfg, m.w, torch.from_numpy(ids).to(DEV).long(), m.first_position)
    assert ((out.to(F64) - ref).norm() / ref.norm()).item() < 0.01  # (test_short_sequence; a layer's roundings grow with their number)


@pytest.mark.parametrize("layers,calls", [(2, 0), (3, 0), (4, 1), (24, 7)])
def test_the_last_call_alone_gives_up_the_interpreter_lock(native, monkeypatch, layers, calls):
    """A thread of plain Python keeps the lock for 5 ms each time it is given up: once for all layers, not every three."""
    cfg = E.EncoderConfig(model_type="bert", vocab_size=500, hidden_size=128, num_hidden_layers=layers, num_attention_heads=4,
                          intermediate_size=256, max_position_embeddings=64, pooling="mean")
    m = E.EncoderModel(cfg, E.EncoderWeights.random(cfg, DEV, seed=2), DEV)
    ids, row, lens, out = np.arange(5, 17, dtype=np.int32), np.array([0]), np.array([12], dtype=np.int64), torch.zeros(1, 128, device=DEV)
    python_api, real, took = 4, native._lib.lib(), []  # ctypes' flag of functions that keep the lock

    class Watched:
        def __getattr__(self, name):
            if name == "ragk_encoder_forward":
                took.append("given up")
            return getattr(real, name)

    held = native._lib.held
    monkeypatch.setattr(native._lib, "held", lambda name: (took.append("held"), held(name))[1])
    held("ragk_encoder_forward")
    monkeypatch.setattr(native._lib, "lib", Watched)
    m.embed_into(ids, lens, out, row)
    assert took == ["held"] * calls + ["given up"] and bool(out.any())
    assert held("ragk_encoder_forward")._flags_ & python_api and not real.ragk_encoder_forward._flags_ & python_api


def test_a_weight_of_a_later_call_that_is_not_taken(native):
    """Launches made by then are given up, and the layers go through the checked entry points."""
    cfg = E.EncoderConfig(model_type="bert", vocab_size=500, hidden_size=128, num_hidden_layers=5, num_attention_heads=4,
                          intermediate_size=256, max_position_embeddings=64, pooling="mean")
    m = E.EncoderModel(cfg, E.EncoderWeights.random(cfg, DEV, seed=1), DEV)
    ids, row, lens = np.arange(5, 17, dtype=np.int32), np.array([0]), np.array([12], dtype=np.int64)
    out = torch.zeros(1, 128, device=DEV)
    m.w.layers[4]["wi"] = torch.cat([m.w.layers[4]["wi"]] * 2, 1)[:, :128]
    assert native.encoder_pointers(cfg, m.w, 0, 3) is not None and native.encoder_pointers(cfg, m.w, 3, 5) is None
    m.embed_into(ids, lens, out, row)
    ref = exact(cfg, m.w, torch.from_numpy(ids).to(DEV).long(), m.first_position)
    assert ((out.to(F64) - ref).norm() / ref.norm()).item() < 0.01
    m.w.layers[4]["wi"] = m.w.layers[4]["wi"].half()
    out.fill_(9.0)
    with pytest.raises(ValueError):
        m.embed_into(ids, lens, out, row)
    assert bool((out == 9.0).all())
