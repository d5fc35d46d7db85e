"""The work that a user of the framework has it do, as cases that can be timed and checked.

A retrieval-augmented query goes through four stages, each through its public entry point:

  embed    EmbeddingEngine.embed_flat: token ids of a batch of texts -> unit-norm sentence embeddings
  search   FlatL2Index.search: query embeddings -> distances and ids of the k nearest chunks, on the host
  prefill  DecoderModel.forward over packed prompts: last-row logits and the filled caches
  decode   one decode step of running sequences, captured once as a graph and replayed per step, as the
           serving engine does: logits, with the step's token appended to the caches

Decoders have the widths, heads and feed-forward sizes of the layer benchmark (utils/layer_bench.SIZES: "4k" are those
of an 8B Llama, "2k" a model of half the width), four layers each and its vocabulary. Encoders are whole.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

from rag_llm_k8s_amd.engine.encoder_engine import EmbeddingEngine
from rag_llm_k8s_amd.engine.llm_engine import no_cyclic_gc
from rag_llm_k8s_amd.index.flat import FlatL2Index
from rag_llm_k8s_amd.models import encoder as E
from rag_llm_k8s_amd.models import llama as L
from rag_llm_k8s_amd.models import niduvik as N
from rag_llm_k8s_amd.models import rolesun as R
from rag_llm_k8s_amd.models.base import StepInput
from rag_llm_k8s_amd.ops.backend import AttnMeta
from rag_llm_k8s_amd.utils import layer_bench, layer_bench_rolesun

DEV = "cuda"
PAGE = 64
MAX_LEN = 8192  # longest context the decode workspaces are sized for (the serving benchmark's limit)
F64 = torch.float64
ENCODERS = {"minilm": E.minilm_l6, "bge_m3": E.bge_m3}


def listed():
    return [
        # the question of one /query request, embedded on its own
        dict(name="embed_query", path="embed", model="minilm", seqs=1, tokens=14),
        # ingest: chunks of about 1000 words through the encoder that the reference deployment uses
        dict(name="embed_chunks", path="embed", model="bge_m3", seqs=12, tokens=1330),
        # the question against the headline benchmark's 10000 chunks
        dict(name="search_query", path="search", rows=10000, dim=384, seqs=1, k=4),
        # a batch of concurrent questions against a large collection
        dict(name="search_batch", path="search", rows=500000, dim=1024, seqs=32, k=5),
        # a short question without retrieved context
        dict(name="prefill_short", path="prefill", family="llama", size="4k", seqs=1, tokens=300),
        # prompts with four retrieved chunks in them, as a full serving step packs them
        dict(name="prefill_rag", path="prefill", family="llama", size="4k", seqs=3, tokens=5192),
        # a batch of unequal prompts on the smaller width (shaped attention and state space layers)
        dict(name="prefill_niduvik", path="prefill", family="niduvik", size="2k", seqs=5, tokens=1900),
        # one prompt of an odd length (latent attention)
        dict(name="prefill_rolesun", path="prefill", family="rolesun", size="4k", seqs=1, tokens=1777),
        # one user's answer, token by token
        dict(name="decode_one", path="decode", family="llama", size="4k", dtype="bf16", seqs=1, tokens=5267),
        # the headline benchmark's 32 concurrent answers
        dict(name="decode_batch", path="decode", family="llama", size="4k", dtype="bf16", seqs=32, tokens=5267),
        # an uneven handful of answers from fp8 weights
        dict(name="decode_fp8", path="decode", family="llama", size="4k", dtype="fp8", seqs=11, tokens=2500),
        # concurrent answers of a model with recurrent layers
        dict(name="decode_niduvik", path="decode", family="niduvik", size="4k", dtype="bf16", seqs=17, tokens=3000),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    path = rng.choice(["embed", "search", "prefill", "prefill", "decode", "decode"])
    if path == "embed":
        model = rng.choice(["minilm", "bge_m3"])
        tokens = _log_int(rng, 5, 256 if model == "minilm" else 1500)
        return dict(path=path, model=model, seqs=_log_int(rng, 1, max(1, min(256, 16000 // tokens))), tokens=tokens)
    if path == "search":
        dim = rng.choice([384, 1024])
        return dict(path=path, rows=_log_int(rng, 1000, 500000), dim=dim, seqs=_log_int(rng, 1, 32), k=rng.randint(1, 10))
    family, size = rng.choice(["llama", "llama", "niduvik", "rolesun"]), rng.choice(["2k", "4k"])
    if path == "prefill":
        tokens = _log_int(rng, 20, 5500)
        most = (14000 if family == "llama" else 7000) // tokens
        return dict(path=path, family=family, size=size, seqs=_log_int(rng, 1, max(1, min(32, most))), tokens=tokens)
    dtype = rng.choice(["bf16", "bf16", "fp8"]) if family == "llama" else "bf16"
    return dict(path=path, family=family, size=size, dtype=dtype, seqs=_log_int(rng, 1, 64), tokens=_log_int(rng, 64, 6000))


def lengths(case):
    """The first sequence has the case's length, the others between 60 % of it and all of it."""
    r = random.Random(case["seqs"] * 100003 + case["tokens"])
    n = case["tokens"]
    return [n] + [r.randint(max(1, 3 * n // 5), n) for _ in range(case["seqs"] - 1)]


# ------------------------------------------------------------------------------------- weights and inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape, dtype=torch.bfloat16, scale=1.0):
    return (torch.randn(*shape, generator=g, device=DEV) * scale).to(dtype)


def _config(case):
    s = layer_bench.SIZES[case["size"]]
    make = {"llama": layer_bench.llama_config, "niduvik": layer_bench.niduvik_config, "rolesun": layer_bench_rolesun.config}
    return make[case["family"]](s)


def _llama_weights(c, g):
    """Checkpoint tensors of random weights: unit-variance activations stay of that order through the layers."""
    H, I, D = c.hidden_size, c.intermediate_size, c.head_dim
    kv = c.num_key_value_heads * D
    sd = {"model.embed_tokens.weight": _randn(g, c.vocab_size, H), "lm_head.weight": _randn(g, c.vocab_size, H, scale=H ** -0.5),
          "model.norm.weight": 1 + _randn(g, H, scale=0.1)}
    for i in range(c.num_hidden_layers):
        p = "model.layers.%d." % i
        for n, rows, cols in (("self_attn.q_proj", H, H), ("self_attn.k_proj", kv, H), ("self_attn.v_proj", kv, H),
                              ("self_attn.o_proj", H, H), ("mlp.gate_proj", I, H), ("mlp.up_proj", I, H), ("mlp.down_proj", H, I)):
            sd[p + n + ".weight"] = _randn(g, rows, cols, scale=cols ** -0.5)
        for n in ("input_layernorm", "post_attention_layernorm"):
            sd[p + n + ".weight"] = 1 + _randn(g, H, scale=0.1)
    return sd


def _encoder_weights(c, g):
    H, I = c.hidden_size, c.intermediate_size
    e = "embeddings."
    sd = {e + "word_embeddings.weight": _randn(g, c.vocab_size, H, scale=0.5),
          e + "position_embeddings.weight": _randn(g, c.max_position_embeddings, H, scale=0.5),
          e + "token_type_embeddings.weight": _randn(g, c.type_vocab_size, H, scale=0.5)}

    def norm(p):
        sd[p + ".weight"], sd[p + ".bias"] = 1 + _randn(g, H, scale=0.05), _randn(g, H, scale=0.05)

    norm(e + "LayerNorm")
    for i in range(c.num_hidden_layers):
        p = "encoder.layer.%d." % i
        for n, rows, cols in (("attention.self.query", H, H), ("attention.self.key", H, H), ("attention.self.value", H, H),
                              ("attention.output.dense", H, H), ("intermediate.dense", I, H), ("output.dense", H, I)):
            sd[p + n + ".weight"] = _randn(g, rows, cols, scale=cols ** -0.5)
            sd[p + n + ".bias"] = _randn(g, rows, scale=0.05)
        norm(p + "attention.output.LayerNorm")
        norm(p + "output.LayerNorm")
    return sd


_LEAVES = {"vmix": (0.0, 0.0), "dt_bias": (-2.5, 1.0), "A_log": (-1.0, 1.5), "D": (1.0, 0.3), "b": (0.0, 0.5), "rel": (0.0, 0.5)}


def _layered_weights(shapes, g):
    """Checkpoint tensors of the layer-listed families from {name: shape}."""
    sd = {}
    for name, shape in shapes.items():
        leaf = name.split(".")[-1]
        r = torch.randn(shape, generator=g, device=DEV)
        if "norm" in leaf:
            r = 1 + 0.1 * r
        elif leaf in _LEAVES:
            r = _LEAVES[leaf][0] + _LEAVES[leaf][1] * r
        elif leaf == "shift":
            r = torch.sigmoid(r)
        elif leaf == "conv":
            r = r * shape[1] ** -0.5
        elif name != "embed":
            r = r * shape[-1] ** -0.5
        sd[name] = r.to(torch.bfloat16)
    return sd


def _weights(case, g):
    c = _config(case)
    if case["family"] == "llama":
        return c, _llama_weights(c, g)
    return c, _layered_weights((N if case["family"] == "niduvik" else R).tensor_shapes(c), g)


def _model(case, c, sd):
    if case["family"] == "llama":
        w = L.LlamaWeights.from_state_dict(c, sd, DEV)
        return L.LlamaModel(c, w.quantize_fp8() if case.get("dtype") == "fp8" else w, DEV, max_positions=MAX_LEN)
    if case["family"] == "niduvik":
        return N.NiduvikModel(c, N.NiduvikWeights.from_state_dict(c, sd, DEV), DEV)
    return R.RolesunModel(c, R.RolesunWeights.from_state_dict(c, sd, DEV), DEV)


def _pages(lens, seed):
    """Block tables of pages in the scattered order that a running server hands them out in; page 0 is nobody's."""
    need = [-(-n // PAGE) for n in lens]
    order = 1 + np.random.RandomState(seed % (1 << 31)).permutation(sum(need))
    bt = np.zeros((len(lens), max(need)), dtype=np.int64)
    at = 0
    for i, n in enumerate(need):
        bt[i, :n] = order[at:at + n]
        at += n
    return torch.from_numpy(bt), sum(need) + 1


def _i32(x):
    return torch.as_tensor(x, dtype=torch.int32).to(DEV).contiguous()


def _states(model, case):
    """The model's recurrent state buffers."""
    if case["family"] == "niduvik":
        return [t for s in model.ssm for t in (s.conv_state, s.ssm_state)]
    return [model.shift_state] if case["family"] == "rolesun" else []


def _caches(model, num_blocks):
    out = model.allocate_kv_cache(num_blocks)
    return [t for x in out for t in (x if isinstance(x, tuple) else (x,))]


def _fill(case, caches, states, g):
    """Contexts of running sequences: normal numbers of the size that projections of normed rows have."""
    for t in caches:
        t.normal_(generator=g)
        t[0].zero_()
    for t in states:
        t.normal_(generator=g)


def _ids(case, c, n, g):
    return torch.randint(0, c.vocab_size, (n,), generator=g, device=DEV, dtype=torch.int32)


# ------------------------------------------------------------------------------------- prepare
def _prepare_embed(case, seed):
    g, c = _gen(seed), ENCODERS[case["model"]]()
    sd = _encoder_weights(c, g)
    engine = EmbeddingEngine(E.EncoderModel(c, E.EncoderWeights.from_state_dict(c, sd, DEV), DEV), None)
    lens = np.asarray(lengths(case), dtype=np.int32)
    ids = torch.randint(5, c.vocab_size, (int(lens.sum()),), generator=g, device=DEV, dtype=torch.int32).cpu().numpy()
    return dict(case=case, engine=engine, ids=ids, lens=lens)


def _vectors(case, seed):
    """Unit-norm embeddings around topics, and queries near some of them."""
    g, d = _gen(seed), case["dim"]
    topics = torch.randn(64, d, generator=g, device=DEV)

    def some(n, spread):
        t = topics[torch.randint(0, 64, (n,), generator=g, device=DEV)]
        return torch.nn.functional.normalize(t + spread * torch.randn(n, d, generator=g, device=DEV), dim=1)

    return some(case["rows"], 1.0), some(case["seqs"], 0.7)


def _prepare_search(case, seed):
    x, q = _vectors(case, seed)
    index = FlatL2Index(case["dim"], device=DEV, capacity=case["rows"])
    index.add(x)
    return dict(case=case, index=index, q=q)


def _prepare_prefill(case, seed):
    g, lens = _gen(seed), lengths(case)
    c, sd = _weights(case, g)
    model = _model(case, c, sd)
    bt, blocks = _pages(lens, seed)
    caches = _caches(model, blocks)
    model.allocate_state(len(lens) + 1)
    pos = np.concatenate([np.arange(n) for n in lens])
    seq = np.repeat(np.arange(len(lens)), lens)
    slots = bt.numpy()[seq, pos // PAGE] * PAGE + pos % PAGE
    cu = np.concatenate([[0], np.cumsum(lens)])
    tiles, qtiles = model.prefill_work(lens, DEV)
    meta = AttnMeta("prefill", _i32(lens), _i32(bt), cu_q=_i32(cu), tiles=tiles, qtiles=qtiles, host_kv_lens=lens,
                    host_q_lens=lens, max_kv=MAX_LEN, key_rows=model.key_rows(lens, lens, DEV),
                    states=_i32(np.arange(1, len(lens) + 1)))
    inp = StepInput(_ids(case, c, len(pos), g), _i32(pos), _i32(slots), meta, _i32(cu[1:] - 1))
    return dict(case=case, model=model, inp=inp, caches=caches, states=_states(model, case))


def _prepare_decode(case, seed):
    g, lens = _gen(seed), lengths(case)
    B = len(lens)
    c, sd = _weights(case, g)
    model = _model(case, c, sd)
    bt, blocks = _pages(lens, seed)
    caches = _caches(model, blocks)
    model.allocate_state(B + 1)
    states = _states(model, case)
    _fill(case, caches, states, g)
    pos = np.asarray(lens) - 1
    slots = bt.numpy()[np.arange(B), pos // PAGE] * PAGE + pos % PAGE
    table = torch.zeros(B, MAX_LEN // PAGE, dtype=torch.int64)
    table[:, :bt.shape[1]] = bt
    pt, mp, ws_o, ws_ml = model.decode_work(MAX_LEN, B)
    meta = AttnMeta("decode", _i32(lens), _i32(table), part_tiles=pt, max_parts=mp, ws_o=ws_o, ws_ml=ws_ml,
                    states=_i32(np.arange(1, B + 1)), max_kv=MAX_LEN)
    inp = StepInput(_ids(case, c, B, g), _i32(pos), _i32(slots), meta)
    before = [t.clone() for t in states]
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        for _ in range(2):
            model.forward(inp)
    torch.cuda.current_stream().wait_stream(stream)
    graph = torch.cuda.CUDAGraph()
    with no_cyclic_gc(), torch.cuda.graph(graph, stream=stream):
        logits = model.forward(inp)
    for t, b in zip(states, before):
        t.copy_(b)
    return dict(case=case, model=model, inp=inp, graph=graph, logits=logits, caches=caches, states=states)


@torch.no_grad()
def prepare(case, seed):
    return {"embed": _prepare_embed, "search": _prepare_search, "prefill": _prepare_prefill,
            "decode": _prepare_decode}[case["path"]](case, int(seed))


# ------------------------------------------------------------------------------------- run
@torch.no_grad()
def run(state):
    path = state["case"]["path"]
    if path == "embed":
        return {"embeddings": state["engine"].embed_flat(state["ids"], state["lens"])}
    if path == "search":
        dist, ids = state["index"].search(state["q"], state["case"]["k"])
        return {"distances": dist, "ids": ids}
    if path == "prefill":
        logits = state["model"].forward(state["inp"])
    else:
        state["graph"].replay()
        logits = state["logits"]
    return {"logits": logits, "caches": state["caches"], "states": state["states"]}


# ------------------------------------------------------------------------------------- work
def work(case):
    path = case["path"]
    if path == "search":
        n, d, q = case["rows"], case["dim"], case["seqs"]
        return {"bytes": 4 * n * d + 4 * q * d + 12 * q * case["k"], "flops": 2 * n * d * q}
    lens = lengths(case)
    T, sq = sum(lens), sum(n * n for n in lens)
    if path == "embed":
        c = ENCODERS[case["model"]]()
        H, nl = c.hidden_size, c.num_hidden_layers
        mats = nl * (4 * H * H + 2 * H * c.intermediate_size)
        return {"bytes": 2 * mats + 2 * T * H + 4 * len(lens) * H, "flops": 2 * mats * T + 4 * nl * sq * H}
    c, B = _config(case), len(lens)
    s = layer_bench.SIZES[case["size"]]
    W, ff, heads, V = s["width"], s["ff"], s["heads"], layer_bench.VOCAB
    mats = flops = memory = 0
    rows = T if path == "prefill" else B
    for i in range(4):
        mats += 3 * W * ff
        if case["family"] == "llama" or (case["family"] == "niduvik" and i % 2 == 0):
            mats += 2 * W * heads * 128 + 2 * W * s["kv_heads"] * 128
            memory += T * 2 * s["kv_heads"] * 128 * 2  # keys and values: written by a prompt, read by a decode step
            flops += 4 * heads * 128 * (sq / 2 if path == "prefill" else T)
        elif case["family"] == "niduvik":
            m = c.layers[i]["mixer"]
            inner, gn = m["heads"] * m["vdim"], m["groups"] * m["state"]
            mats += W * (3 * inner + 2 * gn + m["heads"])
            state = 4 * inner * m["state"]
            memory += B * state * (1 if path == "prefill" else 2)
            flops += 4 * inner * m["state"] * rows
        else:
            rank = c.layers[i]["mixer"]["kv_rank"]
            own = c.layers[i]["mixer"].get("kv_from") is None
            mats += 3 * W * heads * 128 + 2 * W * W + (W * rank if own else 0)
            maps = 2 * heads * 128 * rank
            memory += 2 * maps + (T * rank * 2 if own or path == "decode" else 0)
            flops += 2 * maps * rows + (4 * heads * 128 * sq / 2 if path == "prefill" else 4 * heads * rank * T)
    nbytes = mats * (1 if case.get("dtype") == "fp8" else 2) + memory + 2 * V * W + 2 * rows * W + 4 * B * V
    return {"bytes": nbytes, "flops": flops + 2 * mats * rows + 2 * V * W * B}


def tolerance(case):
    if case["path"] == "search":  # fp32 sums of up to 1024 squares in another order; ids may swap where distances tie
        return {"rel": 2e-6, "max": 1e-5, "differ": 0.01}
    if case["path"] == "embed":
        return {"rel": 0.02, "max": 0.3}
    return {"rel": 0.02, "max": 0.5}


# ------------------------------------------------------------------------------------- the same in 64 bits
def _lin(x, w, b=None, step=4096):
    """x @ w^T (+ b) in 64 bits, a slice of the weight's rows at a time."""
    y = torch.cat([x @ w[i:i + step].to(F64).t() for i in range(0, w.shape[0], step)], 1)
    return y if b is None else y + b.to(F64)


def _rms(x, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def _softmax(s, sink=False):
    """In place over the last dimension; `sink`: one more score of zero in the denominator."""
    m = s.amax(-1, keepdim=True)
    if sink:
        m = m.clamp_min(0)
    s.sub_(m).exp_()
    return s.div_(s.sum(-1, keepdim=True) + (torch.exp(-m) if sink else 0))


def _attend(q, k, v, start, scale, shape=None, window=0, keep=0, sink=False, causal=True, step=512):
    """q [n, H, d] at positions start.., k [m, G, d], v [m, G, e] -> [n, H, e]. shape(scores, distances) -> scores."""
    n, H, _ = q.shape
    m, G, e = v.shape
    out = torch.empty(n, H, e, dtype=F64, device=q.device)
    kt, vt = k.permute(1, 2, 0).contiguous(), v.permute(1, 0, 2).contiguous()
    j = torch.arange(m, device=q.device)
    for a in range(0, n, step):
        z = min(n, a + step)
        dist = torch.arange(start + a, start + z, device=q.device)[:, None] - j[None]
        hide = dist < 0
        if window:
            hide |= (dist >= window) & (j[None] >= keep)
        for g in range(G):
            for h in range(g * (H // G), (g + 1) * (H // G)):
                s = (q[a:z, h] @ kt[g]) * scale
                if shape is not None:
                    s = shape(s, dist.clamp_min(0), h)
                if causal:
                    s.masked_fill_(hide, -math.inf)
                out[a:z, h] = _softmax(s, sink) @ vt[g]
    return out


def _exact_embed(case, seed):
    g, c = _gen(seed), ENCODERS[case["model"]]()
    sd = _encoder_weights(c, g)
    lens = lengths(case)
    ids = torch.randint(5, c.vocab_size, (sum(lens),), generator=g, device=DEV, dtype=torch.int32).long()
    H, nh, eps = c.hidden_size, c.num_attention_heads, c.layer_norm_eps

    def norm(x, p):
        return torch.nn.functional.layer_norm(x, (H,), sd[p + ".weight"].to(F64), sd[p + ".bias"].to(F64), eps)

    def lin(x, p):
        return _lin(x, sd[p + ".weight"], sd[p + ".bias"])

    first = c.pad_token_id + 1 if c.model_type == "xlm-roberta" else 0
    pos = torch.cat([torch.arange(first, first + n) for n in lens]).to(DEV)
    e = "embeddings."
    x = norm(sd[e + "word_embeddings.weight"][ids].to(F64) + sd[e + "position_embeddings.weight"][pos].to(F64)
             + sd[e + "token_type_embeddings.weight"][0].to(F64), e + "LayerNorm")
    for i in range(c.num_hidden_layers):
        p = "encoder.layer.%d." % i
        q, k, v = (lin(x, p + "attention.self." + n).view(-1, nh, H // nh) for n in ("query", "key", "value"))
        o, at = [], 0
        for n in lens:
            s = slice(at, at + n)
            o.append(_attend(q[s], k[s], v[s], 0, (H // nh) ** -0.5, causal=False, step=2048).reshape(n, H))
            at += n
        x = norm(x + lin(torch.cat(o), p + "attention.output.dense"), p + "attention.output.LayerNorm")
        f = torch.nn.functional.gelu(lin(x, p + "intermediate.dense"))
        x = norm(x + lin(f, p + "output.dense"), p + "output.LayerNorm")
    rows, at = [], 0
    for n in lens:
        rows.append(x[at] if c.pooling == "cls" else x[at:at + n].mean(0))
        at += n
    return {"embeddings": torch.nn.functional.normalize(torch.stack(rows), dim=1)}


def _exact_search(case, seed):
    x, q = _vectors(case, seed)
    q = q.to(F64)
    d = torch.cat([((x[i:i + 65536].to(F64) ** 2).sum(1)[None] - 2 * q @ x[i:i + 65536].to(F64).t())
                   for i in range(0, x.shape[0], 65536)], 1) + (q * q).sum(1, keepdim=True)
    v, i = torch.sort(d, dim=1, stable=True)
    return {"distances": v[:, :case["k"]].cpu(), "ids": i[:, :case["k"]].cpu()}


class _Step:
    """The sequences of a prefill or decode step: their new rows, their cached rows before them, and the pages."""

    def __init__(self, case, seed):
        self.case, self.g, self.lens = case, _gen(seed), lengths(case)
        self.new = self.lens if case["path"] == "prefill" else [1] * len(self.lens)
        self.cfg, self.sd = _weights(case, self.g)
        self.bt, self.blocks = _pages(self.lens, seed)
        self.pos = torch.cat([torch.arange(n - k, n) for n, k in zip(self.lens, self.new)]).to(DEV)
        self.at = np.concatenate([[0], np.cumsum(self.new)])

    def start(self, caches, states):
        """What prepare() puts into the caches and states, then the step's tokens."""
        caches = [torch.zeros(self.blocks, *s, dtype=torch.bfloat16, device=DEV) for s in caches]
        states = [torch.zeros(*s, device=DEV) for s in states]
        if self.case["path"] == "decode":
            _fill(self.case, caches, states, self.g)
        self.ids = _ids(self.case, self.cfg, len(self.pos), self.g).long()
        return [t.to(F64) for t in caches], [t.to(F64) for t in states]

    def rows(self, i):
        return slice(int(self.at[i]), int(self.at[i + 1]))

    def append(self, cache, rows):
        """Each sequence's rows [n, ...] into its pages [blocks, G, 64, d] (or [blocks, 64, d]); yields all its rows."""
        out = []
        for i, n in enumerate(self.lens):
            p = torch.arange(n - self.new[i], n, device=DEV)
            b = self.bt[i].to(DEV)
            if cache.dim() == 4:
                cache[b[p // PAGE], :, p % PAGE] = rows[self.rows(i)]
                t = cache[b[:-(-n // PAGE)]].transpose(1, 2)
            else:
                cache[b[p // PAGE], p % PAGE] = rows[self.rows(i)]
                t = cache[b[:-(-n // PAGE)]]
            out.append(t.reshape(-1, *t.shape[2:])[:n])
        return out

    def attend(self, q, keys, values, scale, **kw):
        return torch.cat([_attend(q[self.rows(i)], keys[i], values[i], self.lens[i] - self.new[i], scale, **kw)
                          for i in range(len(self.lens))])

    def last(self, x):
        return x[torch.from_numpy(self.at[1:] - 1).to(DEV)]


def _rope_angles(c, pos):
    inv = 1.0 / (c.rope_theta ** (torch.arange(0, c.head_dim, 2, dtype=F64) / c.head_dim))
    r = c.rope_scaling
    wave = 2 * math.pi / inv
    lo, hi = r["original_max_position_embeddings"] / r["low_freq_factor"], r["original_max_position_embeddings"] / r["high_freq_factor"]
    mix = (r["original_max_position_embeddings"] / wave - r["low_freq_factor"]) / (r["high_freq_factor"] - r["low_freq_factor"])
    inv = torch.where(wave > lo, inv / r["factor"], torch.where(wave < hi, inv, (1 - mix) * inv / r["factor"] + mix * inv))
    a = torch.outer(pos.to(F64), inv.to(pos.device))
    return torch.cat([a, a], 1)[:, None]


def _exact_llama(st):
    c, sd = st.cfg, st.sd
    G, D, nl, eps = c.num_key_value_heads, c.head_dim, c.num_hidden_layers, c.rms_norm_eps
    caches, _ = st.start([(G, PAGE, D)] * (2 * nl), [])
    ang = _rope_angles(c, st.pos)

    def mat(name):
        w = sd[name + ".weight"]
        if st.case.get("dtype") != "fp8" or name == "lm_head":
            return w
        w = w.float()  # each row in steps of its largest value / 448, as the 8-bit weights hold it
        s = w.abs().amax(1, keepdim=True).clamp_min(1e-12) / 448.0
        return (w / s).to(torch.float8_e4m3fn).to(F64) * s.to(F64)

    def norm(x, name):
        return _rms(x, eps) * sd[name + ".weight"].to(F64)

    def rope(x):
        h = D // 2
        return x * ang.cos() + torch.cat([-x[..., h:], x[..., :h]], -1) * ang.sin()

    x = sd["model.embed_tokens.weight"][st.ids].to(F64)
    for i in range(nl):
        p = "model.layers.%d." % i
        h = norm(x, p + "input_layernorm")
        q, k, v = (_lin(h, mat(p + "self_attn.%s_proj" % n)).view(len(h), -1, D) for n in "qkv")
        ks, vs = st.append(caches[2 * i], rope(k)), st.append(caches[2 * i + 1], v)
        o = st.attend(rope(q), ks, vs, D ** -0.5)
        x = x + _lin(o.reshape(len(x), -1), mat(p + "self_attn.o_proj"))
        h = norm(x, p + "post_attention_layernorm")
        a = torch.nn.functional.silu(_lin(h, mat(p + "mlp.gate_proj"))) * _lin(h, mat(p + "mlp.up_proj"))
        x = x + _lin(a, mat(p + "mlp.down_proj"))
    return _lin(norm(st.last(x), "model.norm"), sd["lm_head.weight"]), caches, []


def _distance_bias(rel, far):
    """[far + 1, heads]: rows below half the table exact, then logarithmic buckets up to `far`."""
    rows, half = rel.shape[0], rel.shape[0] // 2
    idx = []
    for n in range(far + 1):
        if n < half:
            idx.append(n)
            continue
        k = 0
        while half + k < rows - 1 and far ** (k + 1) * half ** (rows - half) <= n ** (rows - half) * half ** (k + 1):
            k += 1
        idx.append(half + k)
    return rel[torch.tensor(idx, device=rel.device)].to(F64)


def _exact_mamba(st, W, p, m, eps, h, conv, ssm):
    """One Mamba-2 layer; conv [slots, taps - 1, channels] and ssm [slots, heads, N, P] advance in place."""
    H, P, n, G, taps = m["heads"], m["vdim"], m["state"], m["groups"], m["conv"]
    inner = H * P
    z, u, dt = torch.split(_lin(h, W[p + "in"]), [inner, inner + 2 * G * n, H], 1)
    dt = torch.nn.functional.softplus(dt + W[p + "dt_bias"].to(F64), threshold=40)
    w, b = W[p + "conv"].to(F64), W[p + "conv.b"].to(F64)
    B, T = len(st.lens), max(st.new)
    pad = torch.zeros(B, T, inner + 2 * G * n + H, dtype=F64, device=h.device)  # shorter sequences end in steps of no length
    for i in range(B):
        r = torch.cat([conv[i + 1], u[st.rows(i)]])
        y = b + sum(r[t:t + st.new[i]] * w[:, t] for t in range(taps))
        pad[i, :st.new[i], :-H] = torch.nn.functional.silu(y)
        pad[i, :st.new[i], -H:] = dt[st.rows(i)]
        conv[i + 1] = r[len(r) - taps + 1:]
    x, Bm, C, d = torch.split(pad, [inner, G * n, G * n, H], 2)
    x, Bm, C = x.reshape(B, T, H, P), Bm.reshape(B, T, G, n), C.reshape(B, T, G, n)
    decay = torch.exp(-torch.exp(W[p + "A_log"].to(F64)) * d)
    S = ssm[1:].clone()
    y = torch.empty(B, T, H, P, dtype=F64, device=h.device)
    xd = (x * d[..., None]).reshape(B, T, G, H // G, 1, P)
    for t in range(T):
        S.mul_(decay[:, t, :, None, None])
        v = S.view(B, G, H // G, n, P)
        v.addcmul_(Bm[:, t, :, None, :, None], xd[:, t])
        y[:, t] = torch.matmul(C[:, t, :, None, None, :], v).reshape(B, H, P)
    ssm[1:] = S
    y += W[p + "D"].to(F64)[:, None] * x
    y = torch.cat([y[i, :st.new[i]].reshape(-1, inner) for i in range(B)]) * torch.nn.functional.silu(z)
    y = _rms(y.reshape(len(y), m["norm_groups"], -1), eps).reshape(len(y), inner) * W[p + "norm"].to(F64)
    return _lin(y, W[p + "o"])


def _exact_niduvik(st):
    c, W = st.cfg, st.sd
    eps = c.eps
    att = [Ly["mixer"] for Ly in c.layers if Ly["type"] == "attention"]
    ssm = [Ly["mixer"] for Ly in c.layers if Ly["type"] != "attention"]
    S = len(st.lens) + 1
    caches, states = st.start([(m["kv_heads"], PAGE, m["dim"]) for m in att for _ in range(2)],
                              [s for m in ssm for s in ((S, m["conv"] - 1, m["heads"] * m["vdim"] + 2 * m["groups"] * m["state"]),
                                                        (S, m["heads"], m["state"], m["vdim"]))])

    def norm(x, name):
        return _rms(x, eps) * W[name].to(F64)

    x = W["embed"][st.ids].to(F64)
    first, ai, si = None, 0, 0
    for i, Ly in enumerate(c.layers):
        p, m = "l%d." % i, Ly["mixer"]
        h, q = norm(x, p + "norm1"), p + "mix."
        if Ly["type"] == "attention":
            qr, k, v = (_lin(h, W[q + n], W[q + n + ".b"]).view(len(h), -1, m["dim"]) for n in "qkv")
            own, lam = v, W[q + "vmix"].to(F64)
            v = v if first is None else (1 - lam) * v + lam * first
            first = own if first is None else first
            bias, cap = _distance_bias(W[q + "rel"], m["bias_max"]), m["softcap"]
            ks, vs = st.append(caches[2 * ai], k), st.append(caches[2 * ai + 1], v)
            o = st.attend(qr, ks, vs, m["scale"], window=m["mask"]["size"], keep=m["mask"]["keep_first"], sink=True,
                          shape=lambda s, dist, hd: cap * torch.tanh(s / cap) + bias[:, hd][dist.clamp_max(m["bias_max"])])
            o = o * torch.sigmoid(_lin(h, W[q + "g"]))[..., None]
            y, ai = _lin(o.reshape(len(h), -1), W[q + "o"]), ai + 1
        else:
            y, si = _exact_mamba(st, W, q, m, eps, h, states[2 * si], states[2 * si + 1]), si + 1
        x = x + norm(y, p + "norm1b")
        h, lim = norm(x, p + "norm2"), Ly["mlp"]["limit"]
        gt, up = _lin(h, W[p + "mlp.gate"]).clamp(max=lim), _lin(h, W[p + "mlp.up"]).clamp(-lim, lim)
        x = x + norm(_lin(gt * torch.sigmoid(1.702 * gt) * (up + 1), W[p + "mlp.down"]), p + "norm2b")
    return _lin(norm(st.last(x), "final.norm"), W["embed"]), caches, states


def _exact_rolesun(st):
    c, W = st.cfg, st.sd
    own = [Ly["mixer"] for Ly in c.layers if Ly["mixer"].get("kv_from") is None]
    caches, (shift,) = st.start([(PAGE, m["kv_rank"]) for m in own], [(len(c.layers), len(st.lens) + 1, c.width)])
    n = c.width
    turn = st.pos.to(F64)[:, None] * (10000.0 ** (-2.0 * torch.arange((n + 1) // 2, dtype=F64, device=DEV) / n))[None]
    x = W["embed"][st.ids].to(F64) * c.embed_scale + torch.stack([turn.sin(), turn.cos()], 2).reshape(len(st.pos), -1)[:, :n]
    lat, ci = {}, 0

    def add(x, y, z, zb, g):
        y = y * torch.sigmoid(_lin(x, W[z], W[zb]))
        return x + c.residual_mult * _rms(y, c.eps) * W[g].to(F64)

    for i, Ly in enumerate(c.layers):
        p, m = "l%d." % i, Ly["mixer"]
        prev = torch.cat([torch.cat([shift[i, b + 1][None], x[st.rows(b)][:-1]]) for b in range(len(st.lens))])
        shift[i, 1:] = st.last(x)
        h, q = x + (prev - x) * W[p + "shift"].to(F64), p + "mix."
        src = m.get("kv_from")
        if src is None:
            src, rows = i, _rms(_lin(h, W[q + "dkv"]), c.eps) * W[q + "dkv.norm"].to(F64)
            lat[i], ci = st.append(caches[ci], rows), ci + 1
        ks = [_lin(t, W[q + "uk"]).view(len(t), m["heads"], -1) for t in lat[src]]
        vs = [_lin(t, W[q + "uv"]).view(len(t), m["heads"], -1) for t in lat[src]]
        o = st.attend(_lin(h, W[q + "q"]).view(len(h), m["heads"], -1), ks, vs, m["scale"], window=m["mask"]["size"])
        y = _lin(o.reshape(len(h), -1) * torch.sigmoid(_lin(h, W[q + "g"])), W[q + "o"])
        x = add(x, y, p + "rg1", p + "rg1.b", p + "norm1")
        a = torch.nn.functional.silu(_lin(x, W[p + "mlp.gate"])) * _lin(x, W[p + "mlp.up"])
        x = add(x, _lin(a, W[p + "mlp.down"]), p + "rg2", p + "rg2.b", p + "norm2")
    return _lin(_rms(st.last(x), c.eps) * W["final.norm"].to(F64) * c.logit_scale, W["head"]), caches, [shift]


@torch.no_grad()
def exact(case, seed):
    if case["path"] == "embed":
        return _exact_embed(case, seed)
    if case["path"] == "search":
        return _exact_search(case, seed)
    f = {"llama": _exact_llama, "niduvik": _exact_niduvik, "rolesun": _exact_rolesun}[case["family"]]
    logits, caches, states = f(_Step(case, seed))
    return {"logits": logits, "caches": caches, "states": states}
