"""The first layer's norm of a decode step is computed once: with the embedding, or inside the first product."""
import pytest
import torch

from rag_llm_k8s_amd.engine.llm_engine import LLMEngine, SamplingParams
from rag_llm_k8s_amd.models import llama as L


@pytest.mark.parametrize("batch,inside", [(1, True), (4, True), (5, False)])
def test_first_norm_of_a_decode_step(batch, inside):
    cfg = L.llama_tiny()
    w = L.LlamaWeights.random(cfg, "cpu", seed=3)
    g = torch.Generator().manual_seed(4)
    prompts = [torch.randint(3, cfg.vocab_size, (9 + i,), generator=g).tolist() for i in range(batch)]
    outs, norms, embeds = [], [], []
    for part in (False, True):
        model = L.LlamaModel(cfg, w, "cpu", max_positions=256)
        be = model.be
        be.enable_part = part
        if part:
            run, embed = model.hidden_states_decode_part, be.embed_rmsnorm
            model.hidden_states_decode_part = lambda inp, hn: (norms.append((hn[0].shape[0], hn[1] is None)), run(inp, hn))[1]
            be.embed_rmsnorm = lambda ids, *a, **k: (embeds.append(ids.shape[0]), embed(ids, *a, **k))[1]
        eng = LLMEngine(model, num_blocks=32, max_batch=8, max_model_len=256, use_graphs=False)
        outs.append(eng.generate(prompts, SamplingParams(max_new_tokens=5, do_sample=False, ignore_eos=True)))
    assert outs[0] == outs[1] and norms
    assert all(n == inside for m, n in norms if m == batch) and any(m == batch for m, _ in norms)
    assert (batch in embeds) == (not inside)  # (prompts have more rows)
