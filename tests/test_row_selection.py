"""Norms of selected rows where the selection is empty or has gaps."""
import pytest
import torch

from rag_llm_k8s_amd.ops import _lib

DEV = "cuda"
INVALID = 1  # hipErrorInvalidValue


def test_no_address_alone_is_not_all_rows():
    """A tensor without elements has a null address: n tells it from no selection, on the host."""
    call = lambda M, n: _lib.lib().ragk_add_partials_rmsnorm(None, 1, M, None, 512, None, None, 512, 512, 1e-5, 0, None, n, None)
    assert call(4, 0) == INVALID and call(4, 3) == INVALID and call(0, 0) == 0
    assert _lib.lib().ragk_rmsnorm_rows(None, 512, None, None, None, 512, 0, 512, 1e-5, None) == 0


@pytest.mark.gpu
def test_rows_of_a_selection():
    from rag_llm_k8s_amd.ops import native

    h, w, P = torch.randn(70, 512, device=DEV).bfloat16(), torch.randn(512, device=DEV).bfloat16(), torch.randn(2, 70, 512, device=DEV)
    none, gaps, before = torch.empty(0, dtype=torch.int32, device=DEV), torch.arange(8, dtype=torch.int32, device=DEV)[::2], h.clone()
    assert native.rmsnorm_rows(h, none, w, 1e-5).shape == (0, 512)
    for rounded in (True, False):
        assert native.add_partials_rmsnorm(P, h, w, 1e-5, rounded=rounded, rows=none).shape == (0, 512)
        with pytest.raises(ValueError):
            native.add_partials_rmsnorm(P, h, w, 1e-5, rounded=rounded, rows=gaps)
    with pytest.raises(ValueError):
        native.rmsnorm_rows(h, gaps, w, 1e-5)
    assert torch.equal(h, before)


@pytest.mark.gpu
@pytest.mark.parametrize("n,way", [(20, "hidden_states_few"), (80, "hidden_states_splitk"), (80, None)])
def test_a_prompt_without_logits_rows(monkeypatch, n, way):
    """No logits, and the caches of the step that has some."""
    from rag_llm_k8s_amd.models import llama as L
    from rag_llm_k8s_amd.models.base import StepInput
    from rag_llm_k8s_amd.ops.backend import AttnMeta

    cfg = L.LlamaConfig(vocab_size=512, hidden_size=1024, intermediate_size=2048, num_hidden_layers=2, num_attention_heads=8,
                        num_key_value_heads=2, head_dim=128)
    m = L.LlamaModel(cfg, L.LlamaWeights.random(cfg, DEV, seed=1), DEV, max_positions=256)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    taken = []
    monkeypatch.setattr(m.be, "splits", lambda M, w: way == "hidden_states_few")
    monkeypatch.setattr(m.be, "prefill_nsplit", lambda M, w: 2 if way == "hidden_states_splitk" else 1)
    if way:
        run = getattr(L.LlamaModel, way)
        monkeypatch.setattr(m, way, lambda *a: (taken.append(1), run(m, *a))[1])
    tiles, qtiles = m.prefill_work([n], DEV)
    meta = AttnMeta("prefill", i32([n]), i32([[1, 2]]), cu_q=i32([0, n]), tiles=tiles, qtiles=qtiles, host_kv_lens=[n], host_q_lens=[n])

    def step(rows):
        m.allocate_kv_cache(3)
        lg = m.forward(StepInput(i32([3 + i for i in range(n)]), i32(list(range(n))), i32([64 + p for p in range(n)]), meta, rows))
        return lg, torch.cat([t.flatten() for kv in m.kv_cache for t in kv])

    some, c1 = step(i32([n - 1]))
    none, c0 = step(torch.empty(0, dtype=torch.int32, device=DEV))
    assert some.shape == (1, 512) and none.shape == (0, 512) and torch.equal(c0, c1) and len(taken) == (2 if way else 0)
