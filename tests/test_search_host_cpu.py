"""The block that a search's results arrive in: not given back while the device may still write to it, whatever is raised."""
import types

import pytest
import torch

from rag_llm_k8s_amd.ops import native


@pytest.mark.parametrize("at", ["launch", "results", "collect", None])
def test_block_is_held_until_the_stream_is_done(monkeypatch, at):
    calls = []
    block = torch.zeros(64, dtype=torch.int32)
    empty = torch.empty

    def step(name, rc=0):
        def f(*_):
            calls.append(name)
            if at == name == "launch":
                raise KeyboardInterrupt
            return 1 if at == name else rc
        return f

    def fail(*a, **k):
        if at == "results":
            raise MemoryError
        return empty(*a, **k)

    lib = types.SimpleNamespace(ragk_search_arm=step("arm"), ragk_search_collect=step("collect"), ragk_stream_wait=step("wait"))
    monkeypatch.setattr(native._lib, "lib", lambda: lib)
    monkeypatch.setattr(native, "search_block", lambda: block)
    monkeypatch.setattr(native, "stream_ptr", lambda: 0)
    monkeypatch.setattr(torch, "empty", fail)
    if at is None:
        native._search_to_host(2, 3, step("launch"))
        assert calls == ["arm", "launch", "collect"]
    else:
        with pytest.raises({"launch": KeyboardInterrupt, "results": MemoryError, "collect": RuntimeError}[at]):
            native._search_to_host(2, 3, step("launch"))
        assert calls[-1] == "wait"
