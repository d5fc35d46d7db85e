"""Build reuse is checked, not assumed: the kernel library carries the content hash of the kernel
sources it was built from, and the loader refuses a library that does not match the tree."""
import ctypes
import os

import pytest

from rag_llm_k8s_amd import _build
from rag_llm_k8s_amd.ops import _lib


def test_source_hash_is_content_based(tmp_path, monkeypatch):
    h = _build.source_hash()
    assert len(h) == 32 and h == _build.source_hash()
    srcs, _ = _build.hip_sources()
    assert any(s.endswith("search.hip") for s in srcs)
    monkeypatch.setattr(_build, "EXTRA_FLAGS", dict(_build.EXTRA_FLAGS, **{"x.hip": ["-DX"]}))
    assert _build.source_hash() != h  # flags are part of the stamp


@pytest.mark.skipif(not _lib.available(), reason="kernel library not built")
def test_library_stamp_matches_tree_and_stale_is_refused(monkeypatch):
    h = ctypes.CDLL(_lib.LIB_PATH, mode=ctypes.RTLD_GLOBAL)
    _lib._check_stamp(h)  # the in-tree library was built from these sources
    monkeypatch.setattr(_build, "source_hash", lambda: "0" * 32)
    monkeypatch.delenv("RAGK_ALLOW_STALE_LIB", raising=False)
    with pytest.raises(_lib.NativeLibraryError, match="other kernel sources"):
        _lib._check_stamp(h)
    monkeypatch.setenv("RAGK_ALLOW_STALE_LIB", "1")
    _lib._check_stamp(h)
    assert os.path.exists(os.path.join(_build.OBJ_DIR, "ragk_stamp.txt"))


def test_runtime_hash_is_content_based(monkeypatch):
    h = _build.runtime_source_hash()
    assert len(h) == 32 and h == _build.runtime_source_hash()
    monkeypatch.setattr(_build, "RT_FLAGS", _build.RT_FLAGS + ["-DX"])
    assert _build.runtime_source_hash() != h


@pytest.mark.skipif(not os.path.exists(_build.runtime_ext_path()), reason="runtime not built")
def test_runtime_stamp_matches_tree_and_stale_is_refused(monkeypatch):
    from rag_llm_k8s_amd import runtime

    mod = runtime.native_rt()
    assert mod is not None and mod.build_stamp() == _build.runtime_source_hash()
    monkeypatch.delenv("RAGK_ALLOW_STALE_LIB", raising=False)
    monkeypatch.setattr(_build, "runtime_source_hash", lambda: "0" * 32)
    with pytest.raises(runtime.StaleRuntimeError, match="other runtime sources"):
        runtime.check_rt_stamp(mod)
    monkeypatch.setenv("RAGK_ALLOW_STALE_LIB", "1")
    runtime.check_rt_stamp(mod)


@pytest.mark.skipif(not _lib.available(), reason="kernel library not built")
def test_struct_mirrors_have_the_library_s_size(monkeypatch):
    """A struct passed by pointer that differs from the library's is refused when it is loaded."""
    monkeypatch.setattr(_lib, "_lib", None)
    assert ctypes.sizeof(_lib.EncoderCall) == _lib.lib().ragk_encoder_call_bytes()

    class Longer(ctypes.Structure):
        _fields_ = _lib.EncoderCall._fields_ + [("more", ctypes.c_void_p)]

    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "EncoderCall", Longer)
    with pytest.raises(_lib.NativeLibraryError, match="bytes here"):
        _lib.lib()


@pytest.mark.skipif(not _lib.available(), reason="kernel library not built")
def test_search_partials_have_one_count():
    """The lists of a search are those of the kernel it launches: batched queries emit more than the scan would."""
    h = _lib.lib()
    assert not hasattr(h, "ragk_l2_scan_groups")
    scan, batched = (h.ragk_l2_search_groups(0, 10000, nq, 5, 384) for nq in (15, 16))
    assert scan == -(-10000 // 64) and batched == 256
