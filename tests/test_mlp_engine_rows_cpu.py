"""The work split of the persistent decode tail by the distance of its gate/up rows: gate, split and launch use one."""
import ctypes

import pytest

from rag_llm_k8s_amd.ops import _lib

ME_KC, ME_MAXA, ME_MAXB = 512, 64, 56


def _split(G, H, I, ld):
    out, rows = (ctypes.c_int * 4)(), []
    for w in range(G):
        assert _lib.lib().ragk_mlp_engine_rows_split(G, w, H, I, ld, ctypes.cast(out, ctypes.c_void_p)) == 0
        rows.append(tuple(out))
    return rows


@pytest.fixture(params=[None, (1, 1), (27, 32), (2, 1)])
def weights(request):
    if request.param:
        assert _lib.lib().ragk_mlp_engine_set_xcd_weights(*request.param) == 0
    yield request.param
    assert _lib.lib().ragk_mlp_engine_set_xcd_weights(0, 0) == 0


@pytest.mark.parametrize("G", [304, 256, 240, 224, 80, 1])
@pytest.mark.parametrize("H,I", [(4096, 14336), (1024, 2048), (2048, 5632)])
@pytest.mark.parametrize("gap", [0, 64])
def test_split_covers_every_group_once_within_capacity(weights, G, H, I, gap):
    rows = _split(G, H, I, H + gap)
    assert rows[0][0] == rows[0][2] == 0 and (rows[-1][1], rows[-1][3]) == (I // 8, H // 16)
    assert all(r[1] == n[0] and r[3] == n[2] for r, n in zip(rows, rows[1:])) and all(r[0] <= r[1] and r[2] <= r[3] for r in rows)
    if _lib.lib().ragk_mlp_engine_rows_ok(1, H, I, G, H + gap):
        assert all((a1 - a0) * max(H // ME_KC, 1) <= ME_MAXA and (d1 - d0) * (I // ME_KC) <= ME_MAXB and (a1 - a0) * 8 <= 64
                   and (d1 - d0) * 16 <= 64 for a0, a1, d0, d1 in rows)


def test_weights_by_the_rows_distance():
    """An 8B Llama on 256 CUs: 6 and 8 groups where rows lie 8 KB apart, 7 with a gap, and what is set for both."""
    share = lambda ld: [r[1] - r[0] for r in _split(256, 4096, 14336, ld)]
    L = _lib.lib()
    assert share(4096) == [6, 8] * 128 and share(4160) == [7] * 256
    try:
        assert L.ragk_mlp_engine_set_xcd_weights(3, 4) == 0
        assert share(4096) == share(4160) == [6, 8] * 128
        assert L.ragk_mlp_engine_set_xcd_weights(1, 1) == 0
        assert share(4096) == share(4160) == [7] * 256
    finally:
        L.ragk_mlp_engine_set_xcd_weights(0, 0)
    assert L.ragk_mlp_engine_set_xcd_weights(0, 1) != 0 and L.ragk_mlp_engine_set_xcd_weights(1, 0) != 0
    # the gate goes by the split that is launched: 224 workgroups hold 8 groups each evenly, not 9 at 3 : 4
    assert L.ragk_mlp_engine_rows_ok(1, 4096, 14336, 224, 4160) and not L.ragk_mlp_engine_rows_ok(1, 4096, 14336, 224, 4096)
    assert not L.ragk_mlp_engine_rows_ok(1, 4096, 14336, 256, 4095) and not L.ragk_mlp_engine_rows_ok(1, 4096, 14336, 256, 4100)
