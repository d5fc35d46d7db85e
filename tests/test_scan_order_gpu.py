"""The chunked scan's blocks sorted by sequence length: a batch gives every sequence the bits that it gets alone, over one
round of blocks and over several, equal lengths, an empty sequence, and more sequences than are sorted."""
import pytest
import torch

from rag_llm_k8s_amd.ops import seq_native as sn
from rag_llm_k8s_amd.ops.backend import AttnMeta
from rag_llm_k8s_amd.ops.specs import SsmSpec

pytestmark = pytest.mark.gpu
DEV, BF16, I32 = "cuda", torch.bfloat16, torch.int32


@pytest.mark.parametrize("heads,lens", [
    (2, [70, 5, 129]), (64, [65, 1, 64]), (64, [190, 125, 124, 168, 185]), (64, [100] * 5), (128, [30, 0, 200]),
    (4, [(37 * i) % 150 + 1 for i in range(64)]), (4, [(37 * i) % 150 + 1 for i in range(65)])])
def test_sequences_as_alone(native, heads, lens):
    g = torch.Generator().manual_seed(heads + len(lens))
    S, T = len(lens), sum(lens)
    spec = SsmSpec(heads=heads, vdim=64, state=32, groups=1, taps=4, norm_groups=1)
    rand = lambda *s: torch.randn(*s, generator=g).to(DEV)  # noqa: E731
    row, xbc = rand(T, spec.row).to(BF16), rand(T, spec.channels).to(BF16)
    w = dict(dt_bias=rand(heads), A=rand(heads).abs() + 0.1, D=rand(heads))
    state = rand(S, heads, spec.state, spec.vdim)

    def scan(lo, part, first):
        n = sum(part)
        cu = torch.tensor([0] + torch.tensor(part).cumsum(0).tolist(), dtype=I32, device=DEV)
        kv = torch.tensor([p + 1 for p in part], dtype=I32, device=DEV)  # one token before: the states are read
        own = torch.arange(first, first + len(part), dtype=I32, device=DEV)
        meta = AttnMeta("prefill", kv, torch.zeros(len(part), 1, dtype=I32, device=DEV), cu_q=cu, states=own,
                        host_q_lens=list(part), host_kv_lens=kv.tolist())
        st = state.clone()
        return sn.ssm_scan_chunk(xbc[lo:lo + n].contiguous(), row[lo:lo + n], spec, w, meta, st), st

    y, st = scan(0, lens, 0)
    lo = 0
    for s, n in enumerate(lens):
        if n:
            y1, st1 = scan(lo, [n], s)
            assert torch.equal(y[lo:lo + n], y1) and torch.equal(st[s], st1[s]), s
        else:
            assert torch.equal(st[s], state[s])
        lo += n
