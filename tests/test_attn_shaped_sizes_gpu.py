"""Prompts' shaped attention over every pair of key and value sizes it is built for, against the plain kernel
(one wave per token and head, fp32 arithmetic on the same bf16 rows and pages)."""
import pytest
import torch

from rag_llm_k8s_amd.ops import seq_native as sn
from rag_llm_k8s_amd.ops.backend import AttnMeta
from rag_llm_k8s_amd.ops.specs import AttnSpec

pytestmark = pytest.mark.gpu
DEV, BF16, I32 = "cuda", torch.bfloat16, torch.int32
FORMS = {
    "plain": dict(window=0),
    "window": dict(window=70),
    "general": dict(window=90, keep_first=67, far=40, softcap=60.0, sink=True, gate=True, bias_bound=9.0),
    "bounded": dict(window=130, keep_first=3, far=200, softcap=9.0, sink=True, gate=True, bias_bound=9.0),
}


@pytest.mark.parametrize("dv", [32, 64, 128, 256])
@pytest.mark.parametrize("dk", [32, 64, 128, 256])
def test_every_size_against_plain_arithmetic(native, dk, dv):
    g = torch.Generator().manual_seed(dk + dv)
    for i, (form, o) in enumerate(FORMS.items()):
        spec = AttnSpec(heads=(4, 2, 3, 8)[i], kv_heads=(1, 2, 1, 2)[i], dim=dk, vdim=dv, scale=1.5 * dk ** -0.5, **o)
        assert spec.bounded == (form == "bounded")
        q_lens, kv_lens = [1, 31, 33, 130], [64, 31, 200, 257]  # with a context of 63, 0, 167 and 127 tokens
        T, n = sum(q_lens), [-(-k // 64) for k in kv_lens]
        kc, vc = (torch.randn(sum(n), spec.kv_heads, 64, d, generator=g).to(DEV, BF16) for d in (dk, dv))
        row = torch.randn(T, spec.row, generator=g).to(DEV, BF16)
        table = (3 * torch.randn(spec.heads, spec.far + 1, generator=g)).clamp(-9, 9).to(DEV) if spec.far else None
        bt, perm = torch.zeros(4, max(n), dtype=I32), torch.randperm(sum(n), generator=g).to(I32)
        for s, part in enumerate(perm.split(n)):
            bt[s, :n[s]] = part
        cu = torch.tensor([0] + torch.tensor(q_lens).cumsum(0).tolist(), dtype=I32, device=DEV)
        meta = AttnMeta("prefill", torch.tensor(kv_lens, dtype=I32, device=DEV), bt.to(DEV), cu_q=cu,
                        qtiles={spec.q_tile: sn.query_tiles(q_lens, spec.q_tile).to(DEV)})
        got, want = (torch.zeros(T, spec.out_row, dtype=BF16, device=DEV) for _ in range(2))
        sn.attn_prefill(row, spec, table, kc, vc, meta, got)
        sn.attn_rows(row, spec, table, kc, vc, meta, want)
        # each side rounds its outputs to bf16 (8 significant bits: 2^-8 of a value, 2^-7 for both); where the values of a sum
        # cancel, the weights' own errors stay: 16 bits kept (2^-16), scores of up to ~30 in fp32 over 256 products, the
        # exponential and the gate's reciprocal of 1 ulp or two: below 2^-14 of the largest value
        w = want.float()
        err = (got.float() - w).abs() - w.abs() * 2.0 ** -7
        assert float(err.max()) <= 2.0 ** -14 * float(vc.abs().max()), (form, float(err.max()))
