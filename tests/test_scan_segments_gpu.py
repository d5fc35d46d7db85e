"""The chunked scan in segments: states handed on between segments, sequences of one segment and of several, kept states."""
import pytest
import torch

from rag_llm_k8s_amd.ops import seq_native as q
from rag_llm_k8s_amd.ops.backend import AttnMeta
from rag_llm_k8s_amd.ops.specs import SsmSpec

pytestmark = pytest.mark.gpu
DEV = "cuda"


def scan64(spec, xbc, dt, A, D, S):
    """y [T, H, P] and the last state, token by token in fp64."""
    H, P, N, G = spec.heads, spec.vdim, spec.state, spec.groups
    x, B, C = torch.split(xbc, [H * P, G * N, G * N], 1)
    x = x.reshape(-1, H, P)
    B, C = (t.reshape(-1, G, N).repeat_interleave(H // G, 1) for t in (B, C))
    y = []
    for t in range(len(x)):
        S = S * torch.exp(-A * dt[t])[:, None, None] + (dt[t][:, None] * B[t])[:, :, None] * x[t][:, None, :]
        y.append((C[t][:, :, None] * S).sum(1) + D[:, None] * x[t])
    return torch.stack(y), S


@pytest.mark.parametrize("vdim,state", [(64, 128), (40, 24), (96, 200)])
@pytest.mark.parametrize("lens,fresh", [([1500], True), ([1500], False), ([833, 64, 1, 130], False), ([200, 770], True)])
def test_scan_segments(native, monkeypatch, vdim, state, lens, fresh):
    spec = SsmSpec(heads=2, vdim=vdim, state=state, groups=1, taps=3, norm_groups=1)
    T, S, H = sum(lens), len(lens), spec.heads
    g = torch.Generator(device=DEV).manual_seed(T + vdim)
    r = lambda *s: torch.randn(*s, device=DEV, generator=g)  # noqa: E731
    xbc, row = r(T, spec.channels).bfloat16(), r(T, spec.row).bfloat16()
    w = dict(dt_bias=r(H) - 1.5, A=torch.exp(1.5 * r(H) - 1), D=r(H))
    kept = r(S + 1, H, state, vdim)
    meta = AttnMeta("prefill", torch.tensor([n + 5 * (not fresh) for n in lens], dtype=torch.int32, device=DEV),
                    torch.zeros(S, 1, dtype=torch.int32, device=DEV))
    meta.cu_q = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device=DEV)
    meta.states = torch.arange(1, S + 1, dtype=torch.int32, device=DEV)
    assert q.scan_segments(max(lens), S, spec)[0] > 1
    res = []
    for seg in (q.scan_segments(max(lens), S, spec), (2, -(-T // 128) * 64), (1, 0)):
        monkeypatch.setattr(q, "scan_segments", lambda *a, seg=seg: seg)
        st = kept.clone()
        y = q.ssm_scan_chunk(xbc, row, spec, w, meta, st)
        assert torch.equal(st[0], kept[0])
        res.append((y.double(), st[1:].double()))
    dt = torch.nn.functional.softplus(row.double()[:, spec.off_dt:spec.off_dt + H] + w["dt_bias"].double())
    for i, n in enumerate(lens):
        a = sum(lens[:i])
        ref, end = scan64(spec, xbc[a:a + n].double(), dt[a:a + n], w["A"].double(), w["D"].double(),
                          kept[i + 1].double() * (not fresh))
        errs = [((s[i] - end).norm() / end.norm()).item() for _, s in res]
        # the state is kept as bf16 pairs (2^-16) between chunks on every path
        assert max(errs) < 1e-4 and errs[0] < 1.5 * errs[2] + 1e-6 and errs[1] < 1.5 * errs[2] + 1e-6, errs
        # y: one rounding to bf16, at most 2^-8 of each value, and the pairs' 2^-16
        for y, _ in res:
            assert ((y[a:a + n] - ref.reshape(n, -1)).norm() / ref.norm()).item() < 2.0 ** -8
