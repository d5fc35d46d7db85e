"""The fp32 gate z sigmoid(z) and step size ln(1 + e^z) of the state space kernels against 64 bits, through the entry points:
a convolution that passes its input on, and one token of the scan whose output is its step size."""
import pytest
import torch

from rag_llm_k8s_amd.ops import seq_native as sn
from rag_llm_k8s_amd.ops.backend import AttnMeta
from rag_llm_k8s_amd.ops.specs import SsmSpec

pytestmark = pytest.mark.gpu
DEV, F32, I32 = "cuda", torch.float32, torch.int32
SPEC = SsmSpec(heads=64, vdim=4, state=4, groups=1, taps=2, norm_groups=1)
S = 512
# 4 half units in the last place: one for the hardware's exponential, the rest for at most four rounded steps behind it
TOL = 2.0 ** -22
SPECIAL = [0.0, -0.0, 1e-40, -1e-40, 20.0, 30.0, 88.0, -87.0, -87.5, -88.5, -89.0, -104.0, 105.0, -200.0, 1e30, -1e30, 3e38, -3e38]
# below the smallest normal number units are absolute: four rounded steps of half a unit, 2^-150 each
TINY = 2.0 ** -148


def metadata():
    return AttnMeta("prefill", torch.ones(S, dtype=I32, device=DEV), torch.zeros(S, 1, dtype=I32, device=DEV),
                    cu_q=torch.arange(S + 1, dtype=I32, device=DEV), states=torch.arange(S, dtype=I32, device=DEV),
                    host_q_lens=[1] * S, host_kv_lens=[1] * S)


def values(lo, hi, n):
    z = torch.rand(S, n, generator=torch.Generator().manual_seed(n)) * (hi - lo) + lo
    z[0, :len(SPECIAL)] = torch.tensor(SPECIAL)
    return z.to(DEV)


def close(got, want):
    err = (got.double() - want).abs()
    assert not got.isnan().any()
    assert bool((err <= TOL * want.abs() + TINY).all()), float((err / want.abs().clamp_min(1e-36)).max())


def silu(z, state):
    row = torch.zeros(S, SPEC.row, device=DEV)
    row[:, SPEC.off_x:SPEC.off_x + SPEC.channels] = z
    w = dict(conv_w=torch.zeros(2, SPEC.channels, device=DEV), conv_b=torch.zeros(SPEC.channels, device=DEV))
    w["conv_w"][1] = 1
    return sn.ssm_conv(row, SPEC, w, metadata(), torch.zeros(S, 1, SPEC.channels, device=DEV), state)


def softplus(z, state):
    row, xbc = torch.zeros(S, SPEC.row, device=DEV), torch.zeros(S, SPEC.channels, device=DEV)
    row[:, SPEC.off_dt:SPEC.off_dt + SPEC.heads] = z
    xbc[:, :SPEC.inner] = xbc[:, SPEC.inner:SPEC.inner + 1] = xbc[:, SPEC.inner + SPEC.state:][:, :1] = 1
    w = {k: torch.zeros(SPEC.heads, device=DEV) for k in ("dt_bias", "A", "D")}
    return sn.ssm_scan_seq(xbc, row, SPEC, w, metadata(), state)[:, ::SPEC.vdim]


@pytest.mark.parametrize("lo,hi", [(-1e-3, 1e-3), (-1, 1), (-8, 8), (8, 40), (-86, -8), (-88.7, -86)])
def test_gate_and_step_against_64_bits(native, lo, hi):
    state = torch.zeros(S, SPEC.heads, SPEC.state, SPEC.vdim, device=DEV)
    z = values(lo, hi, SPEC.channels)
    d = z.double()
    e = torch.exp(-d)
    close(silu(z, state), d / (1 + e.masked_fill(e > torch.finfo(F32).max, float("inf"))))  # fp32's divisor: infinite from -88.73 down
    z = values(lo, hi, SPEC.heads)
    d = z.double()
    close(softplus(z, state), d.clamp_min(0) + torch.log1p(torch.exp(-d.abs())))


def test_infinities_and_nan(native):
    state = torch.zeros(S, SPEC.heads, SPEC.state, SPEC.vdim, device=DEV)
    z = torch.zeros(S, SPEC.channels, device=DEV)
    z[0, :3] = torch.tensor([float("inf"), -float("inf"), float("nan")])
    got = silu(z, state)[0, :3]
    assert got[0] == float("inf") and got[1].isnan() and got[2].isnan()  # inf, -inf / inf, NaN
    got = softplus(z[:, :SPEC.heads], state)[0, 1:3]  # an infinite step times the rate 0 is no number anyway
    assert got[0] == 0 and got[1].isnan()
