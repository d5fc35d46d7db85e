"""Shape-checked Python entry points of the gfx950 kernels (GPU tensors only).

Every function validates dtype / contiguity / shapes on the host *before* the launch
(a mis-shaped launch could fault the GPU), then calls the C ABI with the current
HIP stream, so everything here is capturable in a hipGraph (torch.cuda.CUDAGraph).
"""
from __future__ import annotations

import functools
import itertools
import math
import operator
import os
import threading

import torch

from . import _lib
from ._lib import check, ptr, stream_ptr
from .reference import EPI


PAIR_EPI = ("silu_mul", "glu_clip")  # epilogues over packed [64 gate | 64 up] weight rows


def _req(cond, msg):
    if not cond:
        raise ValueError(msg)


def _bf16_2d(t, name):
    _req(t.is_cuda and t.dtype == torch.bfloat16 and t.dim() == 2, "%s must be a 2-D bf16 GPU tensor" % name)
    _req(t.stride(1) == 1, "%s must be row-contiguous" % name)


# ----------------------------------------------------------------------------- GEMM
# large-M GEMMs (prefill) go to the 256x256 MFMA kernels from this many rows
PP_MIN_M = 1024


def set_w4_grid(g):
    """gemm_w4 persistent grid: -1 = one block per CU (default), 0 = one block per output tile,
    g > 0 = at most g blocks (each block loops over tiles g apart)."""
    check(_lib.lib().ragk_gemm_w4_set_grid(int(g)), "ragk_gemm_w4_set_grid")




DEC_DEFAULT = True
DEC_WS_BYTES = 96 << 20
_dec_ws = {}


def dec_workspace(device):
    """Per-device split-K workspace for the decode GEMM: fp32 slabs + ticket counters (zeroed once;
    the last-arriving block resets its counter). Allocated eagerly, before any graph capture."""
    key = str(device)
    if key not in _dec_ws:
        _dec_ws[key] = (torch.empty(DEC_WS_BYTES // 4, dtype=torch.float32, device=device),
                        torch.zeros(65536, dtype=torch.int32, device=device))
    return _dec_ws[key]


def use_dec(M, N, K, epi):
    """v3 (LDS-shared activations) wins over v1 only on vocab-sized N at M > 16 (lm_head: 5.1 vs
    3.1 TB/s at M=32, cache-cold); v1 stays the default elsewhere (profiles/kernels_r1_decode.json)."""
    return 16 < M <= 64 and N >= 32768 and K % 256 == 0 and epi not in PAIR_EPI


STREAM_DEFAULT = True
STREAM_MIN_ROWS = 16384
# vocab-sized weights (>= 32768 rows, the lm_head) go to the stream GEMM (nt weights) only above batch 16:
# batch 32 6.97 -> 6.94 ms per decode step, batch 4 slower (profiles/decode_lmhead_stream_r4.log)
STREAM_MAX_ROWS = 262144
STREAM_VOCAB_MIN_M = 17


def use_stream(M, N, K, epi, fp8=False):
    """Decode GEMM v4 (glds ring) wins where one launch has >= ~128 n-tiles of long K-streams and
    no split-K: the packed gate/up projection (4.5 vs 3.4 TB/s bf16 at M=32, 4.4 vs 2.2 at M=64;
    fp8 2.6 vs 1.5 at M=32) and other 16k-32k-row weights. Below that, the fixed pipeline-fill +
    split-K reduction latencies lose to the register-streaming kernels (profiles/tune_stream_r1.json)."""
    rows = 2 * N if epi in PAIR_EPI else N
    if M > 64 or not (STREAM_MIN_ROWS <= rows < STREAM_MAX_ROWS) or K % 128:
        return False
    if rows >= 32768 and M < STREAM_VOCAB_MIN_M:
        return False
    return M > 16 if fp8 else True


def use_slabs(M, N, K, epi, out_f32=False):
    """Long projections of large weights at 17 to 64 rows: the LDS-DMA weight stream in fp32 slabs and a pass that sums them
    (gemm_mid.hip ragk_gemm_slabs), where the register-streaming kernel keeps its weights on too few blocks and reads the
    activations again for every 16 columns. 17 / 64 rows: 4096 x 14336 40 / 66 us -> 24 / 28, 14336 x 4096 37 / 74 -> 29 / 32,
    33 / 64 rows: 6144 x 4096 28 / 39 -> 15 / 18; 64 rows of 4096 x 4096 23 -> 13. The second launch, the slabs' allocation and
    this rule cost the host 7 us, so not where the GPU gains little more (20 rows: 6144 x 4096 22 against 14, 4096 x 4096 14
    against 11; a rolesun step of 694 us became 723), nor below 2^24 weights, where the step's launches bound it (2048 x 5632 at
    20 rows 16.6 against 9.4, but the steps that hold it 368 -> 409 and 508 -> 557 us); up to 16 rows the second launch takes
    what the first gains. The other kernel cuts K eight times; a slab is a sum of sums over 512 of K here, so that it is no further
    off (rms error of fp32 sums, other kernel / slabs / slabs of one sum: 64 x 6144 x 4096 1.37 / 1.34 / 1.89e-7, 14336 x 4096
    1.37 / 1.35 / 2.72e-7, 10240 x 8192 1.93 / 1.40 / 3.96e-7; 2 to 4 % of the stream's time). fp32 results keep the one launch."""
    return (not out_f32 and 16 < M <= 64 and K >= 4096 and K % 128 == 0 and N % 8 == 0 and epi not in PAIR_EPI
            and N * K >= 1 << 24 and M * N * K >= 8e8 and stream_part_cfg(M, N, K)[1] > 1)


def use_vocab(M, N, K, epi, gap=False):
    """fp32 logits go to the slab form of the stream GEMM with one slab: its 64-row tiles keep two blocks a CU and no K-split
    ends in a reduction (32000 x 4096, 4 / 32 rows: stream GEMM 64 / 64 us -> 49 / 48; 32768 x 4096, 11 rows: register-streaming
    kernel, which reads the activations for every 16 columns, 58.6 -> 48.3, 32 rows: 65.7 -> 49.6). The register-streaming
    kernel keeps vocabularies from 32768 on below 8 rows (128256 x 4096 at 5 rows: 173 us against 184, at 8: 191 against 182) where
    the weight's rows lie without a gap between them (`gap`, ops/pitch.py; with it 32768 x 4096 at 1 / 4 / 7 rows 48 / 50 / 55 -> 43 / 43 / 43,
    128256 x 4096 175 / 182 / 202 -> 159 / 159 / 160). It cuts K into eight sums; the slab's, over 256 up to K = 2048 and 512 from there
    on, are no longer at multiples of 2048 (rms error in 1e-7, that kernel's and these, K = 2048 / 4096 / 6144 / 8192: 1.02 / 1.37 / 1.67 /
    1.91 and 1.02 / 1.37 / 1.42 / 1.47) and would be in between (1024 / 3072: 0.81 / 1.20 and 0.94 / 1.34)."""
    return (epi == "none" and (1 if N < 32768 or (gap and K % 2048 == 0) else 8) <= M <= 64 and N >= STREAM_MIN_ROWS and N % 4 == 0
            and K % 64 == 0)


def use_pp(M, N, K, epi):
    """Large-M GEMMs go to a 256x256 MFMA kernel: gemm_w4.hip (default, 4 waves x 128x128, 9-16 %
    faster on the Llama-8B prefill shapes, profiles/gemm_w4_r1.txt) or the 8-wave ping-pong gemm_pp.hip."""
    if M < PP_MIN_M or K % 64 or K < 192:  # gemm_w4's continuous ring needs three K-tiles per tile
        return False
    return N % 128 == 0 if epi in PAIR_EPI else N % 8 == 0


# Large-M GEMMs through hipBLASLt (torch) instead of gemm_w4, by epilogue (A/B only). "none" (default):
# every large-M GEMM on the hand-written gemm_w4, no library kernel on the prefill path. "resid": the
# residual-add projections (o_proj, down: h += x @ W^T as one in-place addmm, beta = 1) on hipBLASLt --
# its K-loop is 4-6 % faster on those two shapes, worth 0.85 % of the headline bench (1644 / 1648 vs
# 1660 / 1661 tok/s, same box alternating, profiles/bench_prefill_blas_ab_r5.log); "plain": no-epilogue
# GEMMs only; "all": both. The fused SiLU*up gate/up GEMM has no library form (gemm_w4 is 2.8 % faster
# than hipBLASLt's plain GEMM of the same shape, profiles/gemm_silu_rcp_r5.log).
PREFILL_BLAS = os.environ.get("RAGK_PREFILL_BLAS", "none")


# The prefill qkv projection with rope_kv's work in its epilogue (gemm_w4's, gemm_mid's; RoPE on q / k, k and v rows into
# the paged cache; bit-identical to gemm + rope_kv): one pass over the 32k-token chunk's qkv fewer.
PREFILL_ROPE_FUSED = os.environ.get("RAGK_PREFILL_ROPE", "1") != "0"


def gemm_rope_kv_ok(x, w, positions, cos_t, sin_t, slots, k_cache, v_cache, Hq, Hkv, D):
    """Whether gemm_rope_kv takes these operands (else: gemm + rope_kv)."""
    if not PREFILL_ROPE_FUSED or D != 128 or slots is None or k_cache is None or v_cache is None:
        return False
    if not (isinstance(x, torch.Tensor) and isinstance(w, torch.Tensor) and x.is_cuda and w.dim() == 2):
        return False
    M, K = x.shape
    N = w.shape[0]
    if N != (Hq + 2 * Hkv) * D or N % 256 or w.shape[1] != K or M <= 64 or K % 64 or K < 192:
        return False
    if PREFILL_BLAS in ("plain", "all"):
        return False
    if x.dtype != torch.bfloat16 or w.dtype != torch.bfloat16 or x.stride(1) != 1 or w.stride(1) != 1:
        return False
    if x.stride(0) * M * 2 >= 2 ** 31 or w.stride(0) * N * 2 >= 2 ** 31:
        return False
    if not (k_cache.is_contiguous() and v_cache.is_contiguous() and k_cache.dim() == 4 and k_cache.shape[1] == Hkv
            and k_cache.shape[3] == D and v_cache.shape == k_cache.shape and k_cache.dtype == torch.bfloat16):
        return False
    if not (cos_t.dtype == torch.float32 and sin_t.dtype == torch.float32 and cos_t.is_contiguous()
            and sin_t.is_contiguous() and cos_t.shape[-1] == D // 2):
        return False
    return (positions.dtype == torch.int32 and slots.dtype == torch.int32 and positions.is_contiguous()
            and slots.is_contiguous() and positions.numel() == M and slots.numel() == M)


def gemm_rope_kv(x, w, positions, cos_t, sin_t, slots, k_cache, v_cache, Hq, Hkv, D, out=None, checked=False):
    """qkv = x @ w^T with RoPE applied to q and k and the k / v rows written to the paged cache at `slots`
    (gemm + rope_kv in gemm's own launches, bit-identical to both). checked: the caller has asked gemm_rope_kv_ok."""
    _req(checked or gemm_rope_kv_ok(x, w, positions, cos_t, sin_t, slots, k_cache, v_cache, Hq, Hkv, D), "gemm_rope_kv operands")
    M, K = x.shape
    N = w.shape[0]
    if out is None:
        out = torch.empty((M, N), dtype=torch.bfloat16, device=x.device)
    _req(out.shape == (M, N) and out.stride(1) == 1 and out.stride(0) % 8 == 0, "gemm_rope_kv out")
    L = _lib.lib()
    x, w = _tile_rows(x, w)
    for r0, r1, mi, S in gemm_plan(M, N, K, True, _cu_count()):
        a = (x.data_ptr() + r0 * x.stride(0) * 2, x.stride(0), w.data_ptr(), w.stride(0),
             out.data_ptr() + r0 * out.stride(0) * 2, out.stride(0), r1 - r0, K, positions.data_ptr() + 4 * r0,
             slots.data_ptr() + 4 * r0, cos_t.data_ptr(), sin_t.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(), Hq, Hkv,
             k_cache.shape[2])
        if mi in W4_TILES:
            check(L.ragk_gemm_w4_rope_kv(*a, mi & 15 or 8, stream_ptr()), "ragk_gemm_w4_rope_kv")
        else:
            ws = torch.empty(S * (r1 - r0) * N, dtype=torch.float32, device=x.device) if S > 1 else None
            check(L.ragk_gemm_mid_rope_kv(*a, mi, S, ptr(ws), stream_ptr()), "ragk_gemm_mid_rope_kv")
    return out


def _gemm_blas(x, w, resid, out, epi):
    if epi == "resid":
        if out.data_ptr() == resid.data_ptr() and out.stride() == resid.stride():
            return out.addmm_(x, w.t())
        return torch.addmm(resid, x, w.t(), out=out)
    return torch.mm(x, w.t(), out=out)


def _gemm_operands(x, w, bias, resid, epi):
    """(M, N, K) of a product whose operands are fit for any of its kernels."""
    _bf16_2d(x, "x")
    _bf16_2d(w, "w")
    M, K = x.shape
    N = w.shape[0] // 2 if epi in PAIR_EPI else w.shape[0]
    _req(w.shape[1] == K, "K mismatch %s vs %s" % (tuple(x.shape), tuple(w.shape)))
    _req(K % 128 == 0, "K must be a multiple of 128 (got %d)" % K)
    if epi in PAIR_EPI:
        _req(N % 64 == 0, "%s needs N %% 64 == 0" % epi)
    if epi == "glu_clip":
        _req(bias is not None and bias.is_cuda and bias.dtype == torch.float32 and bias.numel() >= 3
             and bias.is_contiguous(), "glu_clip takes fp32 {limit, alpha, shift} as its bias")
    if "bias" in epi:
        _req(bias is not None and bias.is_cuda and bias.dtype == torch.bfloat16 and bias.numel() == N
             and bias.is_contiguous(), "bias must be bf16[N]")
    if "resid" in epi:
        _bf16_2d(resid, "resid")
        _req(resid.shape == (M, N), "resid shape")
    return M, N, K


def gemm(x, w, bias=None, resid=None, epi="none", out=None, out_f32=False, path=None):
    """out[M,N] = epi(x[M,K] @ w[N,K]^T). For epi='silu_mul', w is the packed
    gate/up weight [2N, K] (see reference.pack_gate_up) and out has N columns."""
    M, N, K = _gemm_operands(x, w, bias, resid, epi)
    e = EPI[epi]
    odt = torch.float32 if out_f32 else torch.bfloat16
    if out is None:
        out = torch.empty((M, N), dtype=odt, device=x.device)
    _req(out.dtype == odt and out.shape == (M, N) and out.stride(1) == 1, "out shape/dtype")
    if M > 64 and N % 8 != 0 and epi not in PAIR_EPI:
        raise ValueError("tile GEMM needs N % 8 == 0")
    if M == 0:
        return out
    if (path is None and PREFILL_BLAS != "none" and not out_f32 and bias is None and use_pp(M, N, K, epi)
            and ((epi == "none" and PREFILL_BLAS in ("plain", "all"))
                 or (epi == "resid" and PREFILL_BLAS in ("resid", "all")))):
        return _gemm_blas(x, w, resid, out, epi)
    if path is None and M > 64:
        rows = 2 * N if epi in PAIR_EPI else N
        x, w = _tile_rows(x, w)
        # gemm_w4 addresses operands with 32-bit buffer offsets
        fits = x.stride(0) * M * 2 < 2 ** 31 and w.stride(0) * rows * 2 < 2 ** 31
        if not fits and use_pp(M, N, K, epi):
            if epi != "glu_clip":
                path = 2  # gemm_pp (8-wave ping-pong, 64-bit addressing): operands past 2 GiB
            else:  # which has no clipped unit: halve the rows until they fit
                h = (M // 2 + 127) // 128 * 128
                gemm(x[:h], w, bias=bias, epi=epi, out=out[:h])
                gemm(x[h:], w, bias=bias, epi=epi, out=out[h:])
                return out
        else:
            w4 = fits and (N % 128 == 0 if epi in PAIR_EPI else N % 8 == 0)
            cols = gemm_columns(M, rows, K, _cu_count()) if w4 else 0
            for c0, c1 in ((0, cols), (cols, rows)) if cols else ((0, rows),):
                wc, bc, rc, oc = _columns(w, bias, resid, out, epi, c0, c1) if cols else (w, bias, resid, out)
                for r0, r1, mi, S in gemm_plan(M, c1 - c0, K, w4, _cu_count(), not cols):
                    _gemm_rows(x, wc, bc, rc, epi, oc, out_f32, r0, r1, mi, S)
            return out
    if path == 0:
        return gemm_mid(x, w, bias=bias, resid=resid, epi=epi, out=out, out_f32=out_f32)
    if path is None and not out_f32 and use_hold(M, N, K, epi) and _vec_rows(x, w) and w.stride(0) < 1 << 24:
        return gemm_hold(x, w, par=bias, epi=epi, out=out)
    if (path is None and use_vocab(M, N, K, epi, w.stride(0) != K) and out_f32 and out.stride(0) == N and _vec_rows(x, w)
            and out.data_ptr() % 16 == 0):
        return gemm_stream_part(x, w, out=out, rows=64, S=1, short_sums=M < 8 and N >= 32768)
    L = _lib.lib()
    ldr = resid.stride(0) if resid is not None else 0
    if path is None and STREAM_DEFAULT and use_stream(M, N, K, epi):
        path = 5
    if path is None and DEC_DEFAULT and use_dec(M, N, K, epi):
        path = 4
    if path is None and M > 16 and use_slabs(M, N, K, epi, out_f32) and _vec_rows(
            x, w, out, *(() if resid is None else (resid,))) and (bias is None or bias.data_ptr() % 16 == 0):
        return _gemm_slabs(x, w, out, bias, resid, ldr, M, N, K, e)
    if path == 5:
        rc = _gemm_stream(x, w, None, out, bias, resid, ldr, M, N, K, epi, e, out_f32)
    elif path == 4:
        ws, cnt = dec_workspace(x.device)
        S = L.ragk_gemm_dec_splits(N, K, e)
        need = S * (2 if epi == "silu_mul" else 1) * M * N
        _req(S == 1 or need <= ws.numel(), "decode GEMM workspace too small (%d > %d floats)" % (need, ws.numel()))
        _req(-(-N // 128) <= cnt.numel(), "too many n-tiles for the counter buffer")
        rc = L.ragk_gemm_dec(x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), out.data_ptr(), out.stride(0),
                             ptr(bias), ptr(resid), ldr, M, N, K, e, int(out_f32), S, ws.data_ptr(), cnt.data_ptr(),
                             stream_ptr())
    elif path == 2:
        rc = L.ragk_gemm_pp(x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), out.data_ptr(), out.stride(0),
                            ptr(bias), ptr(resid), ldr, M, N, K, e, int(out_f32), stream_ptr())
    elif path == 6:
        rc = L.ragk_gemm_w4(x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), out.data_ptr(), out.stride(0),
                            ptr(bias), ptr(resid), ldr, M, N, K, e, int(out_f32), stream_ptr())
    elif path is None:
        rc = L.ragk_gemm(x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), out.data_ptr(), out.stride(0),
                         ptr(bias), ptr(resid), ldr, M, N, K, e, int(out_f32), stream_ptr())
    else:
        rc = L.ragk_gemm_path(path, x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), out.data_ptr(),
                              out.stride(0), ptr(bias), ptr(resid), ldr, M, N, K, e, stream_ptr())
    check(rc, "ragk_gemm")
    return out


def gemm_glu(x, w, par):
    """Packed gate/up projection with the clipped gated unit (par: fp32 {limit, alpha, shift} on the device)."""
    return gemm(x, w, bias=par, epi="glu_clip")


def gemm_mid(x, w, bias=None, resid=None, epi="none", out=None, out_f32=False, mi=4, S=1):
    """gemm() on the ring tiles of gemm_mid.hip: 32 mi rows of 128 columns (mi = 21: 160 of 256), K cut into S slabs (S > 1:
    fp32 slabs in a workspace, summed with the epilogue by a second launch)."""
    M, K = x.shape
    N = w.shape[0] // 2 if epi in PAIR_EPI else w.shape[0]
    x, w = _tile_rows(x, w)
    _req(mi in MID_TILES and 1 <= S <= K // 64 and K % 64 == 0 and w.shape[1] == K, "gemm_mid tile or split")
    _req(out.shape == (M, N) and out.stride(1) == 1, "gemm_mid out")
    _gemm_rows(x, w, bias, resid, epi, out, out_f32, 0, M, mi, S)
    return out


def _columns(w, bias, resid, out, epi, c0, c1):
    """What rows c0 .. c1 of a product's weight take of its operands. A bias may have any shape; what the epilogue does not read
    stays as it is (glu_clip's bias holds the unit's parameters)."""
    o = slice(c0 // 2, c1 // 2) if epi in PAIR_EPI else slice(c0, c1)
    return (w[c0:c1], bias.view(-1)[o] if "bias" in epi else bias, resid[:, o] if "resid" in epi else resid, out[:, o])


_TILE_LD = ~(2 ** 21 - 8)  # bits that no row stride has which _tile_rows leaves: starts off 16 bytes, rows from 4 MB on


def _tile_rows(x, w):
    """x and w, or copies of rows that gemm_mid and gemm_w4 cannot fetch where they lie: their LDS-DMA pieces start on 16 bytes,
    and a tile's 256 rows are reached by 32-bit offsets. (One look at both: this is host time of every product.)"""
    if not ((x.data_ptr() | w.data_ptr()) & 15 or (x.stride(0) | w.stride(0)) & _TILE_LD):
        return x, w
    return tuple(t.clone(memory_format=torch.contiguous_format) if t.data_ptr() & 15 or t.stride(0) & _TILE_LD else t
                 for t in (x, w))


def _gemm_rows(x, w, bias, resid, epi, out, out_f32, r0, r1, mi, S):
    """Rows r0 .. r1 of gemm() on gemm_mid's or gemm_w4's tile mi; operands checked by the caller."""
    M, K = r1 - r0, x.shape[1]
    N = w.shape[0] // 2 if epi in PAIR_EPI else w.shape[0]
    ldx, ldo = x.stride(0), out.stride(0)
    ldr = resid.stride(0) if resid is not None else 0
    px, po = x.data_ptr() + r0 * ldx * 2, out.data_ptr() + r0 * ldo * out.element_size()
    pr = resid.data_ptr() + r0 * ldr * 2 if resid is not None else None
    args = (px, ldx, w.data_ptr(), w.stride(0), po, ldo, ptr(bias), pr, ldr, M, N, K, EPI[epi], int(out_f32))
    if mi in W4_TILES:
        check(_lib.lib().ragk_gemm_w4_tile(*args, mi & 15 or 8, stream_ptr()), "ragk_gemm_w4_tile")
        return
    ws = torch.empty(S * M * w.shape[0], dtype=torch.float32, device=x.device) if S > 1 else None
    check(_lib.lib().ragk_gemm_mid(*args, mi, S, ptr(ws), stream_ptr()), "ragk_gemm_mid")


# Microseconds that one 64-deep K-tile of an output tile takes with few blocks running, and what a full machine adds
# (clocks, L2). Tiles of gemm_mid by rows / 32 (+ 16: of 256 columns, not 128), gemm_w4's by 32 + rows / 32 (always 256 columns),
# its 256 x 256 as 0; below, those of a launch and of a tile's epilogue. Fitted to every tile and split of 20 weights (384 to
# 28672 rows, K 384 to 14336) at 65 .. 32768 rows of x on two cards, for the choices that follow: they take 0.5 % more than the
# best launch in the mean, 4 % in one of twenty. (An earlier fit, with 0.25 added at 160 rows and one us for either epilogue, took
# the next tile up there: 1 and 8 %, and 12 % more than gemm_w4 alone at 2600 x 4096 x 14336.) 224 x 128 and 160 x 256 were fitted
# later to 46 products of 90 .. 8000 rows: with them the choices take 3 % less in the mean, 20 % less at best (600 x 4096 x
# 14336). gemm_w4's three to 166 of 66 .. 16000 rows (0.4 % over the best launch in the mean): on a full
# machine all of them reach the same 1.35 to 1.45 PFLOP/s, so what decides is the last round, and the epilogue where K is short.
MID_US = {3: (0.27, 0.13), 4: (0.34, 0.15), 5: (0.40, 0.17), 6: (0.49, 0.17), 7: (0.54, 0.21), 8: (0.62, 0.21), 21: (0.76, 0.20),
          38: (0.72, 0.39), 39: (0.84, 0.42), 0: (0.87, 0.55)}
W4_TILES = (0, 38, 39)
W4_SPLIT_US = (1.01, 0.29)  # gemm_w4 writing fp32 slabs (256 rows a tile only)
MID_TILES = tuple(mi for mi in MID_US if mi not in W4_TILES)
LAUNCH_US = (4.5, 1.75)
W4_LAUNCH_US = (5.25, {0: 4.25, 38: 2.0, 39: 2.6})
SLAB_US = 8 / 5e6  # one fp32 slab value written and read back


def _tiles_us(M, rows, K, mi, S, cus):
    """Model time of one launch: rounds of tiles over the CUs, each K-tiles long plus an epilogue."""
    bm, bn = 32 * (mi & 15 or 8), 128 if 0 < mi < 16 else 256
    items = -(-M // bm) * -(-rows // bn) * S
    rounds = -(-items // cus)
    a, b = W4_SPLIT_US if mi == 0 and S > 1 else MID_US[mi]
    launch, epilogue = (W4_LAUNCH_US[0], W4_LAUNCH_US[1][mi]) if mi in W4_TILES else LAUNCH_US
    return launch + rounds * (-(-(K // 64) // S) * (a + b * items / (rounds * cus)) + epilogue)


def _mid_best(M, rows, K, cus, slab_us, launch_us, even=False, most=16):
    """(time, mi, S) of the best gemm_mid launch of up to `most` slabs; a split costs launch_us and slab_us per slab value (even:
    equal slabs)."""
    best = (float("inf"), 0, 1)
    for mi in MID_TILES:
        for S in range(1, most + 1):
            if S > 1 and K // 64 // S < 4:
                break
            if even and K // 64 % S:
                continue
            t = _tiles_us(M, rows, K, mi, S, cus) + (launch_us + slab_us * S * M * rows if S > 1 else 0)
            best = min(best, (t, mi, S))
    return best


@functools.lru_cache(maxsize=4096)
def gemm_plan(M, rows, K, w4, cus, split=True):
    """Launches of one product with M > 64 rows: [(first row, end, mi, S)], mi as in MID_US (split: S may be above 1). Candidates:
    gemm_mid alone; gemm_w4 alone (w4: its operands fit), at 256, 224 or 192 rows a tile; its 256-row tiles on as many rows as
    fill whole rounds and gemm_mid on the rest. Where they meet (us, N = K = 4096): 300 rows 24 against gemm_w4's 69, 1777 rows 53
    against 66 (192 rows a tile); at N = 28672 of 1777 rows gemm_w4 322 against 350 (its wave tiles read less LDS per MFMA)."""
    return _timed_plan(M, rows, K, w4, cus, split)[1]


@functools.lru_cache(maxsize=4096)
def gemm_columns(M, rows, K, cus):
    """Weight rows (a multiple of 256) that one plan takes, the others a second one, or 0: where all tiles are little more than
    whole rounds (1777 x 28672: 784 of 256 x 256, three rounds and 16), gemm_w4 on as many columns of tiles as fill the rounds
    and the best plan for the rest. Only products that are summed over K in one piece, with and without the cut: then it changes
    no bit, and gemm_rope_kv and the native encoder forward, which do not ask here, agree with gemm. (Encoders of 384 and 1024
    columns are never cut, of the widths that gemm_rope_kv serves 6144 x 4096 at 2690 .. 2880 rows, for 2 %.) Us: 1777 x 28672 x
    4096 322 -> 310, 1548 x 28672 x 4096 301 -> 281, 1297 x 11264 x 2048 62 -> 56. It cuts 30 of 1284 products drawn from 12
    weights at 66 to 16000 rows; these took 0.81 to 1.015 of the time, 0.95 in the mean (those modelled at 0.95 to 0.96: 0.96 to
    1.015)."""
    if K % 64 or K < 192:
        return 0
    t, plan = _timed_plan(M, rows, K, True, cus)
    if any(S > 1 for _, _, _, S in plan):
        return 0
    t, n1 = COLUMNS_GAIN * t, 0
    for mi in W4_TILES:
        tiles_m = -(-M // (32 * (mi & 15 or 8)))
        c = tiles_m * -(-rows // 256) // cus * cus // tiles_m * 256
        if 0 < c < rows:
            t2 = _timed_plan(M, c, K, True, cus, False)[0] + _timed_plan(M, rows - c, K, True, cus, False)[0]
            if t2 < t:
                t, n1 = t2, c
    return n1


COLUMNS_GAIN = 0.96  # modelled time that a second launch has to save


@functools.lru_cache(maxsize=8192)
def _timed_plan(M, rows, K, w4, cus, split=True):
    """(modelled time, launches) of gemm_plan."""
    most = 16 if split else 1
    t, mi, S = _mid_best(M, rows, K, cus, SLAB_US, 3.0, most=most)
    plan = ((0, M, mi, S),)
    if not w4 or K % 64 or K < 192:  # gemm_w4's ring needs three K-tiles
        return t, plan
    full = _tiles_us(M, rows, K, 0, 1, cus)
    if full < t:
        t, plan = full, ((0, M, 0, 1),)
    tn = -(-rows // 256)
    rounds = -(-M // 256) * tn // cus
    for r in range(max(1, rounds - 1), rounds + 1):
        m1 = r * cus // tn * 256
        if not 0 < m1 < M:
            continue
        t2, mi, S = _mid_best(M - m1, rows, K, cus, SLAB_US, 3.0, most=most)
        t2 += _tiles_us(m1, rows, K, 0, 1, cus)
        # two launches have to earn their keep: of 57 such plans the five modelled at 0.96 to 0.97 of gemm_w4 alone took 0.99 to
        # 1.05 of it (827 x 28672 x 4096 188 us against 180), the others 0.69 to 1.02, 0.88 in the mean
        if t2 < 0.96 * t:
            t, plan = t2, ((0, m1, 0, 1), (m1, M, mi, S))
    # its smaller tiles, where they are well ahead. Against 256 rows: of 70 products of 1500 to 16384 rows those modelled at 0.97
    # to 1 took 0.985 to 1.10 of it, 192 rows from 0.95 on 0.97 to 1.04, the others 0.88 to 0.96; 44 more of 5348 to 16092 rows
    # whose last round of 256 rows is all but empty, 224 rows modelled at 0.97 to 0.99, took 0.98 to 1.08 of it, 1.009 in the mean
    # (14076 x 28672 x 4096 2282 against 2255 us). Against two launches: 14076 x 4096 x 4096 both ways 343 us, modelled 0.985.
    limit = {38: 0.97, 39: 0.97} if len(plan) > 1 else {}
    if plan == ((0, M, 0, 1),):
        limit = {38: 0.95, 39: 0.97}
    score, t3, mi = min((us / limit.get(mi, 1), us, mi) for mi in W4_TILES[1:] for us in [_tiles_us(M, rows, K, mi, 1, cus)])
    if score < t:
        t, plan = t3, ((0, M, mi, 1),)
    return t, plan


PART_MIN_BLOCKS = 512


@functools.lru_cache(maxsize=4096)
def _part_ksteps(M, N, K, min_blocks):
    check(_lib.lib().ragk_gemm_part_set_min_blocks(min_blocks), "ragk_gemm_part_set_min_blocks")
    return _lib.lib().ragk_gemm_part_ksteps(M, N, K)


def gemm_part_slabs(M, N, K, ks=None):
    """(ks_steps, S) of the split-K partial GEMM for this shape (0, 0 if unsupported)."""
    ks = ks or _part_ksteps(M, N, K, PART_MIN_BLOCKS)
    if ks <= 0 or K % (64 * ks):
        return 0, 0
    return ks, K // (64 * ks)


def _fp8_halves(M, N, ks, S):
    """Whether fp8 products take slices half as long as (ks, S): up to 16 rows, where their blocks are little more than whole rounds of
    two a CU, the last of which so leaves most of the chip without work. Us at 1 / 4 / 11 / 16 rows: 9216 x 4096 11.1 / 11.7 / 12.2 /
    12.6 -> 10.0 / 10.5 / 10.7 / 11.3, 18688 x 4096 20.7 / 21.6 / 22.3 / 22.7 -> 18.1 / 19.8 / 19.5 / 20.1, 7168 x 5120 11.4 / 11.9 /
    12.5 / 13.0 -> 10.0 / 10.5 / 11.1 / 11.7, 10240 x 8192 20.8 / 22.1 / 22.5 / 22.7 -> 18.6 / 22.6 / 21.4 / 21.5; in full rounds they
    lose (12288 x 4096 13.6 against 15.0 at 11 rows). More rows read more of x for shorter slices: 18688 x 4096 at 17 21.8, 23.9.
    At four to six rows of weights 8 KB and more apart the halves' gain shrinks with their number, as nowhere else: 8448 x 8192, 528
    blocks, 19.5 / 19.5 / 19.6 -> 18.0 / 18.1 / 18.1, 576 of 9216 x 8192 and 4608 x 16384 19.8 / 19.8 / 19.9 -> 20.1 / 19.6 / 18.9 and 19.7 /
    19.2 / 18.9, 640 of 10240 x 8192 and 5120 x 16384 20.5 / 20.6 / 20.8 against 21.3 / 21.4 / 21.0 (three and seven rows 20.3 -> 18.4,
    20.8 -> 20.6; 576 of 6144 x 12288 and 640 of 20480 x 4096 gain 7 and 6 % there): they end at 0.6 of a round."""
    blocks = -(-N // 64) * S
    most = 0.6 if 4 <= M <= 6 and 64 * ks * S % 8192 == 0 else 0.65
    return M <= 16 and ks in (16, 32) and blocks < most * -(-blocks // PART_MIN_BLOCKS) * PART_MIN_BLOCKS


def gemm_part_norm(h, gamma, eps, w, out=None, ks=None):
    """gemm_part of rmsnorm(h) * gamma (the norm applied inside the GEMM's activation staging, same
    math as rmsnorm): decode batches <= 4, bf16 weights, K <= 8192."""
    _bf16_2d(h, "h")
    _bf16_2d(w, "w")
    M, K = h.shape
    N = w.shape[0]
    _req(w.shape[1] == K and M <= 4 and K <= 8192 and gamma.numel() == K and gamma.dtype == torch.bfloat16
         and gamma.is_contiguous(), "gemm_part_norm shape")
    ks, S = gemm_part_slabs(1, N, K, ks)
    if ks not in (8, 16):  # the norm variant is built for 8- and 16-step K-slices
        ks, S = gemm_part_slabs(1, N, K, 16)
    _req(S > 0 and K in (4096, 8192), "gemm_part_norm: unsupported K=%d" % K)
    if out is None:
        out = torch.empty((S, M, N), dtype=torch.float32, device=h.device)
    check(_lib.lib().ragk_gemm_part_norm(h.data_ptr(), h.stride(0), gamma.data_ptr(), float(eps), w.data_ptr(),
                                         w.stride(0), out.data_ptr(), M, N, K, ks, stream_ptr()),
          "ragk_gemm_part_norm")
    return out


# Split-K partial slabs through the LDS-DMA weight ring (gemm_stream.hip SLAB) instead of gemm_part's
# register-streaming blocks, at decode batches above STREAM_PART_MIN_M: the down projection's 1792-deep
# activation slice needs 114 KB of LDS per gemm_part block at batch 32 (one block per CU, two rounds).
# Batch 32: decode step 7.35 / 7.33 -> 6.91 / 6.98 ms, bench 1568 / 1570 -> 1597 / 1595 tok/s (same box,
# alternating; profiles/bench_stream_part_ab_r4.log).
STREAM_PART = True
STREAM_PART_MIN_M = 5  # batch 8 / 16 -3 %, batch 4 +0.6 %; below, where _part_stream says
STREAM_PART_ROWS = 0  # 0: by occupancy (ties: 128)
STREAM_PART_MAX_S = 64  # slabs the consumer sums


def stream_part_cfg(M, N, K):
    """(rows, S) of the slab-mode stream GEMM."""
    return _stream_part_cfg(N, K, _cu_count(), STREAM_PART_ROWS, STREAM_PART_MAX_S)


@functools.lru_cache(maxsize=1024)
def _stream_part_cfg(N, K, cus, only, max_s):
    """(rows, S) of the slab-mode stream GEMM: the most blocks that are co-resident (128-row tiles one
    block per CU, 64-row tiles two), at least 8 K-steps of 64 per block; (0, 0) if nothing fits."""
    steps = K // 64
    best = (0, 0, 0)
    for rows, per_cu in ((128, 1), (64, 2)):
        if only and rows != only:
            continue
        tiles = -(-N // rows)
        S = 1
        while (tiles * S * 2 <= per_cu * cus and steps % (S * 2) == 0 and steps // (S * 2) >= 8
               and S * 2 <= max_s):
            S *= 2
        blocks = tiles * S
        if blocks <= per_cu * cus and (blocks / per_cu, rows) > (best[2], best[0]):
            best = (rows, S, blocks / per_cu)
    # a grid that fills less than half the CUs (tensor-parallel shards: o_proj K = 512 cannot be split
    # into 8-step slices) stays on gemm_part, whose 64-column blocks split finer
    if best[2] < 0.5 * cus:
        return 0, 0
    # half the chip, or slices as short as the ring is deep: 64-row tiles at one block a CU instead, with as many slabs or half
    # of them (12 rows: 2048 x 5632 8.9 -> 7.1 us, 4096 x 4096 9.3 -> 8.3, 4096 x 7168 12.5 -> 12.2; from 16 steps a slice on
    # the wider tile is ahead: 4096 x 8192 14.3 against 16.4)
    if best[0] == 128 and (best[2] < cus or steps // best[1] < 16):
        tiles, S = -(-N // 64), 1
        while tiles * S * 2 <= cus and steps % (S * 2) == 0 and steps // (S * 2) >= 8 and S * 2 <= max_s:
            S *= 2
        if 0.9 * cus <= tiles * S <= cus:
            return 64, S
    return best[0], best[1]


def _deep_slabs(N, K, cus, only, max_s, few):
    """Slabs of 64-row tiles where stream_part_cfg's blocks, one round of them, leave more than a third of the CUs without work for
    slices of 32 K-steps and more: several rounds of slices half as long and shorter, dealt as places come free. 0: not here. Us, one
    round -> these, at 8 / 17 / 33 / 64 rows: 18688 x 4096 31.9 / 34.0 / 37.9 / 44.4 -> 27.4 / 28.1 / 31.9 / 36.9, 17408 x 4096 31.6 /
    33.4 / 33.3 / 37.8 -> 26.5 / 26.8 / 30.6 / 35.2, 18688 x 8192 69 / 68 / 72 / 78 -> 62 / 62 / 70 / 76, 18688 x 2048 18.9 / 20.1 /
    22.6 / 25.8 -> 17.8 / 17.7 / 19.4 / 22.0; two slabs only up to 32 rows (`few`): 10240 x 8192 38.2 / 39.3 / 38.2 / 41.8 -> 35.4 /
    35.7 / 39.1 / 42.5, 9216 x 4096 18.8 / 20.0 -> 17.8 / 17.6. From 22528 x 4096 on one round is ahead at 33 rows (36.0 against
    38.6), and at half-full slices of 16 steps always (9344 x 2048 10.8 against 11.3). At the rule's edge, 20480 rows of weights, the two
    change places from run to run from 24 rows on (x 8192 at 24 / 64 rows +1 / +6 and -3 / -1 %, x 4096 -7 / +4 and -7 / +5); rows with a gap
    stream better in one round (5 / 8 / 16 / 17 rows of 9216 x 4096 +3 / +2 / +1 / -3 %, 18688 x 2048 +3 / +2 / 0 / -3). Both keep several,
    whose sums are two to four times as close (1.3 and 0.95e-7 against 2.7e-7); one round in short sums takes up to 12 % more."""
    rows, S = _stream_part_cfg(N, K, cus, only, max_s)
    steps = K // 64
    if rows != 128 or -(-N // 128) * S > 0.64 * cus or steps // S < 32 or not (S == 1 or (S == 2 and few)):
        return 0
    deep = S
    while steps % (2 * deep) == 0 and steps // (2 * deep) >= 14 and 2 * deep <= max_s:
        deep *= 2
    return deep if deep > S else 0


@functools.lru_cache(maxsize=4096)
def _part_stream(M, N, K, cus, min_m, only, max_s, min_blocks):
    """(rows, S, whether in short sums) of gemm_part's bf16 products on the LDS-DMA weight stream, S 0: gemm_part.hip's.

    Below STREAM_PART_MIN_M rows they go there only where gemm_part.hip's slices are 28 K-steps long and more, in sums over 512 of K,
    which are no further off (1 / 4 rows, us and rms error in 1e-7: 4096 x 14336 24.9 / 25.2, 1.7 -> 22.0 / 22.0, 1.3; 18688 x 4096
    35.3 / 35.8, 1.9 -> 28.2 / 27.1, 1.3; 8192 x 28672 92.5 / 93.8, 1.8 -> 75 / 75, 1.4; 6144 x 14336 44 -> 32). Shorter slices are as
    fast there, in shorter sums, and so are whole rounds of two blocks a CU over rows a multiple of 16 KB apart (8192 x 8192 31.3
    against 32.6, 4096 x 16384 32.5 against 34.8, 8192 x 16384 61 against 64, 16384 x 8192 56 against 66, but 10240 x 8192 in 1.25 rounds
    39 -> 36, 17408 x 8192 in 1.1 63 -> 59; such rows never have a gap, ops/pitch.py). Slabs of
    _deep_slabs are short sums, too: 18688 x 4096 in one 3.9e-7, in four of 1024 1.8, of 512 1.3, for 0 to 3 % of the time."""
    few = M < min_m
    if K % 64 or N % 4:
        return 0, 0, False
    if few:
        ks = _part_ksteps(M, N, K, min_blocks)
        if ks < 28 or (K % 8192 == 0 and -(-N // 64) * (K // (64 * ks)) % (2 * cus) == 0):
            return 0, 0, False
    deep = _deep_slabs(N, K, cus, only, max_s, M <= 32)
    return (64, deep, True) if deep else _stream_part_cfg(N, K, cus, only, max_s) + (few,)


def gemm_stream_part(x, w, out=None, rows=None, S=None, short_sums=False):
    """Partial slabs P[S, M, N] (fp32) with P.sum(0) = x @ w^T from the LDS-DMA stream GEMM (bf16 weights). short_sums: a slab is
    the sum of sums over 512 of K (256 up to 2048)."""
    _bf16_2d(x, "x")
    _bf16_2d(w, "w")
    M, K = x.shape
    N = w.shape[0]
    _req(w.shape[1] == K and M <= 64 and K % 64 == 0 and N % 4 == 0, "gemm_stream_part shape")
    r0, s0 = stream_part_cfg(M, N, K)
    rows, S = rows or r0, S or s0
    _req(rows in (64, 128) and S >= 1 and (K // 64) % S == 0, "gemm_stream_part config")
    if out is None:
        out = torch.empty((S, M, N), dtype=torch.float32, device=x.device)
    check(_lib.lib().ragk_gemm_stream_part(x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), out.data_ptr(), M, N,
                                           K, S, rows, int(short_sums), stream_ptr()), "ragk_gemm_stream_part")
    return out


def gemm_part(x, w, out=None, ks=None, short_sums=False):
    """Decode GEMM v5 (csrc/kernels/gemm_part.hip): fp32 split-K partials P[S, M, N] with
    P.sum(0) = x @ w^T. The consumer (add_partials_rmsnorm / rope_kv_partials) does the reduction.
    w: bf16 [N, K], or an :class:`ops.fp8.Fp8Weight` (W8A16: e4m3fn rows, per-row scale applied to
    the partials). short_sums: for results that were products of rows before, whose sums were no longer than 512 of K = 4096
    (gemm_stream_part)."""
    from .fp8 import Fp8Weight

    _bf16_2d(x, "x")
    fp8 = isinstance(w, Fp8Weight)
    wt = w.w8 if fp8 else w
    if fp8:
        _req(wt.is_cuda and wt.dim() == 2 and wt.stride(1) == 1 and wt.element_size() == 1, "fp8 weight rows")
        _req(w.scale.dtype == torch.float32 and w.scale.is_contiguous(), "fp8 weight scales fp32")
    else:
        _bf16_2d(wt, "w")
    M, K = x.shape
    N = wt.shape[0]
    _req(wt.shape[1] == K and M <= 64, "gemm_part shape %s x %s" % (tuple(x.shape), tuple(wt.shape)))
    if STREAM_PART and not fp8 and ks is None and out is None:
        rows, S, short = _part_stream(M, N, K, _cu_count(), STREAM_PART_MIN_M, STREAM_PART_ROWS, STREAM_PART_MAX_S, PART_MIN_BLOCKS)
        if S > 0 and (M >= STREAM_PART_MIN_M or _vec_rows(x, wt)):
            return gemm_stream_part(x, wt, rows=rows, S=S, short_sums=short_sums or short)
    if fp8 and ks is None and out is None and use_hold_slabs(M, N, K) and _vec_rows(x, wt) and wt.stride(0) < 1 << 24:
        return gemm_hold_slabs(x, wt, w.scale)
    chosen = ks is None and out is None
    ks, S = gemm_part_slabs(M, N, K, ks)
    _req(S > 0, "gemm_part: unsupported K=%d" % K)
    if fp8 and chosen and _fp8_halves(M, N, ks, S):
        ks, S = ks // 2, 2 * S
    if out is None:
        out = torch.empty((S, M, N), dtype=torch.float32, device=x.device)
    _req(out.dtype == torch.float32 and out.is_contiguous() and out.numel() >= S * M * N, "gemm_part out")
    if fp8:
        check(_lib.lib().ragk_gemm_part_fp8(x.data_ptr(), x.stride(0), wt.data_ptr(), wt.stride(0),
                                            w.scale.data_ptr(), out.data_ptr(), M, N, K, ks, stream_ptr()),
              "ragk_gemm_part_fp8")
    else:
        check(_lib.lib().ragk_gemm_part(x.data_ptr(), x.stride(0), wt.data_ptr(), wt.stride(0), out.data_ptr(), M, N,
                                        K, ks, stream_ptr()), "ragk_gemm_part")
    return out[:S] if out.dim() == 3 else out


PREFILL_SPLITK = True
# measured: M = 5.2k (one RAG prompt) 2 slabs win (o_proj + down 760 -> 656 us per layer); a ~2.2k-token
# tail step with 4 slabs was no faster than unsplit in the bench profile -> split only M >= 4096, 2 slabs
PREFILL_SPLITK_MIN_M = 4096
_n_cus = [0]


def _cu_count():
    if not _n_cus[0]:
        try:
            _n_cus[0] = torch.cuda.get_device_properties(torch.cuda.current_device()).multi_processor_count
        except Exception:
            _n_cus[0] = 256
    return _n_cus[0]


def prefill_nsplit(M, N, K):
    """K-slabs of gemm_w4 alone (its KSPLIT form) by how full its 256x256 tiles leave the CUs: the split with the best
    wave efficiency (tiles / (waves * CUs)), 2 % charged per extra slab for the fp32 slab traffic; 1 = no split. 5200 rows,
    N = 4096: 336 tiles = 1.31 waves (66 %) -> 2 slabs = 2.6 waves (88 %). slab_count weighs it against gemm_mid's tiles: there
    those rows take no split, gemm_w4 on 4096 of them and gemm_mid on the rest."""
    if not PREFILL_SPLITK or M < PREFILL_SPLITK_MIN_M:
        return 1
    return _w4_nsplit(M, N, K, _cu_count())


def _w4_nsplit(M, N, K, cus):
    tiles = -(-M // 256) * -(-N // 256)
    best, best_s = 0.0, 1
    for s in (1, 2):
        if K % (64 * s) or K // s < 4 * 64:
            continue
        wt = tiles * s
        eff = wt / (-(-wt // cus) * cus) - 0.02 * (s - 1)
        if eff > best + 1e-9:
            best, best_s = eff, s
    return best_s


@functools.lru_cache(maxsize=4096)
def _slab_best(M, N, K, cus, w4_min_m=PREFILL_SPLITK_MIN_M):
    """(S, mi) of the cheapest split whose slabs a row norm sums, (1, 0) if the whole product + a plain norm is cheaper.
    Per output value the slabs cost 8 B each through memory, the whole product 6 (bf16 write, residual, norm's read).
    o_proj / down at 300 rows: 28 / 88 us whole, 17 / 42 us as 2 / 4 slabs; at 14076 rows the slabs' traffic (212 us in the
    norm) is more than the last round that they would fill."""
    whole = 0.0
    for r0, r1, mi, S in gemm_plan(M, N, K, True, cus):
        whole += _tiles_us(r1 - r0, N, K, mi, S, cus) + (3.0 + SLAB_US * S * (r1 - r0) * N if S > 1 else 0)
    best, S, mi = min((t - 0.75 * SLAB_US * M * N, S, mi) for t, mi, S in [_mid_best(M, N, K, cus, SLAB_US, 0.0, even=True)])
    w4 = _w4_nsplit(M, N, K, cus) if M >= w4_min_m else 1
    if w4 > 1:
        t = _tiles_us(M, N, K, 0, w4, cus) + SLAB_US * (w4 - 0.75) * M * N
        if t < best:
            best, S, mi = t, w4, 0
    return (S, mi) if S > 1 and best < whole else (1, 0)


def slab_count(M, N, K):
    """K-slabs for a prefill projection in front of a row norm (1: the whole product)."""
    if not PREFILL_SPLITK or M <= 64 or K % 128 or N % 8:
        return 1
    return _slab_best(M, N, K, _cu_count(), PREFILL_SPLITK_MIN_M)[0]


@functools.lru_cache(maxsize=4096)
def _splitk_tile(M, N, K, nsplit, cus):
    """(gemm_mid's tile, whether gemm_w4 is ahead of it) for nsplit slabs."""
    t, mi = min((_tiles_us(M, N, K, m, nsplit, cus), m) for m in MID_TILES)
    return mi, _tiles_us(M, N, K, 0, nsplit, cus) < t


def gemm_splitk(x, w, nsplit, out=None):
    """fp32 split-K slabs P[nsplit, M, N] with P.sum(0) = x @ w^T in one launch, consumed by add_partials_rmsnorm (residual
    add + norm). gemm_mid or gemm_w4's KSPLIT form, whichever the launch model puts first."""
    _bf16_2d(x, "x")
    _bf16_2d(w, "w")
    M, K = x.shape
    N = w.shape[0]
    _req(w.shape[1] == K and K % (64 * nsplit) == 0 and K // nsplit >= 256 and N % 8 == 0, "gemm_splitk shape")
    if out is None:
        out = torch.empty((nsplit, M, N), dtype=torch.float32, device=x.device)
    _req(out.dtype == torch.float32 and out.is_contiguous() and out.numel() >= nsplit * M * N, "gemm_splitk out")
    if M == 0:
        return out
    x, w = _tile_rows(x, w)
    mi, w4 = _splitk_tile(M, N, K, nsplit, _cu_count())
    if w4 and x.stride(0) * M * 2 < 2 ** 31 and w.stride(0) * N * 2 < 2 ** 31:
        check(_lib.lib().ragk_gemm_w4_splitk(x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), out.data_ptr(), M, N, K,
                                             nsplit, stream_ptr()), "ragk_gemm_w4_splitk")
    else:
        check(_lib.lib().ragk_gemm_mid(x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), out.data_ptr(), N, None, None, 0,
                                       M, N, K, EPI["none"], 2, mi, nsplit, None, stream_ptr()), "ragk_gemm_mid")
    return out


def gemm_part_merge_ok(M, w, Hq, max_parts, ws_o):
    """Whether the o_proj split-K GEMM can merge the decode attention's partitions itself
    (gemm_part.hip MergeArgs): batch <= 4, head dim 128, a partition workspace present."""
    from .fp8 import Fp8Weight

    if ws_o is None or max_parts < 2:
        return False
    wt = w.w8 if isinstance(w, Fp8Weight) else w
    N, K = wt.shape
    ks, S = gemm_part_slabs(M, N, K)
    return S > 0 and bool(_lib.lib().ragk_gemm_part_merge_ok(M, K, Hq, max_parts, ks))


def gemm_part_merge(attn_out, kv_lens, part_tiles, max_parts, ws_o, ws_ml, Hq, w, out=None):
    """o_proj partials P[S, M, N] = merge(attention partitions) @ w^T: the decode attention ran with its
    split-K merge deferred (attn_decode_rope(..., defer_merge=True)) and every GEMM block merges the
    heads of its K-slice from ws_o / ws_ml (attn_decode_reduce's math); rows with a single partition
    are read from attn_out, where the attention kernel wrote them. Replaces the reduce launch."""
    from .fp8 import Fp8Weight

    fp8 = isinstance(w, Fp8Weight)
    wt = w.w8 if fp8 else w
    M = kv_lens.numel()
    N, K = wt.shape
    _req(attn_out.dtype == torch.bfloat16 and attn_out.stride(1) == 1 and attn_out.shape[0] >= M
         and attn_out.shape[1] == K, "attention output rows")
    _req(ws_o is not None and ws_o.dtype == torch.float32 and ws_o.numel() >= M * Hq * max_parts * 128
         and ws_ml.numel() >= M * Hq * max_parts * 2, "partition workspace")
    ks, S = gemm_part_slabs(M, N, K)
    _req(S > 0 and _lib.lib().ragk_gemm_part_merge_ok(M, K, Hq, max_parts, ks), "gemm_part_merge shape")
    if out is None:
        out = torch.empty((S, M, N), dtype=torch.float32, device=attn_out.device)
    check(_lib.lib().ragk_gemm_part_merge(
        ws_o.data_ptr(), ws_ml.data_ptr(), attn_out.data_ptr(), attn_out.stride(0), kv_lens.data_ptr(), Hq,
        part_tiles, max_parts, wt.data_ptr(), wt.stride(0), w.scale.data_ptr() if fp8 else None, out.data_ptr(), M, N,
        K, ks, stream_ptr()), "ragk_gemm_part_merge")
    return out


SILU_MAX_SLABS = 4  # gemm_part.hip SG_MAXS


def gemm_part_gu_ks(K):
    """K-slice steps of the packed gate/up partial GEMM feeding gemm_part_silu: at most SILU_MAX_SLABS
    slabs. (8 slabs: the TP=8 shard's gate/up 8.2 -> 7.9 us with 448 blocks, but the down GEMM's
    staging of 8 slabs 7.2 -> 9.4 us; docs/PERF_NOTES.md, TP decode.)"""
    for ks in (4, 8, 16, 32):
        if K % (64 * ks) == 0 and K // (64 * ks) <= SILU_MAX_SLABS:
            return ks
    return 0


def _silu_ks(M, N, K):
    """K-slice steps of gemm_part_silu: the SG variant is built for 4/8/16-step slices with one staging
    item per thread (M * 8 * ks <= 512); as gemm_part_slabs, the widest slice reaching PART_MIN_BLOCKS."""
    legal = [ks for ks in (16, 8, 4) if K % (64 * ks) == 0 and M * 8 * ks <= 512]
    nb = -(-N // 64)
    for ks in legal:
        if nb * (K // (64 * ks)) >= PART_MIN_BLOCKS:
            return ks
    return legal[-1] if legal else 0


def gemm_part_silu_ok(M, w_gu, w_down):
    """Whether the down projection can take silu(gate) * up straight from the gate/up partial slabs."""
    if not (isinstance(w_gu, torch.Tensor) and isinstance(w_down, torch.Tensor)):
        return False
    N, K = w_down.shape
    ks_gu = gemm_part_gu_ks(w_gu.shape[1])
    if w_gu.shape[0] != 2 * K or K % 64 or ks_gu == 0 or M > 4:
        return False
    S1 = w_gu.shape[1] // (64 * ks_gu)
    ks = _silu_ks(M, N, K)
    return ks > 0 and bool(_lib.lib().ragk_gemm_part_silu_ok(M, S1, K, ks))


def gemm_part_gu(x, w_gu):
    """Split-K partials of the packed gate/up projection with at most SILU_MAX_SLABS slabs (gemm_part_silu's input)."""
    return gemm_part(x, w_gu, ks=gemm_part_gu_ks(x.shape[1]))


def gemm_part_silu(pgu, w, out=None):
    """Down-projection partials P[S, M, N] of silu(gate) * up, where gate / up are the sums of the slabs
    of pgu [S1, M, 2K] (gemm_part_gu output, packed [64 gate | 64 up] column tiles): the reduction and
    the activation happen in the down GEMM's LDS staging (gemm_part.hip SG) -- no silu_mul launch and
    the gate/up GEMM streams its weights split-K."""
    _bf16_2d(w, "w")
    _req(pgu.dtype == torch.float32 and pgu.is_cuda and pgu.is_contiguous() and pgu.dim() == 3, "pgu fp32 [S1, M, 2K]")
    S1, M, K2 = pgu.shape
    N, K = w.shape
    _req(K2 == 2 * K, "pgu holds packed gate/up columns of width 2K")
    ks = _silu_ks(M, N, K)
    _req(ks > 0 and _lib.lib().ragk_gemm_part_silu_ok(M, S1, K, ks), "gemm_part_silu shape")
    S = K // (64 * ks)
    if out is None:
        out = torch.empty((S, M, N), dtype=torch.float32, device=pgu.device)
    _req(out.shape == (S, M, N) and out.dtype == torch.float32, "out [S, M, N] fp32")
    check(_lib.lib().ragk_gemm_part_silu(pgu.data_ptr(), S1, w.data_ptr(), w.stride(0), out.data_ptr(), M, N, K, ks,
                                         stream_ptr()), "ragk_gemm_part_silu")
    return out


# ----------------------------------------------------------------------------- persistent decode MLP
# Batch-1 decode MLP as one persistent launch (csrc/kernels/mlp_engine.hip): h += W_down (silu(W_gate x) *
# (W_up x)) with both weight streams going through one LDS ring per CU (RAGK_MLP_ENGINE=0 turns it off). Batch-1 decode step 3.47 -> 3.34 ms (profiles/mlp_engine_r5.log).
MLP_ENGINE = os.environ.get("RAGK_MLP_ENGINE", "1") != "0"
_me_ws = {}


class _MeWorkspace:
    """One launch stream's engine state: act [I] bf16 (the hand-off), the monotonic arrival counters, the
    device error word (a set word makes later launches exit at entry), the deadline word (test hook) and a
    host-mapped pinned error word the engine reads after every step without a device sync."""

    def __init__(self, dev, I):
        L = _lib.lib()
        self.nb = int(L.ragk_mlp_engine_ctr_bytes())
        # int64 words: counters | error (u32 at byte nb) | deadline ticks (u32 at byte nb + 8)
        self.words = torch.zeros(self.nb // 8 + 2, dtype=torch.int64, device=dev)
        self.act = torch.zeros(I, dtype=torch.bfloat16, device=dev)
        self.host = L.ragk_host_word_alloc()
        _req(bool(self.host), "mlp_engine: hipHostMalloc of the host error word failed")
        self.host_dev = L.ragk_host_word_dev(self.host)
        _req(bool(self.host_dev), "mlp_engine: no device address for the host error word")
        import ctypes

        self._host_word = ctypes.c_uint.from_address(self.host)

    @property
    def err_ptr(self):
        return self.words.data_ptr() + self.nb

    @property
    def tmo_ptr(self):
        return self.words.data_ptr() + self.nb + 8

    def fault(self) -> int:
        return int(self._host_word.value)

    def rearm(self):
        """Zero the counters and both error words (the device must be idle: no launch of this workspace in
        flight)."""
        self.words[: self.nb // 8 + 1].zero_()
        self._host_word.value = 0

    def __del__(self):  # pragma: no cover - interpreter shutdown order
        try:
            if self.host:
                _lib.lib().ragk_host_word_free(self.host)
                self.host = None
        except Exception:
            pass


def _me_workspace(dev, I):
    """The workspace of the launching stream: two streams (two engines, or two captured graphs of one
    process) never share arrival counters. Allocated by an eager launch, never inside a hipGraph capture
    (a graph-pool allocation, with its zero-fill captured, would be handed to later eager launches after
    the graph is gone): warm up on the stream the graph is then captured on."""
    key = (str(dev), stream_ptr(), I)
    ws = _me_ws.get(key)
    if ws is None:
        _req(not torch.cuda.is_current_stream_capturing(),
             "mlp_engine workspace: run one eager step on the capture stream before capture")
        ws = _me_ws[key] = _MeWorkspace(dev, I)
    return ws


def mlp_engine_ok(M, w_gu, w_down):
    if not MLP_ENGINE or not (isinstance(w_gu, torch.Tensor) and isinstance(w_down, torch.Tensor)):
        return False
    if w_gu.dtype != torch.bfloat16 or w_down.dtype != torch.bfloat16 or not w_gu.is_cuda:
        return False
    H, I = w_down.shape
    if w_gu.shape != (2 * I, H) or not (_vec_rows(w_gu) and w_gu.stride(1) == 1 and w_gu.stride(0) >= H and w_down.is_contiguous()):
        return False
    return bool(_lib.lib().ragk_mlp_engine_rows_ok(M, H, I, _cu_count(), w_gu.stride(0)))


def mlp_engine(xn, w_gu, w_down, h):
    """h += W_down . (silu(gate) * up) for ONE row (xn = the post-attention RMSNorm of h, bf16 [1, H])."""
    _bf16_2d(xn, "xn")
    _req(xn.shape == (1, w_down.shape[0]) and xn.is_contiguous(), "xn [1, H]")
    return _mlp_engine_launch(xn.data_ptr(), None, 0, None, 0.0, w_gu, w_down, h)


def mlp_engine_tail(P, h, gamma, eps, w_gu, w_down):
    """The batch-1 post-attention tail in one launch: h += bf16(sum of the o_proj slabs P [S, 1, H]);
    x = rmsnorm(h) * gamma (add_partials_rmsnorm's math); h += W_down . (silu(gate) * up)."""
    H = w_down.shape[0]
    _req(P.dtype == torch.float32 and P.is_cuda and P.is_contiguous() and P.dim() == 3 and P.shape[1:] == (1, H),
         "P [S, 1, H] fp32")
    _req(gamma.dtype == torch.bfloat16 and gamma.is_contiguous() and gamma.numel() == H, "gamma [H] bf16")
    return _mlp_engine_launch(None, P.data_ptr(), P.shape[0], gamma.data_ptr(), float(eps), w_gu, w_down, h)


def _mlp_engine_launch(xn_ptr, P_ptr, S, g_ptr, eps, w_gu, w_down, h):
    _bf16_2d(h, "h")
    H, I = w_down.shape
    _req(h.shape == (1, H) and h.is_contiguous(), "h [1, H]")
    _req(mlp_engine_ok(1, w_gu, w_down), "mlp_engine shape")
    ws = _me_workspace(h.device, I)
    check(_lib.lib().ragk_mlp_engine(xn_ptr, P_ptr, S, g_ptr, eps, w_gu.data_ptr(), w_gu.stride(0), w_down.data_ptr(), h.data_ptr(),
                                     ws.act.data_ptr(), ws.words.data_ptr(), ws.err_ptr, ws.host_dev, ws.tmo_ptr, 1, H, I,
                                     _cu_count(), stream_ptr()),
          "ragk_mlp_engine")
    return h


def mlp_engine_fault(dev=None) -> int:
    """Error code of a persistent MLP launch on `dev` that gave up a wait (0 = healthy). Reads the
    host-mapped words only: no device sync, so the engine checks it after every step's event sync."""
    d = torch.device(dev) if dev is not None else None
    for key, ws in list(_me_ws.items()):
        if d is not None and d.index is not None and torch.device(key[0]) != d:
            continue
        e = ws.fault()
        if e:
            return e
    return 0


def mlp_engine_rearm(dev=None):
    """Re-arm every workspace on `dev` after a fault (call with the device idle)."""
    d = torch.device(dev) if dev is not None else None
    for key, ws in list(_me_ws.items()):
        if d is None or d.index is None or torch.device(key[0]) == d:
            ws.rearm()


def mlp_engine_check(dev=None):
    """Raise if a persistent MLP launch on `dev` timed out in a wait (then re-arm its counters). Syncs."""
    if not _me_ws:
        return
    torch.cuda.synchronize(dev)
    e = mlp_engine_fault(dev)
    if e:
        mlp_engine_rearm(dev)
        raise RuntimeError("persistent decode MLP: wait timed out (code %d); counters reset" % e)


def mlp_engine_force_timeout(ticks, dev=None):
    """Test hook: deadline of the following launches in s_memrealtime ticks (0 = the kernel's default). A
    device-side word written on the current stream, so launches captured in a hipGraph see it too."""
    d = torch.device(dev) if dev is not None else None
    for key, ws in list(_me_ws.items()):
        if d is None or d.index is None or torch.device(key[0]) == d:
            ws.words[ws.nb // 8 + 1].fill_(int(ticks))


def set_mlp_engine_nt(nt):
    check(_lib.lib().ragk_mlp_engine_set_nt(int(nt)), "ragk_mlp_engine_set_nt")


STREAM_S_OVERRIDE = 0  # tuning hook (tools/tune_stream.py)


def _gemm_stream(x, w, wscale, out, bias, resid, ldr, M, N, K, epi, e, out_f32):
    """Decode GEMM v4 (csrc/kernels/gemm_stream.hip): glds-ring weight streaming, split-K."""
    L = _lib.lib()
    fp8 = wscale is not None
    S = STREAM_S_OVERRIDE or L.ragk_gemm_stream_splits(N, K, e, int(fp8))
    ws, cnt = dec_workspace(x.device)
    rows = 2 * N if epi in PAIR_EPI else N
    _req(S == 1 or S * M * (-(-rows // 128) * 128) <= ws.numel(), "stream GEMM workspace too small")
    _req(-(-rows // 64) <= cnt.numel(), "too many n-tiles for the counter buffer")
    return L.ragk_gemm_stream(x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), ptr(wscale), out.data_ptr(),
                              out.stride(0), ptr(bias), ptr(resid), ldr, M, N, K, e, int(out_f32), S, ws.data_ptr(),
                              cnt.data_ptr(), stream_ptr())


def _gemm_slabs(x, w, out, bias, resid, ldr, M, N, K, e):
    """gemm() of at most 64 rows through the stream GEMM's fp32 slabs."""
    rows, S = stream_part_cfg(M, N, K)
    ws = torch.empty(S * M * N, dtype=torch.float32, device=x.device)
    check(_lib.lib().ragk_gemm_slabs(x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), out.data_ptr(), out.stride(0),
                                     ptr(bias), ptr(resid), ldr, M, N, K, e, S, rows, ws.data_ptr(), stream_ptr()),
          "ragk_gemm_slabs")
    return out


@functools.lru_cache(maxsize=256)
def _hold_rows(K, fp8):
    return _lib.lib().ragk_gemm_hold_rows(K, int(fp8))


def use_hold(M, N, K, epi, fp8=False):
    """Packed gate/up projections whose activations fit a block's registers go to gemm_hold.hip: 11264 x 2048 bf16 at 12 / 50
    rows 14.7 / 24 -> 11.1 / 16.5 us against the register-streaming kernel, 28672 x 4096 fp8 at 11 / 32 rows 38 / 37 -> 26 / 31
    (gemm_fp8_dec / gemm_stream). Not where they lose: K of 1024 (a barrier for every 16 KB of weights: 28672 rows 10.3 against
    8.7); row tiles that leave the last of a CU's few rounds mostly empty (6144 x 3072 bf16, 1.5 rounds: 11.9 against 11.4);
    bf16 weights that the LDS ring streams without a K-split (28672 x 4096: 43 against 42); and more rows than one launch
    holds, but for 8192 rows of fp8 and up that use_hold_slabs_silu leaves (K = 3072), whose second launch reads the Infinity
    Cache while the ring is down to half its depth."""
    if not 0 < M <= 64 or K < 2048 or epi not in PAIR_EPI or (fp8 and epi != "silu_mul"):
        return False
    per = _hold_rows(K, fp8)
    if per == 0 or not (M <= per or (fp8 and 32 < M <= 2 * per and 2 * N >= 8192)):
        return False
    tiles, cus = N // 8, _cu_count()
    if tiles > cus and tiles < (0.6 if fp8 else 0.78) * (-(-tiles // cus) * cus):
        return False
    return fp8 or not use_stream(M, N, K, epi) or _lib.lib().ragk_gemm_stream_splits(N, K, EPI[epi], 0) > 1


def _vec_rows(*ts):
    """Whether every row starts on 16 bytes."""
    return all((t.stride(0) * t.element_size()) % 16 == 0 and t.data_ptr() % 16 == 0 for t in ts)


def gemm_hold(x, w, wscale=None, par=None, epi="silu_mul", out=None):
    """Packed gate/up projection of at most 64 rows with the activations held in registers (gemm_hold.hip); more rows than
    one launch holds go in equal launches."""
    L = _lib.lib()
    M, K = x.shape
    N = w.shape[0] // 2
    if out is None:
        out = torch.empty((M, N), dtype=torch.bfloat16, device=x.device)
    per = _hold_rows(K, wscale is not None)
    _req(per > 0 and w.shape[1] == K and epi in PAIR_EPI and 0 < M <= 64, "gemm_hold shape")
    _req(out.dtype == torch.bfloat16 and out.shape == (M, N) and out.stride(1) == 1, "gemm_hold out")
    per = -(-M // -(-M // per))
    for r0 in range(0, M, per):
        xs, os_ = x[r0:r0 + per], out[r0:r0 + per]
        check(L.ragk_gemm_hold(xs.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), ptr(wscale), os_.data_ptr(),
                               out.stride(0), ptr(par), xs.shape[0], N, K, EPI[epi], _cu_count(), stream_ptr()),
              "ragk_gemm_hold")
    return out


# ----------------------------------------------------------------------------- fp8 GEMM
def use_hold_slabs(M, N, K):
    """fp8 split-K products whose slabs go through gemm_hold.hip (a slab per 2048 of K) instead of gemm_part.hip, which stages
    the activations of a K-slice in every block of 64 columns: 4096 x 14336 at 17 / 33 / 64 rows 19 / 26 / 33 us -> 16 / 19 / 23,
    5120 x 18432 32 / 38 / 49 -> 23 / 26 / 31, 4096 x 8192 at 33 / 64 rows 14.9 / 18.5 -> 13.9 / 18.1. Smaller weights leave a
    block too few rows for the 128 KB of x that it loads first (4096 x 8192 at 17 rows 10.7 against 12.0, 4096 x 4096 at 33 / 64
    7.8 / 9.5 against 9.9 / 13), and up to 16 rows the two are equal."""
    return (16 < M <= 64 and K % 2048 == 0 and K // 2048 <= _cu_count() and N % 16 == 0
            and N * K >= (5 << 23 if M <= 32 else 1 << 25))


def gemm_hold_slabs(x, w8, scale, out=None):
    """fp32 slabs P[K / 2048, M, N] of x @ dequant(w8)^T with the activations of a slab held in registers (gemm_hold.hip)."""
    M, K = x.shape
    N = w8.shape[0]
    _req(0 < M <= 64 and K % 2048 == 0 and N % 16 == 0 and w8.shape[1] == K, "gemm_hold_slabs shape")
    if out is None:
        out = torch.empty((K // 2048, M, N), dtype=torch.float32, device=x.device)
    check(_lib.lib().ragk_gemm_hold_slabs(x.data_ptr(), x.stride(0), w8.data_ptr(), w8.stride(0), scale.data_ptr(),
                                          out.data_ptr(), M, N, K, _cu_count(), stream_ptr()), "ragk_gemm_hold_slabs")
    return out


def use_hold_slabs_silu(M, K):
    """fp8 gate/up projections of more rows than a launch of gemm_hold holds: slabs of 2048 of K and a pass that sums and pairs
    them, 28672 x 4096 at 33 / 64 rows 54 / 61 us (two launches) -> 33 / 38, 7168 x 4096 22 / 26 (gemm_stream) -> 17 / 21, 16384
    x 6144 at 17 / 64 rows 38 / 72 -> 29 / 37. Up to 16 rows the pass takes what the slabs gain (8192 x 6144 18.6 against 18.1)."""
    return 16 < M <= 64 and K % 2048 == 0 and K // 2048 <= _cu_count() and M > _hold_rows(K, True)


def quant_fp8_rows(x, q=None, scale=None):
    """bf16 [M,K] -> (e4m3fn [M,K], fp32 [M]) with one dynamic scale per row."""
    _bf16_2d(x, "x")
    M, K = x.shape
    _req(K % 8 == 0, "K % 8")
    q = torch.empty((M, K), dtype=torch.float8_e4m3fn, device=x.device) if q is None else q
    scale = torch.empty(M, dtype=torch.float32, device=x.device) if scale is None else scale
    _req(q.shape == (M, K) and q.is_contiguous() and scale.numel() == M, "quant buffers")
    check(_lib.lib().ragk_quant_fp8_rows(x.data_ptr(), x.stride(0), q.data_ptr(), q.stride(0), scale.data_ptr(), M, K,
                                         stream_ptr()), "ragk_quant_fp8_rows")
    return q, scale


FP8_DEC_STREAM = True


def gemm_fp8(x, w, bias=None, resid=None, epi="none", out=None, out_f32=False):
    """out[M,N] = epi(x[M,K] @ dequant(w)^T) for an :class:`ops.fp8.Fp8Weight` w (rows = N, or 2N
    packed gate/up for epi='silu_mul'). M <= 64: W8A16 decode kernel; else W8A8 prefill kernel."""
    from .fp8 import DEC_MAX_M

    _bf16_2d(x, "x")
    M, K = x.shape
    w8, sw = w.w8, w.scale
    _req(w8.dtype == torch.float8_e4m3fn and w8.is_cuda and w8.dim() == 2 and w8.shape[1] == K
         and (w8.is_contiguous() or (w8.stride(1) == 1 and w8.stride(0) >= K and w8.stride(0) % 16 == 0)), "fp8 weight")
    if (w8.data_ptr() | w8.stride(0)) & 15:  # (the kernels' LDS-DMA pieces start on 16 bytes)
        w8 = w8.clone(memory_format=torch.contiguous_format)
    _req(sw.dtype == torch.float32 and sw.numel() == w8.shape[0], "fp8 scale")
    _req(K % 128 == 0, "K must be a multiple of 128")
    e = EPI[epi]
    N = w8.shape[0] // 2 if epi == "silu_mul" else w8.shape[0]
    if epi == "silu_mul":
        _req(N % 64 == 0 and not out_f32, "silu_mul needs N % 64 == 0, bf16 out")
    elif M > DEC_MAX_M:
        _req(N % 8 == 0, "N % 8")
    if "bias" in epi:
        _req(bias is not None and bias.dtype == torch.bfloat16 and bias.numel() == N, "bias bf16[N]")
    if "resid" in epi:
        _bf16_2d(resid, "resid")
        _req(resid.shape == (M, N), "resid shape")
    odt = torch.float32 if out_f32 else torch.bfloat16
    out = torch.empty((M, N), dtype=odt, device=x.device) if out is None else out
    _req(out.dtype == odt and out.shape == (M, N) and out.stride(1) == 1, "out shape/dtype")
    if M == 0:
        return out
    ldr = resid.stride(0) if resid is not None else 0
    near = w8.stride(0) < 1 << 24  # a lane's row is a 32-bit offset in gemm_hold
    if epi == "silu_mul" and use_hold_slabs_silu(M, K) and near and _vec_rows(x, w8, out):
        ws = torch.empty(K // 2048 * M * 2 * N, dtype=torch.float32, device=x.device)
        check(_lib.lib().ragk_gemm_hold_slabs_silu(x.data_ptr(), x.stride(0), w8.data_ptr(), w8.stride(0), sw.data_ptr(),
                                                   out.data_ptr(), out.stride(0), M, N, K, _cu_count(), ws.data_ptr(),
                                                   stream_ptr()), "ragk_gemm_hold_slabs_silu")
        return out
    if use_hold(M, N, K, epi, fp8=True) and near and _vec_rows(x, w8):
        return gemm_hold(x, w8, sw, epi=epi, out=out)
    if M <= DEC_MAX_M and FP8_DEC_STREAM and use_stream(M, N, K, epi, fp8=True):
        rc = _gemm_stream(x, w8, sw, out, bias, resid, ldr, M, N, K, epi, e, out_f32)
    elif M <= DEC_MAX_M:
        rc = _lib.lib().ragk_gemm_fp8(x.data_ptr(), x.stride(0), None, 0, None, w8.data_ptr(), w8.stride(0),
                                      sw.data_ptr(), out.data_ptr(), out.stride(0), ptr(bias), ptr(resid), ldr, M, N,
                                      K, e, int(out_f32), stream_ptr())
    else:
        q, sa = quant_fp8_rows(x)
        rc = _lib.lib().ragk_gemm_fp8(None, 0, q.data_ptr(), q.stride(0), sa.data_ptr(), w8.data_ptr(), w8.stride(0),
                                      sw.data_ptr(), out.data_ptr(), out.stride(0), ptr(bias), ptr(resid), ldr, M, N,
                                      K, e, int(out_f32), stream_ptr())
    check(rc, "ragk_gemm_fp8")
    return out


# ----------------------------------------------------------------------------- norms
def rmsnorm(x, w, eps, out=None, resid=None):
    _bf16_2d(x, "x")
    T, H = x.shape
    _req(w.numel() == H and w.dtype == torch.bfloat16, "weight")
    _req(H % 8 == 0 and H <= 8192, "H must be a multiple of 8, <= 8192")
    if resid is not None:
        _bf16_2d(resid, "resid")
        _req(resid.shape == x.shape, "resid shape")
    out = torch.empty_like(x) if out is None else out
    check(_lib.lib().ragk_rmsnorm(x.data_ptr(), x.stride(0), ptr(resid), resid.stride(0) if resid is not None else 0,
                                  w.data_ptr(), out.data_ptr(), out.stride(0), T, H, float(eps), stream_ptr()),
          "ragk_rmsnorm")
    return out


def rmsnorm_rows(x, rows, w, eps):
    """rmsnorm(x[rows]) * w."""
    _bf16_2d(x, "x")
    H = x.shape[1]
    _req(w.numel() == H and w.dtype == torch.bfloat16, "weight")
    _req(H % 8 == 0 and H <= 8192, "H must be a multiple of 8, <= 8192")
    _req(rows.dtype == torch.int32 and rows.is_cuda and rows.is_contiguous(), "rows int32")
    out = torch.empty((rows.numel(), H), dtype=x.dtype, device=x.device)
    check(_lib.lib().ragk_rmsnorm_rows(x.data_ptr(), x.stride(0), rows.data_ptr(), w.data_ptr(), out.data_ptr(), H, rows.numel(), H,
                                       float(eps), stream_ptr()), "ragk_rmsnorm_rows")
    return out


def layernorm(x, g, b, eps, out=None, resid=None):
    _bf16_2d(x, "x")
    T, H = x.shape
    _req(H % 8 == 0 and H <= 8192, "H")
    out = torch.empty_like(x) if out is None else out
    check(_lib.lib().ragk_layernorm(x.data_ptr(), x.stride(0), ptr(resid), resid.stride(0) if resid is not None else 0,
                                    g.data_ptr(), b.data_ptr(), out.data_ptr(), out.stride(0), T, H, float(eps),
                                    stream_ptr()), "ragk_layernorm")
    return out


def embed(ids, table, out=None, carry=None, prev=None):
    """Embedding gather. carry/prev (asynchronous decode): rows with carry[t] >= 0 take their token id
    from prev[carry[t]] (the previous step's sampled tokens on the device) and store it into ids[t]."""
    _req(ids.dtype == torch.int32 and ids.is_cuda and ids.is_contiguous(), "ids int32")
    _req(table.is_contiguous(), "table rows without gaps")
    V, H = table.shape
    out = torch.empty((ids.numel(), H), dtype=table.dtype, device=table.device) if out is None else out
    if carry is None:
        check(_lib.lib().ragk_embed(ids.data_ptr(), table.data_ptr(), out.data_ptr(), ids.numel(), H, V,
                                    stream_ptr()), "ragk_embed")
        return out
    _req(carry.dtype == torch.int32 and prev.dtype == torch.int32 and carry.numel() >= ids.numel(), "carry int32")
    check(_lib.lib().ragk_embed_carry(ids.data_ptr(), carry.data_ptr(), prev.data_ptr(), table.data_ptr(),
                                      out.data_ptr(), ids.numel(), H, V, stream_ptr()), "ragk_embed_carry")
    return out


def embed_rmsnorm(ids, table, w, eps, carry=None, prev=None):
    """(embed(ids, table, carry, prev), its rmsnorm * w) in one launch."""
    _req(ids.dtype == torch.int32 and ids.is_cuda and ids.is_contiguous(), "ids int32")
    V, H = table.shape
    _req(table.dtype == torch.bfloat16 and table.is_contiguous(), "bf16 table rows without gaps")
    _req(w.dtype == torch.bfloat16 and w.numel() == H, "weight")
    _req(H % 8 == 0 and H <= 8192, "H must be a multiple of 8, <= 8192")
    if carry is not None:
        _req(carry.dtype == torch.int32 and prev.dtype == torch.int32 and carry.numel() >= ids.numel(), "carry int32")
    h = torch.empty((ids.numel(), H), dtype=table.dtype, device=table.device)
    xn = torch.empty_like(h)
    check(_lib.lib().ragk_embed_rmsnorm(ids.data_ptr(), ptr(carry), ptr(prev) if carry is not None else None, table.data_ptr(),
                                        h.data_ptr(), w.data_ptr(), xn.data_ptr(), ids.numel(), H, V, float(eps), stream_ptr()),
          "ragk_embed_rmsnorm")
    return h, xn


def embed_ln(ids, pos_ids, word, pos, type_row, g, b, eps, do_ln=True, out=None):
    _req(ids.dtype == torch.int32 and pos_ids.dtype == torch.int32, "int32 ids")
    _req(int(ids.numel()) == int(pos_ids.numel()), "ids/pos_ids")
    H = word.shape[1]
    out = torch.empty((ids.numel(), H), dtype=word.dtype, device=word.device) if out is None else out
    check(_lib.lib().ragk_embed_ln(ids.data_ptr(), pos_ids.data_ptr(), word.data_ptr(), pos.data_ptr(),
                                   ptr(type_row), ptr(g), ptr(b), out.data_ptr(), ids.numel(), H, float(eps),
                                   int(do_ln), stream_ptr()), "ragk_embed_ln")
    return out


def rope_kv(qkv, positions, cos_t, sin_t, slots, k_cache, v_cache, Hq, Hkv, D, apply_rope=True):
    """In-place RoPE on q and k (inside qkv [T, (Hq+2Hkv)*D]) + paged cache write."""
    _bf16_2d(qkv, "qkv")
    T = qkv.shape[0]
    _req(qkv.shape[1] >= (Hq + 2 * Hkv) * D, "qkv width")
    _req(positions.dtype == torch.int32 and positions.numel() == T, "positions")
    if slots is not None:
        _req(slots.dtype == torch.int32 and slots.numel() == T, "slots")
        _req(k_cache.dim() == 4 and k_cache.shape[1] == Hkv and k_cache.shape[3] == D, "cache layout")
    BS = k_cache.shape[2] if k_cache is not None else 64
    check(_lib.lib().ragk_rope_kv(qkv.data_ptr(), qkv.stride(0), positions.data_ptr(), ptr(cos_t), ptr(sin_t),
                                  ptr(slots), ptr(k_cache), ptr(v_cache), T, Hq, Hkv, D, BS, int(apply_rope),
                                  stream_ptr()), "ragk_rope_kv")


def add_partials_rmsnorm(P, h, w, eps, out=None, rounded=True, rows=None):
    """h <- bf16(h + bf16(P.sum(0))) in place; returns rmsnorm(h) * w (split-K decode consumer). rounded=False: the sum is
    added as it is, as a product's residual epilogue does (prompts, whose steps take either). rows: of these rows only, and h
    stays as it is."""
    _bf16_2d(h, "h")
    M, H = h.shape
    _req(P.dtype == torch.float32 and P.is_contiguous() and P.dim() == 3 and P.shape[1:] == (M, H), "partials shape")
    _req(w.is_cuda and w.dtype == torch.bfloat16 and w.numel() == H, "norm weight")
    n = M
    if rows is not None:
        _req(rows.dtype == torch.int32 and rows.is_cuda and rows.is_contiguous(), "rows int32")
        n = rows.numel()
    out = torch.empty((n, H), dtype=h.dtype, device=h.device) if out is None else out
    _req(out.shape == (n, H) and out.stride(1) == 1, "out")
    if n == 0:
        return out
    check(_lib.lib().ragk_add_partials_rmsnorm(P.data_ptr(), P.shape[0], M, h.data_ptr(), h.stride(0), w.data_ptr(),
                                               out.data_ptr(), out.stride(0), H, float(eps), int(rounded), ptr(rows), n,
                                               stream_ptr()), "ragk_add_partials_rmsnorm")
    return out


def rope_kv_partials(P, q_out, positions, cos_t, sin_t, slots, k_cache, v_cache, Hq, Hkv, D):
    """qkv = bf16(P.sum(0)); RoPE'd q -> q_out[:, :Hq*D]; RoPE'd k and v -> paged cache."""
    _req(P.dtype == torch.float32 and P.is_contiguous() and P.dim() == 3, "partials")
    S, T, ldp = P.shape
    _req(ldp >= (Hq + 2 * Hkv) * D, "qkv width")
    _bf16_2d(q_out, "q_out")
    _req(q_out.shape[0] == T and q_out.shape[1] >= Hq * D, "q_out shape")
    _req(positions.dtype == torch.int32 and positions.numel() == T, "positions")
    _req(slots is not None and slots.dtype == torch.int32 and slots.numel() == T, "slots")
    _req(k_cache.dim() == 4 and k_cache.shape[1] == Hkv and k_cache.shape[3] == D, "cache layout")
    check(_lib.lib().ragk_rope_kv_partials(P.data_ptr(), S, T, ldp, q_out.data_ptr(), q_out.stride(0),
                                           positions.data_ptr(), ptr(cos_t), ptr(sin_t), slots.data_ptr(),
                                           k_cache.data_ptr(), v_cache.data_ptr(), Hq, Hkv, D, k_cache.shape[2],
                                           stream_ptr()), "ragk_rope_kv_partials")


def pool_l2norm(hidden, cu, mode="cls", normalize=True, out=None):
    _bf16_2d(hidden, "hidden")
    B = cu.numel() - 1
    H = hidden.shape[1]
    _req(H <= 2048, "H <= 2048")
    m = {"cls": 0, "mean": 1, "last": 2}[mode]
    out = torch.empty((B, H), dtype=torch.float32, device=hidden.device) if out is None else out
    check(_lib.lib().ragk_pool_l2norm(hidden.data_ptr(), hidden.stride(0), cu.data_ptr(), out.data_ptr(), B, H, m,
                                      int(normalize), stream_ptr()), "ragk_pool_l2norm")
    return out


ENCODER_LAYER = ("wqkv", "bqkv", "wo", "bo", "ln1_g", "ln1_b", "wi", "bi", "wo2", "bo2", "ln2_g", "ln2_b")


def encoder_pointers(cfg, w, l0=0, l1=None):
    """Addresses of what encoder_forward reads of an encoder's weights, [word, pos, ln_g, ln_b, type row (or None), then
    ENCODER_LAYER of every layer], or None if one of them would be read wrongly by its address (then: layer by layer through
    the checked entry points). Of layers l0 to l1, the first five with layer 0. For the call at hand only, a property at a time over
    all tensors: 77 of them take 35 us."""
    H, I, T = cfg.hidden_size, cfg.intermediate_size, torch.Tensor
    if H % 128 or I % 128 or H > 2048 or max(3 * H, I) >= STREAM_MIN_ROWS or H // cfg.num_attention_heads not in (32, 64, 128):
        return None
    ts = list(itertools.chain.from_iterable(map(operator.itemgetter(*ENCODER_LAYER), w.layers[l0:l1])))
    shapes = [(3 * H, H), (3 * H,), (H, H), (H,), (H,), (H,), (I, H), (I,), (H, I), (H,), (H,), (H,)] * (len(ts) // len(ENCODER_LAYER))
    row = None
    if l0 == 0:
        row = w.type_row
        row = row.view(-1) if row is not None and row.is_contiguous() else row
        first = [w.word, w.pos, w.ln_g, w.ln_b] + ([row] if row is not None else [])
        shapes = [(w.word.shape[0], H), (w.pos.shape[0], H)] + [(H,)] * (len(first) - 2) + shapes
        ts = first + ts
    if (all(map(T.is_contiguous, ts)) and list(map(T.size, ts)) == shapes and [t.dtype for t in ts].count(torch.bfloat16) == len(ts)
            and list(map(T.get_device, ts)).count(w.word.get_device()) == len(ts)):
        at = list(map(T.data_ptr, ts))
        if not any(map((15).__and__, at)):  # the kernels' vectors and LDS-DMA pieces
            return at if row is not None or l0 else at[:4] + [None] + at[4:]
    return None


def encoder_forward_ok(cfg, w):
    """Whether encoder_forward takes these weights."""
    return encoder_pointers(cfg, w) is not None


@functools.lru_cache(maxsize=4096)
def _encoder_plans(T, H, I, cus, split, w4_min_m):
    """(launches of the four products of a layer of T rows, floats of the largest one's slabs)."""
    plans, slab = (_lib.GemmPlan * 4)(), 0
    for i, (N, K) in enumerate(((3 * H, H), (H, H), (I, H), (H, I))):
        S, mi = ln_slabs(T, N, K) if i in (1, 3) else (1, 0)
        plan = ((0, T, mi, S),) if S > 1 else ((0, T, -1, 1),) if T <= 64 else gemm_plan(T, N, K, True, cus)
        plans[i].n, plans[i].slabs = len(plan), int(S > 1)
        for j, (r0, r1, mi, S) in enumerate(plan):
            plans[i].p[j] = _lib.GemmPiece(r0, r1, mi, S)
            slab = max(slab, S * (r1 - r0) * N if S > 1 else 0)
    return plans, slab


FEW_ROWS, FEW_COLS = 32, 1024  # csrc/kernels/encoder.h FEW_T, FEW_H
FEW_SIZE = 16384  # rows x columns: the blocks repeat the rows' work
# ints that travel as kernel arguments, 960 a launch of 2 us: copied to the device (a wait for the stream, 15 us when it is idle)
# only where a forward takes milliseconds. Copied / as arguments, us a call of six layers of 384 columns among others: two texts of
# 20 tokens 227 / 220, eight of 14 278 / 246, four of 400 351 / 319; 24 layers of 1024: 919 / 888, 1343 / 1324, 2369 / 2342
PUT_INTS = 3840


def _req_no_capture():
    """Integers of host memory that travel as kernel arguments would be frozen into a graph, which repeats them whatever the
    caller's memory holds by then; a copy of that memory refuses a capture by itself."""
    if torch.cuda.is_current_stream_capturing():
        raise RuntimeError("an encoder forward of ids in host memory cannot be captured")


def encoder_few_ok(cfg, T, B):
    """Whether a batch takes the four launches a layer of csrc/kernels/encoder_few.hip. Us a call against seven launches: six
    layers of 384 columns 103 / 197 at 5 rows, 111 / 202 at 14, 147 / 205 at 32; 24 layers of 1024 600 / 711 at 5 rows, 705 / 761
    at 16, 777 / 790 at 17, but 855 / 820 at 24 and 958 / 839 at 32."""
    H = cfg.hidden_size
    return (B == 1 and 1 <= T <= FEW_ROWS and H <= FEW_COLS and T * H <= FEW_SIZE and cfg.num_hidden_layers > 0
            and H // cfg.num_attention_heads in (32, 64))


def _encoder_call(cfg, weights, bufs, at, T, B):
    """(call, what has to outlive it): addresses of `bufs` ((field, bytes) pairs) within one allocation that begins at `at`."""
    import ctypes

    c = _lib.EncoderCall()
    for name, size in bufs:
        setattr(c, name, at)
        at += -(-size // 256) * 256
    c.word, c.pos_table, c.ln_g, c.ln_b, c.type_row, *table = weights
    ptrs = (ctypes.c_void_p * len(table))(*table)
    c.layers, c.n_layers = ctypes.addressof(ptrs), len(table) // len(ENCODER_LAYER)
    c.T, c.B, c.H, c.I, c.heads = T, B, cfg.hidden_size, cfg.intermediate_size, cfg.num_attention_heads
    c.pooling, c.normalize, c.eps = {"cls": 0, "mean": 1, "last": 2}[cfg.pooling], int(cfg.normalize), float(cfg.layer_norm_eps)
    return c, ptrs


# Layers whose weights are checked and whose launches are made at a time: the device begins behind the first three's, not behind all
# (4 us of checks a layer, 15 to 27 of launches and kernels). A call of one text, waited for, us: 24 layers of 1024, 5 / 16 tokens
# 748 / 836 -> 645 / 734; 6 of 384, 14 / 30 tokens 164 / 203 -> 164 / 184. Calls behind each other 119 / 560 on both sides. The last
# call alone gives up the interpreter lock, as the one call for all layers did.
FEW_LAYERS = 3


def encoder_few(cfg, w, ids, first_pos, out):
    """Embedding of one sequence (encoder_few_ok) into the fp32 row `out`; ids: contiguous int32, on the host (they travel as a
    kernel argument: nothing is uploaded) or on the device. False, with the row untouched, if encoder_pointers refuses a weight."""
    import ctypes

    H, T, n = cfg.hidden_size, len(ids), len(w.layers)
    weights = encoder_pointers(cfg, w, 0, FEW_LAYERS)
    if weights is None:
        return False
    _req(out.dtype == torch.float32 and out.is_cuda and out.is_contiguous() and out.numel() == H, "out fp32 row")
    bufs = [("h", 2 * T * H), ("qkv", 6 * T * H), ("f", 2 * T * cfg.intermediate_size), ("y", 4 * T * H)]
    buf = torch.empty(sum(-(-n // 256) * 256 for _, n in bufs), dtype=torch.uint8, device=out.device)
    size = len(ENCODER_LAYER)
    c, table = _encoder_call(cfg, weights + [None] * (size * n + 5 - len(weights)), bufs, buf.data_ptr(), T, 1)
    c.few, c.first_pos, c.out, c.ldo = 1, first_pos, out.data_ptr(), H
    if isinstance(ids, torch.Tensor):
        _req(ids.is_cuda and ids.dtype == torch.int32 and ids.is_contiguous(), "ids int32")
        c.ids = ids.data_ptr()
    else:
        _req(ids.dtype == "int32" and ids.flags.c_contiguous, "ids int32")
        _req_no_capture()
        c.ids_host = ids.ctypes.data
    c.l1 = min(n, FEW_LAYERS)
    while True:
        forward = _lib.lib().ragk_encoder_forward if c.l1 == n else _lib.held("ragk_encoder_forward")
        check(forward(ctypes.byref(c), stream_ptr()), "ragk_encoder_forward")
        if c.l1 == n:
            return True
        c.l0, c.l1 = c.l1, min(n, c.l1 + FEW_LAYERS)
        weights = encoder_pointers(cfg, w, c.l0, c.l1)
        if weights is None:  # (the last launch writes the row)
            return False
        table[size * c.l0:size * c.l1] = weights


def encoder_forward(cfg, w, ids, lens, first_pos, out, rows):
    """Embeddings of packed sequences (host int32 ids, int64 lens) into rows `rows` of out (fp32 on the device): one upload
    of the step's integers, one workspace, one native call for all launches (csrc/kernels/encoder.hip). False, with nothing written, if
    encoder_pointers refuses a weight."""
    import ctypes

    import numpy as np

    H, I, nh, B, T = cfg.hidden_size, cfg.intermediate_size, cfg.num_attention_heads, len(lens), int(len(ids))
    few = encoder_few_ok(cfg, T, B)
    weights = None if few else encoder_pointers(cfg, w)
    if weights is None and not few:
        return False
    _req(out.dtype == torch.float32 and out.is_cuda and out.stride(1) == 1 and out.shape[1] == H, "out fp32 rows")
    if few:
        row = int(rows[0])
        _req(T == int(lens[0]) and len(rows) == 1 and 0 <= row < out.shape[0], "lens, rows")
        return encoder_few(cfg, w, np.ascontiguousarray(ids), first_pos, out[row])
    _req(T == int(lens.sum()) and len(rows) == B and 0 <= int(rows.min()) and int(rows.max()) < out.shape[0], "lens, rows")
    _req(T * max(3 * H, I) * 2 < 2 ** 31, "packed rows past 2 GiB")
    dev = out.device
    cu = np.zeros(B + 1, dtype=np.int32)
    np.cumsum(lens, out=cu[1:])
    pos = np.arange(first_pos, first_pos + T, dtype=np.int32) - np.repeat(cu[:-1], lens)
    tiles = build_encoder_tiles(lens, nh).numpy().reshape(-1)
    parts = [ids, pos, cu, lens, rows, tiles]
    at = list(itertools.accumulate(map(len, parts), initial=0))
    host = np.concatenate(parts).astype(np.int32, copy=False)
    L = _lib.lib()
    if len(host) <= PUT_INTS:
        _req_no_capture()
        ints = torch.empty(len(host), dtype=torch.int32, device=dev)
        check(L.ragk_put_ints(host.ctypes.data, len(host), ints.data_ptr(), stream_ptr()), "ragk_put_ints")
    else:
        ints = torch.from_numpy(host).to(dev)
    plans, slab = _encoder_plans(T, H, I, _cu_count(), PREFILL_SPLITK, PREFILL_SPLITK_MIN_M)
    bufs = [("h", 2 * T * H), ("a", 2 * T * H), ("attn", 2 * T * H), ("qkv", 6 * T * H), ("f", 2 * T * I), ("ws", 4 * slab)]
    buf = torch.empty(sum(-(-n // 256) * 256 for _, n in bufs), dtype=torch.uint8, device=dev)
    c, keep = _encoder_call(cfg, weights, bufs, buf.data_ptr(), T, B)
    c.plans = plans
    q = ints.data_ptr()
    c.ids, c.pos, c.cu, c.lens, c.rows, c.tiles = (q + 4 * o for o in at[:-1])
    c.out, c.ldo, c.n_tiles = out.data_ptr(), out.stride(0), len(tiles) // 2
    check(L.ragk_encoder_forward(ctypes.byref(c), stream_ptr()), "ragk_encoder_forward")
    return True


def layernorm_slabs(P, bias, resid, g, b, eps, out=None):
    """LN(P.sum(0) + bias + resid) * g + b of a product's fp32 split-K slabs P [S, T, H]."""
    S, T, H = P.shape
    _req(P.dtype == torch.float32 and P.is_cuda and P.is_contiguous(), "slabs fp32")
    _req(H % 8 == 0 and H <= 8192 and resid.shape == (T, H) and bias.numel() == H, "H")
    _bf16_2d(resid, "resid")
    out = torch.empty((T, H), dtype=torch.bfloat16, device=P.device) if out is None else out
    check(_lib.lib().ragk_layernorm_slabs(P.data_ptr(), S, bias.data_ptr(), resid.data_ptr(), resid.stride(0), g.data_ptr(),
                                          b.data_ptr(), out.data_ptr(), out.stride(0), T, H, float(eps), stream_ptr()),
          "ragk_layernorm_slabs")
    return out


def ln_slabs(M, N, K):
    """(slabs, tile) of a product whose bias, residual and LayerNorm follow as one launch over its split-K slabs (tile -1:
    gemm_part, else gemm_mid's), (1, 0): the product with its epilogue and a plain LayerNorm. Pairs of launches, us: 1024 x
    4096 at 30 / 64 rows 15.6 / 23.3 -> 9.5 / 10.8, 384 x 1536 at 16 / 64 7.0 / 11.5 -> 6.5 / 7.6, 1024 x 1024 at 64 9.9 -> 8.3;
    past 64 rows, where the split ended in a reduction or did not pay for one, 384 x 1536 at 100 rows 11.9 -> 10.2, 1024 x
    1024 at 200 13.5 -> 11.6, 1024 x 4096 at 400 19.0 -> 17.1. Under 18432 = 12 x 1536 inputs, or a K that gives fewer than
    four slabs of four K-steps, the register-streaming kernel's epilogue is ahead (1024 x 1024 at 12 rows 6.6 against 7.1)."""
    if K % 64 or N % 8:
        return 1, 0
    if M <= 64:
        ks = 4 if K <= 3072 else 8  # K-steps of a slab: at most twelve slabs of the shorter ones
        return (K // (64 * ks), -1) if K >= 1024 and K % (64 * ks) == 0 and M * K >= 18432 else (1, 0)
    if not PREFILL_SPLITK:
        return 1, 0
    S, mi = _slab_best(M, N, K, _cu_count(), PREFILL_SPLITK_MIN_M)
    return (S, mi) if S > 1 and mi else (1, 0)


def gemm_layernorm(x, w, bias, resid, g, b, eps):
    """LN(x @ w^T + bias + resid) * g + b, the sum kept in fp32 where the product is split (ln_slabs)."""
    M, N, K = _gemm_operands(x, w, bias, resid, "bias_resid")
    S, mi = ln_slabs(M, N, K)
    if S == 1:
        return layernorm(gemm(x, w, bias=bias, resid=resid, epi="bias_resid"), g, b, eps)
    x, w = _tile_rows(x, w)
    if mi < 0:
        return layernorm_slabs(gemm_part(x, w, out=torch.empty((S, M, N), dtype=torch.float32, device=x.device), ks=K // 64 // S),
                               bias, resid, g, b, eps)
    P = torch.empty((S, M, N), dtype=torch.float32, device=x.device)
    check(_lib.lib().ragk_gemm_mid(x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), P.data_ptr(), N, None, None, 0, M, N, K,
                                   EPI["none"], 2, mi, S, None, stream_ptr()), "ragk_gemm_mid")
    return layernorm_slabs(P, bias, resid, g, b, eps)


def silu_mul(x, out=None):
    _bf16_2d(x, "x")
    T, I2 = x.shape
    I = I2 // 2
    out = torch.empty((T, I), dtype=x.dtype, device=x.device) if out is None else out
    check(_lib.lib().ragk_silu_mul(x.data_ptr(), x.stride(0), out.data_ptr(), out.stride(0), T, I, stream_ptr()),
          "ragk_silu_mul")
    return out


def gather_rows(x, idx, out=None):
    _bf16_2d(x, "x")
    _req(idx.dtype == torch.int32 and idx.is_cuda, "idx int32")
    n = idx.numel()
    out = torch.empty((n, x.shape[1]), dtype=x.dtype, device=x.device) if out is None else out
    check(_lib.lib().ragk_gather_rows(x.data_ptr(), x.stride(0), idx.data_ptr(), out.data_ptr(), out.stride(0), n,
                                      x.shape[1], stream_ptr()), "ragk_gather_rows")
    return out


# ----------------------------------------------------------------------------- attention
def prefill_qtile(Hq, Hkv):
    """Query rows per prefill-attention block (the tile list must be built with the kernel's value):
    64 when 4 query heads share a KV head (the 8-wave kernels, two 32-row groups per K/V tile), else
    128 / heads-per-block (attention.hip ragk_attn_prefill_qtile)."""
    G = Hq // Hkv
    GB = 4 if G % 4 == 0 else (2 if G % 2 == 0 else 1)
    return 32 * ((8 if GB == 4 else 4) // GB)


def build_prefill_tiles(q_lens, Hq, Hkv):
    """(seq, q_start) work list, heaviest (latest query positions) first."""
    import numpy as np

    qt = prefill_qtile(Hq, Hkv)
    ql = np.asarray(q_lens, dtype=np.int64)
    top = (int(ql.max()) - 1) // qt if len(ql) else -1
    if len(ql) * (top + 1) <= 64:  # one query's: 10 us as a list, 21 through the arrays below
        lens = ql.tolist()
        tiles = [(s, q0) for q0 in range(top * qt, -1, -qt) for s, n in enumerate(lens) if n > q0]
        return torch.tensor(tiles, dtype=torch.int32).reshape(-1, 2)
    nt = (ql + qt - 1) // qt
    seq = np.repeat(np.arange(len(ql)), nt)
    first = np.repeat(np.cumsum(nt) - nt, nt)
    q0 = (np.arange(int(nt.sum())) - first) * qt
    order = np.argsort(-q0, kind="stable")
    return torch.from_numpy(np.stack([seq[order], q0[order]], 1).astype(np.int32)).reshape(-1, 2)


def build_encoder_tiles(lens, heads):
    """(seq, q_start) work list of bidirectional attention: every block of a sequence reads all of its keys, so its tiles stay
    together (they share K / V in the L2 of each head's XCD: 64 sequences of 1344 rows 939 us as build_prefill_tiles orders them,
    671 so, 12 sequences of 13764 rows 100 and 97), longest sequences first."""
    import numpy as np

    qt = prefill_qtile(heads, heads)
    if len(lens) <= 8:  # a query's: host time
        ls = [int(n) for n in lens]
        tiles = [(s, q0) for s in sorted(range(len(ls)), key=lambda s: -ls[s]) for q0 in range(0, ls[s], qt)]
        return torch.tensor(tiles, dtype=torch.int32).reshape(-1, 2)
    ql = np.asarray(lens, dtype=np.int64)
    order = np.argsort(-ql, kind="stable")
    nt = (ql[order] + qt - 1) // qt
    q0 = (np.arange(int(nt.sum())) - np.repeat(np.cumsum(nt) - nt, nt)) * qt
    return torch.from_numpy(np.stack([np.repeat(order, nt), q0], 1).astype(np.int32))


def attn_prefill(q, k, v, cu_q, kv_lens, tiles, out, Hq, Hkv, D, causal=True, paged=True, block_tables=None,
                 cu_kv=None, kv_stride=0, scale=None):
    """q: [T, >=Hq*D] bf16 (row stride arbitrary). paged: k/v caches [nb, Hkv, 64, D];
    else packed k/v row pointers with `kv_stride` (element stride per token)."""
    _req(q.dtype == torch.bfloat16 and q.stride(-1) == 1, "q")
    _req(tiles.dtype == torch.int32 and tiles.is_cuda and tiles.is_contiguous(), "tiles int32 on GPU")
    _req(D in (32, 64, 128), "head_dim must be 32/64/128")
    if paged:
        _req(k.dim() == 4 and k.shape[2] == 64 and k.shape[1] == Hkv and k.shape[3] == D, "paged cache [nb,Hkv,64,D]")
        _req(block_tables is not None and block_tables.dtype == torch.int32, "block_tables int32")
        _req(block_tables.stride(0) <= 2048, "prefill block tables wider than 2048 blocks (128k tokens)")
    scale = 1.0 / math.sqrt(D) if scale is None else scale
    n_tiles = tiles.shape[0]
    if paged:
        _req(v.shape == k.shape, "paged k/v caches differ in shape")
        kv_stride = k.shape[0]  # paged: the cache block count (sizes the kernel's buffer descriptors)
    check(_lib.lib().ragk_attn_prefill(
        q.data_ptr(), q.stride(0), k.data_ptr(), v.data_ptr(), kv_stride, ptr(block_tables),
        block_tables.stride(0) if block_tables is not None else 0, cu_q.data_ptr(), ptr(cu_kv), kv_lens.data_ptr(),
        tiles.data_ptr(), n_tiles, out.data_ptr(), out.stride(0), Hq, Hkv, D, int(causal), int(paged), float(scale),
        stream_ptr()), "ragk_attn_prefill")
    return out


DECODE_TARGET_BLOCKS = 512
DECODE_MIN_TILES = 4


def decode_partitions(max_kv_len, batch, Hkv, target_blocks=None, min_tiles=None):
    """(part_tiles, max_parts) for split-K decode: grid = max_parts x Hkv x batch <= target_blocks, two blocks a CU. More than fit
    at once run as a round of their own behind the first (20 rows of 5000 tokens, 8 KV heads: 59.4 us in 480 blocks, 63.4 in 640),
    and fewer, larger ones beat a third of a CU's slots (16 rows of 6000, 4 KV heads: 33.7 in 512, 34.7 in 768). The shaped
    kernel's blocks follow a rule of their own (seq_native.decode_parts).

    Once batch x KV heads would fill the CUs by itself, one partition per pair (attention.hip KL) where its rounds of one block a
    CU are at least four fifths full, else three, or as many as the longest context has keys for: 264 pairs of 1600 tokens 52.4 ->
    45.2 us, 320 of 560 28.0 -> 23.7, 384 of 2400 87.5 -> 86.0, 400 of 1250 52.6 -> 51.1; 512 full ones of 3200 tokens 134 in one,
    146 in three (eight query heads a KV head, which have no KL: 264 of 60 / 300 / 1000 / 4000 tokens 10.3 / 19.4 / 36.1 / 125 ->
    12.2 / 18.9 / 29.5 / 87; the shortest pay for the join's launch). A context without keys for the third leaves those blocks, two
    thirds of the workspace and the join to nothing.
    Where all three are at work in more than two and a quarter rounds, short contexts fill fewer, larger ones: three tiles at least,
    not two (384 pairs of 150 / 300 / 600 tokens 17.0 / 21.5 / 26.3 us -> 13.0 / 18.2 / 26.3, 408 of 200 / 300 20.1 / 22.7 -> 16.8
    / 21.1; below, 264 of 200 / 600 14.7 / 19.8 against 16.2 / 21.6).

    The kernel spreads each sequence's actual KV tiles evenly over the max_parts partitions (at least ``part_tiles`` tiles each,
    attention.hip:decode_part_units), so the grid can be sized once for the longest allowed context (hipGraph capture) without
    idle partitions. part_tiles is half of min_tiles, which caps max_parts: one unit a wave (one row of 500 tokens, 8 KV heads 8.4
    -> 7.4 us, 2 of 2000 with 4 8.7 -> 8.4, 3 of 4000 with 8 14.7 -> 14.4; 5 of 1000, 320 blocks instead of 160, 9.6 -> 10.3),
    while a join of more than 32 partitions costs what they save (one of 5267: 10.2 in 28, 13.3 in 42)."""
    target_blocks = DECODE_TARGET_BLOCKS if target_blocks is None else target_blocks
    min_tiles = DECODE_MIN_TILES if min_tiles is None else min_tiles
    part_tiles = max(1, min_tiles // 2)
    max_kt = max(1, (max_kv_len + 63) // 64)
    pairs = batch * Hkv
    if DECODE_NW8_MIN_PAIRS > 0 and pairs >= DECODE_NW8_MIN_PAIRS:
        rounds = -(-pairs // DECODE_NW8_MIN_PAIRS)
        if 5 * pairs >= 4 * rounds * DECODE_NW8_MIN_PAIRS:
            return part_tiles, 1
        if 4 * 3 * pairs >= 9 * target_blocks:
            part_tiles = max(1, 3 * min_tiles // 4)
        return part_tiles, min(3, -(-max_kt // min_tiles))
    return part_tiles, max(1, min(target_blocks // pairs, -(-max_kt // min_tiles)))


# From this many (sequence, KV head) pairs on, a block a CU, decode_partitions weighs one partition a pair, without a merge
# launch, against three (0 = off). One, with 128 columns and four query heads a KV head, runs as below, in 8-wave blocks without
# DECODE_KL; batch 32: decode step 6.96 -> 6.86-6.90 ms (profiles/decode_nw8_ab_r4.log).
DECODE_NW8_MIN_PAIRS = 256


# Non-temporal K / V loads in the split-K decode attention once batch x KV heads reaches this: at batch 32
# over 5.2k-token contexts (TP=1, 8 KV heads) the KV stream (681 MB per layer) is read once per step, and
# the nt policy keeps it from evicting the L2 / Infinity Cache lines the other kernels reuse: decode step
# 7.60 -> 7.33 ms (profiles/decode_nt_ab_r4.log); batch 1 / 4 neutral-to-worse, and the TP=8 shard's
# 1-KV-head stream at batch 32 (85 MB per layer) 2.33 -> 2.40 ms with nt (profiles/tp_nt_ab_r4.log).
DECODE_NT_MIN_BH = 64


# The single-partition grid (DECODE_NW8_MIN_PAIRS) on 4-wave blocks whose K tiles arrive by LDS-DMA in 1 KiB
# pieces like the V tiles (attention.hip KL), instead of 8-wave blocks loading K as 64-B row pieces into
# registers: batch-32 decode attention over 5.2k-token contexts 114.2-116.8 -> 109.5-110.1 us per layer
# (5.9-6.0 -> 6.3 TB/s of KV; with +-150-token context jitter 116-118 -> 110-111 us),
# tools/attn_decode_probe.py, profiles/attn_decode_probe_r6.log.
DECODE_KL = os.environ.get("RAGK_DECODE_KL", "1") != "0"


def _set_decode_nt(B, Hkv):
    L = _lib.lib()
    check(L.ragk_attn_decode_set_nt(1 if B * Hkv >= DECODE_NT_MIN_BH else 0), "ragk_attn_decode_set_nt")
    check(L.ragk_attn_decode_set_nw8(DECODE_NW8_MIN_PAIRS), "ragk_attn_decode_set_nw8")
    check(L.ragk_attn_decode_set_kl(1 if DECODE_KL else 0), "ragk_attn_decode_set_kl")


def attn_decode(q, k_cache, v_cache, block_tables, kv_lens, out, Hq, Hkv, D, part_tiles, max_parts, ws_o=None,
                ws_ml=None, scale=None):
    B = kv_lens.numel()
    _req(k_cache.dim() == 4 and k_cache.shape[2] == 64 and k_cache.shape[3] == D, "paged cache")
    _req(block_tables.dtype == torch.int32 and block_tables.shape[0] >= B, "block_tables")
    _req(kv_lens.dtype == torch.int32, "kv_lens int32")
    G = Hq // Hkv
    _req(G <= 16, "G <= 16")
    if max_parts > 1:
        if ws_o is None:
            ws_o = torch.empty((B, Hq, max_parts, D), dtype=torch.float32, device=q.device)
            ws_ml = torch.empty((B, Hq, max_parts, 2), dtype=torch.float32, device=q.device)
        _req(ws_o.numel() >= B * Hq * max_parts * D and ws_ml.numel() >= B * Hq * max_parts * 2, "workspace")
    scale = 1.0 / math.sqrt(D) if scale is None else scale
    _set_decode_nt(B, Hkv)
    check(_lib.lib().ragk_attn_decode(
        q.data_ptr(), q.stride(0), k_cache.data_ptr(), v_cache.data_ptr(), block_tables.data_ptr(),
        block_tables.stride(0), block_tables.shape[1], kv_lens.data_ptr(), ptr(ws_o), ptr(ws_ml), out.data_ptr(), out.stride(0),
        B, Hq, Hkv, D, part_tiles, max_parts, float(scale), stream_ptr()), "ragk_attn_decode")
    return out


def attn_decode_rope(P, positions, cos_t, sin_t, slots, k_cache, v_cache, block_tables, kv_lens, out, Hq, Hkv, D,
                     part_tiles, max_parts, ws_o=None, ws_ml=None, scale=None, defer_merge=False):
    """Decode attention straight from the qkv projection's split-K partial slabs P [S, B, ldp] (fp32):
    q / k RoPE, the KV append at `slots` and the attention in one launch -- the same result as
    rope_kv_partials followed by attn_decode (bit-identical), one kernel fewer per layer."""
    _req(P.dtype == torch.float32 and P.is_contiguous() and P.dim() == 3, "partials")
    S, B, ldp = P.shape
    _req(ldp >= (Hq + 2 * Hkv) * D and D % 64 == 0, "qkv width")
    _req(kv_lens.numel() == B, "one partial row per sequence")
    _req(positions.dtype == torch.int32 and positions.numel() == B, "positions")
    _req(slots is not None and slots.dtype == torch.int32 and slots.numel() == B, "slots")
    _req(k_cache.dim() == 4 and k_cache.shape[1] == Hkv and k_cache.shape[2] == 64 and k_cache.shape[3] == D,
         "paged cache")
    _req(block_tables.dtype == torch.int32 and block_tables.shape[0] >= B, "block_tables")
    _req(kv_lens.dtype == torch.int32, "kv_lens int32")
    _req(Hq // Hkv <= 16, "G <= 16")
    if max_parts > 1:
        if ws_o is None:
            ws_o = torch.empty((B, Hq, max_parts, D), dtype=torch.float32, device=P.device)
            ws_ml = torch.empty((B, Hq, max_parts, 2), dtype=torch.float32, device=P.device)
        _req(ws_o.numel() >= B * Hq * max_parts * D and ws_ml.numel() >= B * Hq * max_parts * 2, "workspace")
    scale = 1.0 / math.sqrt(D) if scale is None else scale
    if defer_merge:  # the partitions stay unmerged for gemm_part_merge (no reduce launch)
        _req(max_parts > 1 and ws_o is not None, "deferred merge needs a partition workspace")
    lib = _lib.lib()
    _set_decode_nt(B, Hkv)
    if defer_merge:
        lib.ragk_attn_decode_set_defer(1)
    try:
        check(lib.ragk_attn_decode_rope(
            P.data_ptr(), S, ldp, positions.data_ptr(), slots.data_ptr(), cos_t.data_ptr(), sin_t.data_ptr(),
            k_cache.data_ptr(), v_cache.data_ptr(), block_tables.data_ptr(), block_tables.stride(0),
            block_tables.shape[1], kv_lens.data_ptr(), ptr(ws_o), ptr(ws_ml), out.data_ptr(), out.stride(0), B, Hq, Hkv, D, part_tiles,
            max_parts, float(scale), stream_ptr()), "ragk_attn_decode_rope")
    finally:
        if defer_merge:
            lib.ragk_attn_decode_set_defer(0)
    return out


# ----------------------------------------------------------------------------- sampling
TOPK_CHUNK = 16384  # vocab entries per top-k workgroup (128k vocab -> 7 workgroups per row)


def topk_chunks(V, K, max_cand=512):
    """Workgroups per row for the candidate top-k: enough to fill the chip at decode batch
    sizes, few enough that chunks*K candidates (x TP ranks) stay cheap to merge."""
    return max(1, min(V // TOPK_CHUNK, max_cand // K, 64))


def topk_candidates(logits, K, vocab_offset=0, max_cand=512, chunks=None, cand_v=None, cand_i=None):
    """Per-row top-K of a (vocab-shard of) fp32 logits -> (values, global ids) [B, chunks*K]:
    `chunks` sorted-descending lists of K, one per vocab chunk; the sampler merges them."""
    _req(logits.dtype == torch.float32 and logits.is_cuda and logits.stride(1) == 1, "logits fp32")
    B, V = logits.shape
    _req(1 <= K <= 256, "1 <= K <= 256")
    chunks = topk_chunks(V, K, max_cand) if chunks is None else int(chunks)
    _req(1 <= chunks <= 64, "1 <= chunks <= 64")
    if cand_v is None:
        cand_v = torch.empty((B, chunks * K), dtype=torch.float32, device=logits.device)
        cand_i = torch.empty((B, chunks * K), dtype=torch.int32, device=logits.device)
    _req(cand_v.shape == (B, chunks * K) and cand_i.shape == (B, chunks * K), "candidate buffers [B, chunks*K]")
    check(_lib.lib().ragk_topk_candidates(logits.data_ptr(), logits.stride(0), B, V, K, vocab_offset, chunks,
                                          cand_v.data_ptr(), cand_i.data_ptr(), stream_ptr()), "ragk_topk_candidates")
    return cand_v, cand_i


# candidate lists rank-merged in the sampler (no full sort) when rows ask for top_k <= 64
SAMPLE_LIST_MERGE = True


def sample_candidates(cand_v, cand_i, temps, top_ks, top_ps, seeds, steps, out_tok=None, out_lp=None, list_len=None):
    """list_len: the candidates are n / list_len sorted lists of list_len (topk_candidates output);
    lets rows with top_k <= 64 merge the lists by rank instead of sorting every candidate."""
    B, n = cand_v.shape
    _req(n <= 2048, "<= 2048 candidates")
    _req(temps.dtype == torch.float32 and top_ks.dtype == torch.int32 and top_ps.dtype == torch.float32, "param dtypes")
    _req(seeds.dtype == torch.int64 and steps.dtype == torch.int32, "seeds int64 / steps int32")
    out_tok = torch.empty(B, dtype=torch.int32, device=cand_v.device) if out_tok is None else out_tok
    if list_len and SAMPLE_LIST_MERGE:
        _req(n % list_len == 0, "candidate lists")
        check(_lib.lib().ragk_sample_candidates_lists(cand_v.data_ptr(), cand_i.data_ptr(), B, n, int(list_len),
                                                      temps.data_ptr(), top_ks.data_ptr(), top_ps.data_ptr(),
                                                      seeds.data_ptr(), steps.data_ptr(), out_tok.data_ptr(),
                                                      ptr(out_lp), stream_ptr()), "ragk_sample_candidates_lists")
        return out_tok
    check(_lib.lib().ragk_sample_candidates(cand_v.data_ptr(), cand_i.data_ptr(), B, n, temps.data_ptr(),
                                            top_ks.data_ptr(), top_ps.data_ptr(), seeds.data_ptr(), steps.data_ptr(),
                                            out_tok.data_ptr(), ptr(out_lp), stream_ptr()), "ragk_sample_candidates")
    return out_tok


# ----------------------------------------------------------------------------- search
def l2_search_set_mfma_min_nq(n):
    """Batches of at least n queries (k <= 8, d % 32 == 0) take the MFMA ||x||^2+||q||^2-2x.q path."""
    check(_lib.lib().ragk_l2_search_set_mfma_min_nq(int(n)), "ragk_l2_search_set_mfma_min_nq")


_search_ws = {}
_search_lock = threading.Lock()


# Results in host memory up to this many are stored there by the merge itself (pinned, 12 bytes each) and watched arriving
# (search.hip ragk_search_collect), instead of copied behind it: one query of 10000 x 384 40.4 us copied, 38.0 stored and the stream
# waited for, 26 watched; 5 of 2000 x 384 47 -> 37, 256 of 10000 x 384 110 -> 102, 32 of 500000 x 1024 411 -> 402.
SEARCH_STORE = 16384


def search_block():
    """Pinned memory for the results of any one search. Always this size, so that torch's pool has a block for every search once
    it has one (one more for each search that runs beside it): by the results' own sizes the first search of each power of two of
    them paid for an allocation (10000 x 384 rows, 1 x 10, 4 x 10, 64 x 10 results: 150 to 200 us against 50 to 70). An index
    that lies on the device makes it with its store."""
    return torch.empty(3 * SEARCH_STORE, dtype=torch.int32, pin_memory=True)


def _search_to_host(nq, k, launch):
    """(D, I) of a search that launch(ids' address, distances' address) enqueues, in pageable memory of their own."""
    L, n, block = _lib.lib(), nq * k, search_block()
    at, st = block.data_ptr(), stream_ptr()
    check(L.ragk_search_arm(at, n, st), "ragk_search_arm")
    try:
        launch(at, at + 8 * n)
        D, I = torch.empty(nq, k), torch.empty(nq, k, dtype=torch.int64)  # (while the search runs)
        check(L.ragk_search_collect(at, n, I.data_ptr(), D.data_ptr(), st), "ragk_search_collect")
    except BaseException:  # (an interrupt too, wherever it comes)
        L.ragk_stream_wait(st)  # the block goes back to its pool once nothing can write to it
        raise
    return D, I


def _search_views(buf, nq, k, host):
    """(D fp32 [nq, k], I int64 [nq, k]) as views of the ONE allocation a search writes, int64 ids first; host: of a copy in
    pageable memory (a copy of each result waits for the device twice)."""
    if host:
        buf = buf.cpu()
    return (buf.as_strided((nq, k), (k, 1), 2 * nq * k).view(torch.float32),
            buf.as_strided((nq, 2 * k), (2 * k, 1)).view(torch.int64))


def _search(nq, k, device, host, launch):
    """Results of launch(ids' address, distances' address), on the device or (host) in host memory."""
    n = nq * k
    if host and 0 < n <= SEARCH_STORE:
        return _search_to_host(nq, k, launch)
    out = torch.empty(3 * n, dtype=torch.int32, device=device)
    if n:
        launch(out.data_ptr(), out.data_ptr() + 8 * n)
    return _search_views(out, nq, k, host)


def _search_partials(n_entries, device):
    """Addresses of the partial lists (fp32 distances, int32 ids) in a grow-only workspace of this device and stream. Callers hold
    _search_lock from here until both kernels of the search are enqueued, so two searches on one stream
    never interleave their scan / merge pair over the same buffer."""
    key = (device.index, stream_ptr())
    ws = _search_ws.get(key)
    if ws is None or ws.numel() < 2 * n_entries:
        ws = torch.empty(max(2 * n_entries, 1 << 16), dtype=torch.int32, device=device)
        _search_ws[key] = ws
    at = ws.data_ptr()
    return at, at + 4 * n_entries


def l2_search(xt, cap, n, q, k, row_begin=0, ids_map=None, host=False):
    """Exact squared-L2 top-k over rows [row_begin, n) of a column-major store xt[d][cap]
    (csrc/kernels/search.hip: l2_scan with wave-resident running top lists + one list merge; batches
    of >= 16 queries with k <= 8 on the fp32-MFMA distance GEMM, faiss' BLAS form).
    Returns (D fp32 [nq,k], I int64 [nq,k]) with faiss padding semantics (-1, FLT_MAX), on the device or (host) in host memory.
    Host cost per call: one output block, two ctypes calls (the partial lists live in a cached
    workspace) and, for results in host memory, the marks ahead of them and the watch for them."""
    _req(xt.is_cuda and xt.dtype == torch.float32 and xt.is_contiguous() and xt.dim() == 2, "xt fp32 [d, cap]")
    _req(q.is_cuda and q.dtype == torch.float32 and q.is_contiguous() and q.dim() == 2, "q fp32 [nq, d]")
    d = xt.shape[0]
    nq = q.shape[0]
    _req(q.shape[1] == d, "dim mismatch")
    _req(1 <= k <= 64, "1 <= k <= 64")
    _req(xt.shape[1] == cap and 0 <= row_begin <= max(row_begin, n) <= cap, "rows within the store")
    _req(ids_map is None or (ids_map.dtype == torch.int32 and ids_map.is_cuda and ids_map.numel() >= n), "ids_map")
    L = _lib.lib()

    def launch(ids, dist):
        G = L.ragk_l2_search_groups(row_begin, max(n, row_begin), nq, k, d)
        with _search_lock:
            pd, pi = _search_partials(nq * G * k, q.device)
            check(L.ragk_l2_search(xt.data_ptr(), cap, d, row_begin, max(n, row_begin), q.data_ptr(), nq, k, ptr(ids_map), pd, pi,
                                   dist, ids, stream_ptr()), "ragk_l2_search")

    return _search(nq, k, q.device, host, launch)


def ivf_search(xt, cap, q, probes, offsets, ids_map, k, max_list=None, ends=None, host=False):
    """IVF-Flat scan of the probed lists (one block per (query, probe), wave-resident top lists,
    then one list merge). probes int32 [nq, nprobe] (device; -1 = no list); list i occupies store rows
    [offsets[i], ends[i]) (ends None: packed lists, offsets has nlist+1 entries); ids_map int32 [cap]
    original id of every store row. max_list is accepted for API compatibility (unused)."""
    _req(xt.dtype == torch.float32 and q.dtype == torch.float32 and q.is_contiguous(), "fp32")
    _req(probes.dtype == torch.int32 and offsets.dtype == torch.int32 and ids_map.dtype == torch.int32, "int32")
    _req(probes.is_contiguous() and probes.is_cuda and offsets.is_cuda and ids_map.is_cuda, "device int32")
    _req(ends is None or (ends.dtype == torch.int32 and ends.is_cuda), "ends int32")
    d = xt.shape[0]
    nq, nprobe = probes.shape
    _req(1 <= k <= 64 and d <= 2048 and nprobe >= 1, "k <= 64, d <= 2048")

    def launch(ids, dist):
        with _search_lock:
            pd, pi = _search_partials(nq * nprobe * k, q.device)
            check(_lib.lib().ragk_ivf_search(xt.data_ptr(), cap, d, q.data_ptr(), nq, probes.data_ptr(), nprobe,
                                             offsets.data_ptr(), ptr(ends), ids_map.data_ptr(), k, pd, pi, dist, ids,
                                             stream_ptr()), "ragk_ivf_search")

    return _search(nq, k, q.device, host, launch)


def kmeans_assign(x, c, cnorm=None, scores=None):
    """argmin_j ||x_i - c_j||^2 (ties -> lower j) and that squared distance, on the MFMA distance-GEMM
    kernel (exact fp32 products). x [n, d], c [k, d] fp32 contiguous on the GPU; d % 64 == 0, <= 1024.
    scores (optional fp32 [n, k]): receives -(||c_j||^2 - 2 x_i.c_j), the numbers the argmin ranks."""
    _req(x.is_cuda and x.dtype == torch.float32 and x.is_contiguous() and x.dim() == 2, "x fp32 [n, d]")
    _req(c.is_cuda and c.dtype == torch.float32 and c.is_contiguous() and c.shape[1] == x.shape[1], "c fp32 [k, d]")
    n, d = x.shape
    _req(d % 64 == 0 and d <= 1024, "d % 64 == 0 and d <= 1024")
    _req(scores is None or (scores.is_cuda and scores.dtype == torch.float32 and scores.is_contiguous()
                            and tuple(scores.shape) == (n, c.shape[0])), "scores fp32 [n, k]")
    if cnorm is None:
        cnorm = (c * c).sum(1)
    a = torch.empty(n, dtype=torch.int32, device=x.device)
    dist = torch.empty(n, dtype=torch.float32, device=x.device)
    check(_lib.lib().ragk_kmeans_assign(x.data_ptr(), n, d, c.data_ptr(), cnorm.contiguous().data_ptr(), c.shape[0],
                                        a.data_ptr(), dist.data_ptr(), ptr(scores), stream_ptr()), "ragk_kmeans_assign")
    return a, dist


def coarse_probes(x, c, cnorm, nprobe):
    """IVF coarse search: the nprobe nearest centroids of every row of x (int32 [n, nprobe], ties ->
    lower id), ranked by the SAME scores kmeans_assign's argmin uses, so top-1 == the list assignment."""
    n, nl = x.shape[0], c.shape[0]
    _req(1 <= nprobe <= min(256, nl) and nl <= 24576, "1 <= nprobe <= min(256, nlist), nlist <= 24576")
    sc = torch.empty((n, nl), dtype=torch.float32, device=x.device)
    kmeans_assign(x, c, cnorm, scores=sc)
    _, idx = topk_candidates(sc, nprobe, chunks=1)
    return idx


def l2_scatter(xt, cap, pos, x):
    """Store rows x [n, d] at slots pos (int32, each < cap) of the column-major store xt[d][cap]."""
    _req(x.dtype == torch.float32 and x.is_contiguous() and x.shape[1] == xt.shape[0], "x fp32 [n,d]")
    _req(pos.dtype == torch.int32 and pos.is_cuda and pos.numel() == x.shape[0], "pos int32 [n]")
    check(_lib.lib().ragk_l2_scatter(xt.data_ptr(), cap, xt.shape[0], pos.data_ptr(), x.data_ptr(), x.shape[0],
                                     stream_ptr()), "ragk_l2_scatter")


def l2_append(xt, cap, n0, x):
    _req(x.dtype == torch.float32 and x.is_contiguous() and x.shape[1] == xt.shape[0], "x fp32 [n,d]")
    check(_lib.lib().ragk_l2_append(xt.data_ptr(), cap, xt.shape[0], n0, x.data_ptr(), x.shape[0], stream_ptr()),
          "ragk_l2_append")


