// bf16 GEMMs of decode steps (M <= 64) for gfx950: C[M,N] = A[M,K] . B[N,K]^T  (+ fused epilogue)
//
// B is the HF weight layout [out_features, in_features], so both operands are
// K-contiguous and every MFMA fragment is one 16-byte load.
//
//  * gemm_skinny : weight-streaming: every weight byte is
//                  read exactly once straight into VGPRs (no LDS round trip), 8
//                  waves per block split K, MFMA with the activations as the A
//                  operand, cross-wave reduction through LDS, fused epilogue.
//  * gemm_gemv   : the same software-pipelined (explicit path 3).
//
// Replaces reference ops K3/K7/K8/K9/K10/K11 (the reference
// runs them as fp32 ATen CPU matmuls inside transformers' LlamaForCausalLM,
// /root/reference/llm/rag.py:24,172) and encoder ops E2/E4/E5/E6.
#include <stdlib.h>

#include "common.h"
using namespace ragk;

namespace {

// ------------------------------------------------------------------------------------
// Skinny (decode) GEMM. Block = WAVES waves handling one 16-column output tile; the
// waves take interleaved 128-deep K blocks (4 MFMA k-steps each), so the block
// streams each of its 16 weight rows front-to-back exactly once.
// ------------------------------------------------------------------------------------
constexpr int SK_WAVES = 8;

// (16 waves per block measured slower on the batch-1 down projection: more waves lengthen the LDS
// reduction and the per-block tail more than the extra loads in flight gain; two K blocks in flight per
// wave and non-temporal weight loads were slower at C=1 too -- profiles/c1_skinny_*_ab_r4.log.)
template <int MT, int EPI, bool OUT_F32>
__global__ __launch_bounds__(SK_WAVES * 64) void gemm_skinny_kernel(
    const bf16_t* __restrict__ X, int ldx, const bf16_t* __restrict__ W, int ldw, void* C, int ldc,
    const bf16_t* __restrict__ bias, const bf16_t* resid, int ldr, int M, int N, int K) {
  constexpr int WV = SK_WAVES;
  constexpr bool PAIR = epi_pair(EPI);
  constexpr int NACC = PAIR ? 2 : 1;
  __shared__ __attribute__((aligned(16))) f32x4 red[WV][NACC * MT][64];

  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int fr = lane & 15, fh = lane >> 4;
  const int n0 = blockIdx.x * 16;
  // weight rows for this lane's output column (packed gate/up layout for SILU_MUL:
  // 128-row tiles = [64 gate | 64 up])
  int wrow0, wrow1 = 0;
  if constexpr (PAIR) {
    const int g = n0 + fr;
    wrow0 = (g >> 6) * 128 + (g & 63);
    wrow1 = wrow0 + 64;
  } else {
    wrow0 = min(n0 + fr, N - 1);
  }
  const bf16_t* w0 = W + (size_t)wrow0 * ldw + fh * 8;
  const bf16_t* w1 = W + (size_t)wrow1 * ldw + fh * 8;
  const bf16_t* xr[MT];
  bool xv[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int m = t * 16 + fr;
    xv[t] = m < M;
    xr[t] = X + (size_t)(xv[t] ? m : 0) * ldx + fh * 8;
  }

  f32x4 acc[NACC][MT];
#pragma unroll
  for (int a = 0; a < NACC; ++a)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[a][t] = (f32x4){0.f, 0.f, 0.f, 0.f};

  const int nkb = K >> 7;  // 128-deep K blocks
  const bf16x8 zero = (bf16x8){0, 0, 0, 0, 0, 0, 0, 0};
  constexpr int U = 1;  // K blocks per wave per iteration (default cache policy for the weights)
  for (int kb = wid; kb < nkb; kb += U * WV) {
    bf16x8 wf[U][NACC][4];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = min(kb + u * WV, nkb - 1) * 128;  // clamped: a missing second block is loaded, not used
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        wf[u][0][s] = *reinterpret_cast<const bf16x8*>(w0 + k + 32 * s);
        if constexpr (PAIR) wf[u][1][s] = *reinterpret_cast<const bf16x8*>(w1 + k + 32 * s);
      }
    }
    bf16x8 xf[U][MT][4];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = min(kb + u * WV, nkb - 1) * 128;
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int s = 0; s < 4; ++s)
          xf[u][t][s] = xv[t] ? *reinterpret_cast<const bf16x8*>(xr[t] + k + 32 * s) : zero;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (kb + u * WV >= nkb) break;  // wave-uniform
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
          for (int a = 0; a < NACC; ++a)
            acc[a][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf[u][t][s], wf[u][a][s], acc[a][t], 0, 0, 0);
    }
  }

#pragma unroll
  for (int a = 0; a < NACC; ++a)
#pragma unroll
    for (int t = 0; t < MT; ++t) red[wid][a * MT + t][lane] = acc[a][t];
  __syncthreads();

  // reduce over waves; element e = (t, lane, r): row = 16t + 4*(lane>>4) + r, col = n0 + (lane&15)
  for (int e = threadIdx.x; e < MT * 64 * 4; e += WV * 64) {
    const int t = e >> 8, ln = (e >> 2) & 63, r = e & 3;
    const int row = t * 16 + 4 * (ln >> 4) + r;
    const int col = n0 + (ln & 15);
    if (row >= M || col >= N) continue;
    float v = 0.f, u = 0.f;
#pragma unroll
    for (int w = 0; w < WV; ++w) {
      v += red[w][t][ln][r];
      if constexpr (PAIR) u += red[w][MT + t][ln][r];
    }
    if constexpr (PAIR) v = glu_act<EPI>(v, u, glu_par<EPI>(bias));
    if constexpr (EPI == EPI_BIAS || EPI == EPI_BIAS_RESID || EPI == EPI_BIAS_GELU ||
                  EPI == EPI_BIAS_GELU_TANH)
      v += bf2f(bias[col]);
    if constexpr (EPI == EPI_RESID || EPI == EPI_BIAS_RESID) v += bf2f(resid[(size_t)row * ldr + col]);
    if constexpr (EPI == EPI_BIAS_GELU || EPI == EPI_GELU) v = gelu_erf(v);
    if constexpr (EPI == EPI_BIAS_GELU_TANH) v = gelu_tanh(v);
    if constexpr (OUT_F32)
      reinterpret_cast<float*>(C)[(size_t)row * ldc + col] = v;
    else
      reinterpret_cast<bf16_t*>(C)[(size_t)row * ldc + col] = f2bf(v);
  }
}

// ------------------------------------------------------------------------------------
// Pipelined weight-streaming GEMV/GEMM for decode (M <= 64), v2.
//  * software pipeline: the next 128-deep K block's weights + activations are loaded into a
//    second register set while the MFMAs of the current one run (the v1 loop was latency-bound:
//    load -> wait -> 4 MFMAs, ~4 iterations per wave);
//  * weights are streamed with non-temporal loads (read exactly once);
//  * NT n-tiles per wave reuse each activation fragment NT times (cuts the L2 activation
//    traffic that dominated at M = 32..64);
//  * rows >= M read a clamped (valid) row: their outputs are garbage but never stored, so no
//    per-element select sits between a load and its MFMA.
// ------------------------------------------------------------------------------------
template <int MT, int NT, int NACC>
struct GemvFrags {
  bf16x8 w[NACC][NT][4];
  bf16x8 x[MT][4];
};

template <int MT, int NT, int EPI, bool OUT_F32>
__global__ __launch_bounds__(SK_WAVES * 64) void gemm_gemv_kernel(
    const bf16_t* __restrict__ X, int ldx, const bf16_t* __restrict__ W, int ldw, void* C, int ldc,
    const bf16_t* __restrict__ bias, const bf16_t* resid, int ldr, int M, int N, int K) {
  constexpr bool PAIR = epi_pair(EPI);
  constexpr int NACC = PAIR ? 2 : 1;
  __shared__ __attribute__((aligned(16))) f32x4 red[SK_WAVES][NACC * NT * MT][64];

  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int fr = lane & 15, fh = lane >> 4;
  const int nbase = blockIdx.x * 16 * NT;
  const bf16_t* wp[NACC][NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int col = nbase + 16 * j + fr;
    if constexpr (PAIR) {
      const int r0 = (col >> 6) * 128 + (col & 63);
      wp[0][j] = W + (size_t)r0 * ldw + fh * 8;
      wp[1][j] = W + (size_t)(r0 + 64) * ldw + fh * 8;
    } else {
      wp[0][j] = W + (size_t)min(col, N - 1) * ldw + fh * 8;
    }
  }
  const bf16_t* xp[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) xp[t] = X + (size_t)min(t * 16 + fr, M - 1) * ldx + fh * 8;

  f32x4 acc[NACC][NT][MT];
#pragma unroll
  for (int a = 0; a < NACC; ++a)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int t = 0; t < MT; ++t) acc[a][j][t] = (f32x4){0.f, 0.f, 0.f, 0.f};

  auto load = [&](GemvFrags<MT, NT, NACC>& f, int kb) {
    const int k = kb * 128;
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int a = 0; a < NACC; ++a)
#pragma unroll
        for (int j = 0; j < NT; ++j)
          f.w[a][j][s] = __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(wp[a][j] + k + 32 * s));
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int s = 0; s < 4; ++s) f.x[t][s] = *reinterpret_cast<const bf16x8*>(xp[t] + k + 32 * s);
  };
  auto compute = [&](const GemvFrags<MT, NT, NACC>& f) {
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int a = 0; a < NACC; ++a)
#pragma unroll
          for (int j = 0; j < NT; ++j)
            acc[a][j][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.x[t][s], f.w[a][j][s], acc[a][j][t], 0, 0, 0);
  };

  const int nkb = K >> 7;
  GemvFrags<MT, NT, NACC> fa, fb;
  int kb = wid;
  if (kb < nkb) load(fa, kb);
  for (; kb < nkb; kb += 2 * SK_WAVES) {
    const int kb2 = kb + SK_WAVES;
    if (kb2 < nkb) load(fb, kb2);
    compute(fa);
    const int kb3 = kb2 + SK_WAVES;
    if (kb3 < nkb) load(fa, kb3);
    if (kb2 < nkb) compute(fb);
  }

#pragma unroll
  for (int a = 0; a < NACC; ++a)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int t = 0; t < MT; ++t) red[wid][(a * NT + j) * MT + t][lane] = acc[a][j][t];
  __syncthreads();

  // element e = (j, t, lane, r): row = 16t + 4*(lane>>4) + r, col = nbase + 16j + (lane&15)
  for (int e = threadIdx.x; e < NT * MT * 64 * 4; e += SK_WAVES * 64) {
    const int j = e / (MT * 256), rem = e % (MT * 256);
    const int t = rem >> 8, ln = (rem >> 2) & 63, r = rem & 3;
    const int row = t * 16 + 4 * (ln >> 4) + r;
    const int col = nbase + 16 * j + (ln & 15);
    if (row >= M || col >= N) continue;
    float v = 0.f, u = 0.f;
#pragma unroll
    for (int w = 0; w < SK_WAVES; ++w) {
      v += red[w][j * MT + t][ln][r];
      if constexpr (PAIR) u += red[w][(NT + j) * MT + t][ln][r];
    }
    if constexpr (PAIR) v = glu_act<EPI>(v, u, glu_par<EPI>(bias));
    if constexpr (EPI == EPI_BIAS || EPI == EPI_BIAS_RESID || EPI == EPI_BIAS_GELU || EPI == EPI_BIAS_GELU_TANH)
      v += bf2f(bias[col]);
    if constexpr (EPI == EPI_RESID || EPI == EPI_BIAS_RESID) v += bf2f(resid[(size_t)row * ldr + col]);
    if constexpr (EPI == EPI_BIAS_GELU || EPI == EPI_GELU) v = gelu_erf(v);
    if constexpr (EPI == EPI_BIAS_GELU_TANH) v = gelu_tanh(v);
    if constexpr (OUT_F32)
      reinterpret_cast<float*>(C)[(size_t)row * ldc + col] = v;
    else
      reinterpret_cast<bf16_t*>(C)[(size_t)row * ldc + col] = f2bf(v);
  }
}

template <int MT, int NT, int EPI, bool F32>
hipError_t launch_gemv(const void* X, int ldx, const void* W, int ldw, void* C, int ldc, const void* bias,
                       const void* resid, int ldr, int M, int N, int K, hipStream_t st) {
  hipLaunchKernelGGL((gemm_gemv_kernel<MT, NT, EPI, F32>), dim3((N + 16 * NT - 1) / (16 * NT)), dim3(SK_WAVES * 64),
                     0, st, (const bf16_t*)X, ldx, (const bf16_t*)W, ldw, C, ldc, (const bf16_t*)bias,
                     (const bf16_t*)resid, ldr, M, N, K);
  return hipGetLastError();
}

// NT=2 when it still leaves >= 2 blocks per CU (and PAIR needs N % 32 for whole tiles)
template <int EPI, bool F32>
hipError_t dispatch_gemv(const void* X, int ldx, const void* W, int ldw, void* C, int ldc, const void* bias,
                         const void* resid, int ldr, int M, int N, int K, hipStream_t st) {
  const int mt = (M + 15) / 16;
  const bool nt2 = M > 16 && N >= 32 * 512 && (!epi_pair(EPI) || N % 32 == 0);
#define RAGK_GV(MTV)                                                                                         \
  case MTV:                                                                                                  \
    if (nt2 && MTV <= 2)                                                                                     \
      return launch_gemv<MTV, (MTV <= 2 ? 2 : 1), EPI, F32>(X, ldx, W, ldw, C, ldc, bias, resid, ldr, M, N, K, st); \
    return launch_gemv<MTV, 1, EPI, F32>(X, ldx, W, ldw, C, ldc, bias, resid, ldr, M, N, K, st);
  switch (mt) {
    RAGK_GV(1)
    RAGK_GV(2)
    RAGK_GV(3)
    RAGK_GV(4)
    default: return hipErrorInvalidValue;
  }
#undef RAGK_GV
}

template <int MT, int EPI, bool F32>
hipError_t launch_skinny(const void* X, int ldx, const void* W, int ldw, void* C, int ldc, const void* bias,
                         const void* resid, int ldr, int M, int N, int K, hipStream_t st) {
  hipLaunchKernelGGL((gemm_skinny_kernel<MT, EPI, F32>), dim3((N + 15) / 16), dim3(SK_WAVES * 64), 0, st,
                     (const bf16_t*)X, ldx, (const bf16_t*)W, ldw, C, ldc, (const bf16_t*)bias,
                     (const bf16_t*)resid, ldr, M, N, K);
  return hipGetLastError();
}

template <int EPI, bool F32>
hipError_t dispatch_skinny(const void* X, int ldx, const void* W, int ldw, void* C, int ldc, const void* bias,
                           const void* resid, int ldr, int M, int N, int K, hipStream_t st) {
  const int mt = (M + 15) / 16;
  switch (mt) {
    case 1: return launch_skinny<1, EPI, F32>(X, ldx, W, ldw, C, ldc, bias, resid, ldr, M, N, K, st);
    case 2: return launch_skinny<2, EPI, F32>(X, ldx, W, ldw, C, ldc, bias, resid, ldr, M, N, K, st);
    case 3: return launch_skinny<3, EPI, F32>(X, ldx, W, ldw, C, ldc, bias, resid, ldr, M, N, K, st);
    case 4: return launch_skinny<4, EPI, F32>(X, ldx, W, ldw, C, ldc, bias, resid, ldr, M, N, K, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

// N here is the number of OUTPUT columns. For EPI_SILU_MUL / EPI_GLU_CLIP the weight has 2*N rows
// in the packed [64 gate | 64 up] tile layout and N must be a multiple of 64. M <= 64.
RAGK_API int ragk_gemm(const void* A, int lda, const void* B, int ldb, void* C, int ldc, const void* bias,
                       const void* resid, int ldr, int M, int N, int K, int epi, int out_f32, hipStream_t st) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  if (K % 128 != 0 || M > 64) return (int)hipErrorInvalidValue;
  if (epi_pair(epi) && (N % 64 != 0 || out_f32)) return (int)hipErrorInvalidValue;
  if (epi == EPI_SILU_MUL)
    return (int)dispatch_skinny<EPI_SILU_MUL, false>(A, lda, B, ldb, C, ldc, bias, resid, ldr, M, N, K, st);
  if (epi == EPI_GLU_CLIP) {
    if (!bias) return (int)hipErrorInvalidValue;
    return (int)dispatch_skinny<EPI_GLU_CLIP, false>(A, lda, B, ldb, C, ldc, bias, resid, ldr, M, N, K, st);
  }
#define RAGK_GEMM_CASE(E)                                                                               \
  case E:                                                                                               \
    return out_f32 ? (int)dispatch_skinny<E, true>(A, lda, B, ldb, C, ldc, bias, resid, ldr, M, N, K, st) \
                   : (int)dispatch_skinny<E, false>(A, lda, B, ldb, C, ldc, bias, resid, ldr, M, N, K, st);
  switch (epi) {
    RAGK_GEMM_CASE(EPI_NONE)
    RAGK_GEMM_CASE(EPI_BIAS)
    RAGK_GEMM_CASE(EPI_RESID)
    RAGK_GEMM_CASE(EPI_BIAS_RESID)
    RAGK_GEMM_CASE(EPI_BIAS_GELU)
    RAGK_GEMM_CASE(EPI_GELU)
    RAGK_GEMM_CASE(EPI_BIAS_GELU_TANH)
    default: return (int)hipErrorInvalidValue;
  }
#undef RAGK_GEMM_CASE
}

// Force a specific path (tests / benchmarks): path 1 = skinny v1, 3 = pipelined gemv v2.
RAGK_API int ragk_gemm_path(int path, const void* A, int lda, const void* B, int ldb, void* C, int ldc,
                            const void* bias, const void* resid, int ldr, int M, int N, int K, int epi,
                            hipStream_t st) {
  if (K % 128 != 0 || M > 64) return (int)hipErrorInvalidValue;
  if (path == 3) {
    if (epi == EPI_SILU_MUL) return (int)dispatch_gemv<EPI_SILU_MUL, false>(A, lda, B, ldb, C, ldc, bias, resid, ldr, M, N, K, st);
    if (epi == EPI_NONE) return (int)dispatch_gemv<EPI_NONE, false>(A, lda, B, ldb, C, ldc, bias, resid, ldr, M, N, K, st);
    if (epi == EPI_RESID) return (int)dispatch_gemv<EPI_RESID, false>(A, lda, B, ldb, C, ldc, bias, resid, ldr, M, N, K, st);
    return (int)hipErrorInvalidValue;
  }
  if (path != 1) return (int)hipErrorInvalidValue;
  if (epi == EPI_SILU_MUL) return (int)dispatch_skinny<EPI_SILU_MUL, false>(A, lda, B, ldb, C, ldc, bias, resid, ldr, M, N, K, st);
  if (epi == EPI_NONE) return (int)dispatch_skinny<EPI_NONE, false>(A, lda, B, ldb, C, ldc, bias, resid, ldr, M, N, K, st);
  if (epi == EPI_RESID) return (int)dispatch_skinny<EPI_RESID, false>(A, lda, B, ldb, C, ldc, bias, resid, ldr, M, N, K, st);
  return (int)hipErrorInvalidValue;
}
