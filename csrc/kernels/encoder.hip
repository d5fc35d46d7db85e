// Sentence encoders: pooling + L2 normalise (E7: CLS / masked mean, sentence-transformers Normalize(),
// /root/reference/llm/rag.py:55 normalize_embeddings=True), and one forward over packed sequences as a single host call.
//
// A short text's embedding is about 45 launches of 2 to 5 us each (6 layers); issued one by one from Python they took 14 us each and
// the GPU idled between them. The kernels of the layers are those of gemm*.hip, attention.hip and norm.hip; a single sequence of
// at most 32 rows takes encoder_few.hip's.
#include "encoder.h"
using namespace ragk;

extern "C" {
int ragk_gemm(const void*, int, const void*, int, void*, int, const void*, const void*, int, int, int, int, int, int, hipStream_t);
int ragk_gemm_w4_tile(const void*, int, const void*, int, void*, int, const void*, const void*, int, int, int, int, int, int, int,
                      hipStream_t);
int ragk_gemm_mid(const void*, int, const void*, int, void*, int, const void*, const void*, int, int, int, int, int, int, int,
                  int, float*, hipStream_t);
int ragk_attn_prefill(const void*, int, const void*, const void*, int, const int*, int, const int*, const int*, const int*,
                      const int*, int, void*, int, int, int, int, int, int, float, hipStream_t);
int ragk_gemm_part(const void*, int, const void*, int, float*, int, int, int, int, hipStream_t);
int ragk_layernorm_slabs(const float*, int, const void*, const void*, int, const void*, const void*, void*, int, int, int, float,
                         hipStream_t);
int ragk_layernorm(const void*, int, const void*, int, const void*, const void*, void*, int, int, int, float, hipStream_t);
int ragk_embed_ln(const int*, const int*, const void*, const void*, const void*, const void*, const void*, void*, int, int,
                  float, int, hipStream_t);
}

namespace {

// out[b] = normalize(pool(hidden[cu[b]:cu[b+1]])) in fp32. mode 0 = CLS (first token),
// mode 1 = masked mean over the sequence, mode 2 = last token. One block a sequence: a thread owns eight columns of every
// RG-th row (a column a thread and a row at a time before: mean of 80 x 160 rows of 384 columns 45 -> 9.4 us, of 12 x 1146 of 1024
// 1207 -> 25). Modes 0 and 2 read one row: NT = 256 threads and one row group, not the mean's 1024 (300 sequences of 384
// columns 5.4 -> 3.6 us).
// VEC = 1 for widths or row strides that are no multiple of eight.
constexpr int POOL_MAXH = 2048;
template <int VEC, int NT>
__global__ __launch_bounds__(NT) void pool_l2norm_kernel(const bf16_t* __restrict__ hidden, int ld,
                                                              const int* __restrict__ cu, const int* __restrict__ rows,
                                                              float* out, int ldo, int H, int mode, int normalize) {
  __shared__ float part[NT == 256 ? 1 : NT * 8];
  __shared__ float red[NT / 64];
  const int b = blockIdx.x;
  const int s0 = cu[b], s1 = cu[b + 1];
  const int len = s1 - s0;
  const int first = mode == 2 ? s1 - 1 : s0, last = mode == 1 ? s1 : first + 1;
  const int groups = (H + VEC - 1) / VEC;            // column groups of VEC
  const int RG = NT > 256 && groups < NT ? NT / groups : 1;  // row groups
  constexpr int CG = (POOL_MAXH / VEC + NT - 1) / NT;  // column groups of a thread
  const int rg = RG > 1 ? threadIdx.x / groups : 0, c0 = RG > 1 ? threadIdx.x % groups : threadIdx.x;
  float acc[CG][VEC];
#pragma unroll
  for (int k = 0; k < CG; ++k)
#pragma unroll
    for (int e = 0; e < VEC; ++e) acc[k][e] = 0.f;
  if (rg < RG) {
#pragma unroll
    for (int k = 0; k < CG; ++k) {
      const int c = c0 + k * NT;
      if (c >= groups) continue;
      const bf16_t* col = hidden + (size_t)c * VEC;
#pragma unroll 4
      for (int t = first + rg; t < last; t += RG) {
        if constexpr (VEC == 8) {
          float f[8];
          unpack8(*reinterpret_cast<const u32x4*>(col + (size_t)t * ld), f);
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[k][e] += f[e];
        } else {
          acc[k][0] += bf2f(col[(size_t)t * ld]);
        }
      }
    }
  }
  // row groups -> the first one, in order
  if (RG > 1) {
#pragma unroll
    for (int e = 0; e < VEC; ++e) part[threadIdx.x * VEC + e] = acc[0][e];
    __syncthreads();
    if (threadIdx.x < groups)
      for (int r = 1; r < RG; ++r)
#pragma unroll
        for (int e = 0; e < VEC; ++e) acc[0][e] += part[(r * groups + threadIdx.x) * VEC + e];
  }
  const float inv = mode == 1 ? (len > 0 ? 1.f / (float)len : 0.f) : 1.f;
  const bool mine = RG == 1 || threadIdx.x < groups;
  float ss = 0.f;
#pragma unroll
  for (int k = 0; k < CG; ++k)
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      acc[k][e] *= inv;
      if (mine) ss += acc[k][e] * acc[k][e];
    }
  float scale = 1.f;
  if (normalize) {
    ss = block_sum(ss, red);
    scale = 1.f / fmaxf(sqrtf(ss), 1e-12f);  // torch.nn.functional.normalize eps
  }
  if (!mine) return;
  float* o = out + (size_t)(rows ? rows[b] : b) * ldo;
#pragma unroll
  for (int k = 0; k < CG; ++k) {
    const int c = c0 + k * NT;
    if (c < groups)
#pragma unroll
      for (int e = 0; e < VEC; ++e) o[c * VEC + e] = acc[k][e] * scale;
  }
}


int product(const Plan& plan, const void* x, int K, const void* w, int N, const void* bias, const void* resid, void* out, int epi,
            float* ws, hipStream_t st) {
  for (int i = 0; i < plan.n; ++i) {
    const Piece& p = plan.p[i];
    const char* px = (const char*)x + (size_t)p.r0 * K * 2;
    const char* pr = resid ? (const char*)resid + (size_t)p.r0 * N * 2 : nullptr;
    char* po = (char*)out + (size_t)p.r0 * N * 2;
    const int M = p.r1 - p.r0;
    const int rc = p.mi < 0    ? ragk_gemm(px, K, w, K, po, N, bias, pr, N, M, N, K, epi, 0, st)
                   : p.mi == 0 || p.mi > 32
                       ? ragk_gemm_w4_tile(px, K, w, K, po, N, bias, pr, N, M, N, K, epi, 0, p.mi ? p.mi - 32 : 8, st)
                       : ragk_gemm_mid(px, K, w, K, po, N, bias, pr, N, M, N, K, epi, 0, p.mi, p.S, ws, st);
    if (rc) return rc;
  }
  return 0;
}

// norm(x . w^T + bias + h) into h
int product_norm(const EncoderCall& c, const Plan& plan, const void* x, int K, const void* w, const void* bias, const void* g,
                 const void* b, hipStream_t st) {
  const Piece& p = plan.p[0];
  if (!plan.slabs) {
    const int rc = product(plan, x, K, w, c.H, bias, c.h, c.a, EPI_BIAS_RESID, c.ws, st);
    return rc ? rc : ragk_layernorm(c.a, c.H, nullptr, 0, g, b, c.h, c.H, c.T, c.H, c.eps, st);
  }
  const int rc = p.mi < 0 ? ragk_gemm_part(x, K, w, K, c.ws, c.T, c.H, K, K / 64 / p.S, st)
                          : ragk_gemm_mid(x, K, w, K, c.ws, c.H, nullptr, nullptr, 0, c.T, c.H, K, EPI_NONE, 2, p.mi, p.S,
                                          nullptr, st);
  return rc ? rc : ragk_layernorm_slabs(c.ws, p.S, bias, c.h, c.H, g, b, c.h, c.H, c.T, c.H, c.eps, st);
}

// Host integers as a kernel's argument: no copy engine, no wait for what the stream still has to do.
constexpr int PUT_N = 960;
struct PutInts { int v[PUT_N]; };
__global__ __launch_bounds__(256) void put_ints_kernel(PutInts a, int* out, int n) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) out[i] = a.v[i];
}

}  // namespace

// n integers of host memory (read before the call returns) to dst.
RAGK_API int ragk_put_ints(const int* src, int n, int* dst, hipStream_t st) {
  for (int at = 0; at < n; at += PUT_N) {
    PutInts a;
    const int m = n - at < PUT_N ? n - at : PUT_N;
    __builtin_memcpy(a.v, src + at, (size_t)m * 4);
    hipLaunchKernelGGL(put_ints_kernel, dim3((m + 255) / 256), dim3(256), 0, st, a, dst + at, m);
  }
  return (int)hipGetLastError();
}

// The pooled sequence b goes to row rows[b] of out (rows null: row b), row stride ldo.
RAGK_API int ragk_pool_l2norm_rows(const void* hidden, int ld, const int* cu, const int* rows, float* out, int ldo, int B, int H,
                                   int mode, int normalize, hipStream_t st) {
  if (B <= 0) return 0;
  if (H > POOL_MAXH) return (int)hipErrorInvalidValue;
  const bool vec = H % 8 == 0 && ld % 8 == 0 && (uintptr_t)hidden % 16 == 0;
  const auto kernel = mode == 1 ? (vec ? pool_l2norm_kernel<8, 1024> : pool_l2norm_kernel<1, 1024>)
                                : (vec ? pool_l2norm_kernel<8, 256> : pool_l2norm_kernel<1, 256>);
  hipLaunchKernelGGL(kernel, dim3(B), dim3(mode == 1 ? 1024 : 256), 0, st, (const bf16_t*)hidden, ld, cu, rows, out, ldo, H, mode, normalize);
  return (int)hipGetLastError();
}

RAGK_API int ragk_pool_l2norm(const void* hidden, int ld, const int* cu, float* out, int B, int H, int mode,
                              int normalize, hipStream_t st) {
  return ragk_pool_l2norm_rows(hidden, ld, cu, nullptr, out, H, B, H, mode, normalize, st);
}

RAGK_API int ragk_encoder_call_bytes() { return (int)sizeof(EncoderCall); }

RAGK_API int ragk_encoder_forward(const EncoderCall* cp, hipStream_t st) {
  const EncoderCall& c = *cp;
  const int H = c.H, D = H / c.heads, T = c.T;
  if (T <= 0 || c.B <= 0) return 0;
  if (c.few) return encoder_few_forward(c, st);
  const float scale = 1.f / sqrtf((float)D);
#define RAGK_TRY(x) \
  if (const int rc = (x)) return rc
  RAGK_TRY(ragk_embed_ln(c.ids, c.pos, c.word, c.pos_table, c.type_row, c.ln_g, c.ln_b, c.h, T, H, c.eps, 1, st));
  for (int l = 0; l < c.n_layers; ++l) {
    const void* const* w = c.layers + 12 * l;
    RAGK_TRY(product(c.plans[0], c.h, H, w[0], 3 * H, w[1], nullptr, c.qkv, EPI_BIAS, c.ws, st));
    const char* q = (const char*)c.qkv;
    RAGK_TRY(ragk_attn_prefill(q, 3 * H, q + 2 * H, q + 4 * H, 3 * H, nullptr, 0, c.cu, c.cu, c.lens, c.tiles, c.n_tiles, c.attn,
                               H, c.heads, c.heads, D, 0, 0, scale, st));
    RAGK_TRY(product_norm(c, c.plans[1], c.attn, H, w[2], w[3], w[4], w[5], st));
    RAGK_TRY(product(c.plans[2], c.h, H, w[6], c.I, w[7], nullptr, c.f, EPI_BIAS_GELU, c.ws, st));
    RAGK_TRY(product_norm(c, c.plans[3], c.f, c.I, w[8], w[9], w[10], w[11], st));
  }
  RAGK_TRY(ragk_pool_l2norm_rows(c.h, H, c.cu, c.rows, c.out, c.ldo, c.B, H, c.pooling, c.normalize, st));
#undef RAGK_TRY
  return 0;
}
