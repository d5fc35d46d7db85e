// Sentence encoders: pooling + L2 normalise (E7: CLS / masked mean, sentence-transformers Normalize(),
// /root/reference/llm/rag.py:55 normalize_embeddings=True).
#include "common.h"
using namespace ragk;

namespace {

// out[b] = normalize(pool(hidden[cu[b]:cu[b+1]])) in fp32. mode 0 = CLS (first token),
// mode 1 = masked mean over the sequence, mode 2 = last token. One block a sequence: a thread owns eight columns of every
// RG-th row (a column a thread and a row at a time before: mean of 80 x 160 rows of 384 columns 45 -> 9.4 us, of 12 x 1146 of 1024
// 1207 -> 25). VEC = 1 for widths
// or row strides that are no multiple of eight.
constexpr int POOL_NT = 1024, POOL_MAXH = 2048;
template <int VEC>
__global__ __launch_bounds__(POOL_NT) void pool_l2norm_kernel(const bf16_t* __restrict__ hidden, int ld,
                                                              const int* __restrict__ cu, const int* __restrict__ rows,
                                                              float* out, int ldo, int H, int mode, int normalize) {
  __shared__ float part[POOL_NT * 8];
  __shared__ float red[POOL_NT / 64];
  const int b = blockIdx.x;
  const int s0 = cu[b], s1 = cu[b + 1];
  const int len = s1 - s0;
  const int first = mode == 2 ? s1 - 1 : s0, last = mode == 1 ? s1 : first + 1;
  const int groups = (H + VEC - 1) / VEC;            // column groups of VEC
  const int RG = groups < POOL_NT ? POOL_NT / groups : 1;  // row groups
  constexpr int CG = VEC == 8 ? 1 : (POOL_MAXH + POOL_NT - 1) / POOL_NT;  // column groups of a thread
  const int rg = RG > 1 ? threadIdx.x / groups : 0, c0 = RG > 1 ? threadIdx.x % groups : threadIdx.x;
  float acc[CG][VEC];
#pragma unroll
  for (int k = 0; k < CG; ++k)
#pragma unroll
    for (int e = 0; e < VEC; ++e) acc[k][e] = 0.f;
  if (rg < RG) {
#pragma unroll
    for (int k = 0; k < CG; ++k) {
      const int c = c0 + k * POOL_NT;
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
    const int c = c0 + k * POOL_NT;
    if (c < groups)
#pragma unroll
      for (int e = 0; e < VEC; ++e) o[c * VEC + e] = acc[k][e] * scale;
  }
}


}  // namespace

// The pooled sequence b goes to row rows[b] of out (rows null: row b), row stride ldo.
RAGK_API int ragk_pool_l2norm_rows(const void* hidden, int ld, const int* cu, const int* rows, float* out, int ldo, int B, int H,
                                   int mode, int normalize, hipStream_t st) {
  if (B <= 0) return 0;
  if (H > POOL_MAXH) return (int)hipErrorInvalidValue;
  const auto kernel = H % 8 == 0 && ld % 8 == 0 && (uintptr_t)hidden % 16 == 0 ? pool_l2norm_kernel<8> : pool_l2norm_kernel<1>;
  hipLaunchKernelGGL(kernel, dim3(B), dim3(POOL_NT), 0, st, (const bf16_t*)hidden, ld, cu, rows, out, ldo, H, mode, normalize);
  return (int)hipGetLastError();
}

RAGK_API int ragk_pool_l2norm(const void* hidden, int ld, const int* cu, float* out, int B, int H, int mode,
                              int normalize, hipStream_t st) {
  return ragk_pool_l2norm_rows(hidden, ld, cu, nullptr, out, H, B, H, mode, normalize, st);
}
