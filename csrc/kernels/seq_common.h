// Element helpers shared by the kernels that run in bf16 (serving) or fp32 (exact replay).
#pragma once
#include "common.h"

namespace ragk {

template <typename T>
__device__ __forceinline__ float ld1(const T* p);
template <>
__device__ __forceinline__ float ld1<bf16_t>(const bf16_t* p) { return bf2f(*p); }
template <>
__device__ __forceinline__ float ld1<float>(const float* p) { return *p; }

__device__ __forceinline__ void st1(bf16_t* p, float v) { *p = f2bf(v); }
__device__ __forceinline__ void st1(float* p, float v) { *p = v; }

__device__ __forceinline__ void ld8(const bf16_t* p, float* f) { unpack8(*reinterpret_cast<const u32x4*>(p), f); }
__device__ __forceinline__ void ld8(const float* p, float* f) {
  const f32x4 a = reinterpret_cast<const f32x4*>(p)[0], b = reinterpret_cast<const f32x4*>(p)[1];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    f[e] = a[e];
    f[4 + e] = b[e];
  }
}
__device__ __forceinline__ void st8(bf16_t* p, const float* f) { *reinterpret_cast<u32x4*>(p) = pack8(f); }
__device__ __forceinline__ void st8(float* p, const float* f) {
  reinterpret_cast<f32x4*>(p)[0] = (f32x4){f[0], f[1], f[2], f[3]};
  reinterpret_cast<f32x4*>(p)[1] = (f32x4){f[4], f[5], f[6], f[7]};
}

// sequence that packed token t belongs to: the last s with cu[s] <= t (cu has S + 1 entries, cu[0] = 0)
__device__ __forceinline__ int seq_of(const int* cu, int S, int t) {
  int lo = 0, hi = S - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (cu[mid] <= t) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// e^x for |x| <= 104 (infinite from 89 on): the exponent's whole part apart, so that the rest is rounded for its own size only
__device__ __forceinline__ float exp_near(float x) {
  const float n = __builtin_rintf(x * 1.44269502f);
  const float f = __builtin_fmaf(x, 1.92596299e-8f, __builtin_fmaf(x, 1.44269502f, -n));
  return __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f(f), (int)n);
}
// ln(1 + e^z) = max(z, 0) + ln(1 + e), e = e^-|z|; ln(1 + e) = 2 artanh(s), s = e / (2 + e) <= 1 / 3, with the quotient's and
// the sum's rounding carried on (s_lo) and artanh's series beyond s as a polynomial in s^2 (own minimax fit, 5e-9 of the value).
// Where both are of a size the sum's rounding is carried too. A quarter of the instructions of log1pf(expf(z)), which were 130 of
// the 560 vector instructions that a wave of the chunked scan issues a chunk (7917 tokens of 64 heads 152 -> 140 us, 5000 of 128
// 180 -> 163). Errors over [-30, 30]: rms 3.1e-8 or less and 1.29e-7 at most (before: 3.2e-8 and 1.29e-7).
__device__ __forceinline__ float softplusf(float z) {
  const float e = exp_near(-fminf(fabsf(z), 104.f)), d = 2.f + e, d_lo = e - (d - 2.f), r = __builtin_amdgcn_rcpf(d);
  const float s = e * r, s_lo = __builtin_fmaf(-d_lo, s, __builtin_fmaf(-d, s, e)) * r, w = s * s, s2 = s + s;
  float p = 0.140122294f;
  p = __builtin_fmaf(p, w, 0.139995709f);
  p = __builtin_fmaf(p, w, 0.200108498f);
  p = __builtin_fmaf(p, w, 0.333332062f);
  const float pos = z <= 0.f ? 0.f : z, sum = pos + s2, lo = (fmaxf(pos, s2) - sum) + fminf(pos, s2);
  return z > 30.f ? z : sum + (lo + __builtin_fmaf(s2 * w, p, s_lo + s_lo));
}
// z * sigmoid(z) as a quotient with one corrected step, the divisor's own rounding included; infinities and NaN as the quotient
// z / (1 + expf(-z)) gives them, which took twice the instructions (gate and norm of 7917 rows of 4096: 40.4 -> 35.7 us, now at
// the rate of its stream). The reciprocal is taken of a quarter: of a divisor past 2^126 (z under -87.33) its own would be
// subnormal, which the instruction flushes. Errors over [-30, 30]: rms 2.8e-8 to 3.8e-8 (before: 2.7e-8 to 4.4e-8).
__device__ __forceinline__ float silu_exact(float z) {
  const float e = exp_near(__builtin_amdgcn_fmed3f(-z, -104.f, 104.f)), d = 1.f + e, d_lo = e - (d - 1.f);
  const float r = 0.25f * __builtin_amdgcn_rcpf(0.25f * d), q = z * r;
  return __builtin_amdgcn_div_fixupf(__builtin_fmaf(__builtin_fmaf(-d_lo, q, __builtin_fmaf(-d, q, z)), r, q), d, z);
}

}  // namespace ragk
