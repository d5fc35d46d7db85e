// Memory-bound row kernels for gfx950: RMSNorm, LayerNorm, embedding gathers,
// fused RoPE + paged-KV write, standalone SiLU*up.
//
// All loads/stores are 16-byte vectors (8 x bf16) -- hipcc does not vectorise
// bf16 on its own. Rows map to blocks of 256 threads (4 waves); reductions are
// wave shuffles + one LDS exchange.
//
// Reference semantics reproduced here:
//   K1 embed_tokens gather, K2 LlamaRMSNorm (fp32 variance, cast back, *weight),
//   K4 llama3-scaled RoPE in rotate_half layout, K13 KV-cache append,
//   E1 BERT/XLM-R embeddings (+LayerNorm), E4/E6 post-LN LayerNorm.
#include <algorithm>
#include <type_traits>

#include "common.h"
using namespace ragk;

namespace {

constexpr int NT = 256;

// out = bf16( w * bf16( x * rsqrt(mean(x^2) + eps) ) )      (HF LlamaRMSNorm exactly)
// If resid != nullptr: x = bf16(x + resid) is computed first and written back to resid
// (fused residual add: resid holds the new residual stream).
__global__ __launch_bounds__(NT) void rmsnorm_kernel(const bf16_t* x, int ldx, bf16_t* resid, int ldr,
                                                     const bf16_t* __restrict__ w, bf16_t* out, int ldo,
                                                     int H, float eps, const int* __restrict__ rows) {
  __shared__ float red[NT / 64];
  const int row = blockIdx.x;
  const bf16_t* xr = x + (size_t)(rows ? rows[row] : row) * ldx;
  bf16_t* rr = resid ? resid + (size_t)row * ldr : nullptr;
  bf16_t* orow = out + (size_t)row * ldo;
  constexpr int MAXV = 4;  // up to 4 x 8 x 256 = 8192 columns held in registers
  float v[MAXV][8];
  const int nvec = H >> 3;
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const int vi = threadIdx.x + i * NT;
    if (vi < nvec) {
      unpack8(*reinterpret_cast<const u32x4*>(xr + vi * 8), v[i]);
      if (rr) {
        float r8[8];
        unpack8(*reinterpret_cast<const u32x4*>(rr + vi * 8), r8);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[i][e] = bf2f(f2bf(v[i][e] + r8[e]));
        *reinterpret_cast<u32x4*>(rr + vi * 8) = pack8(v[i]);
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) ss += v[i][e] * v[i][e];
    }
  }
  ss = block_sum(ss, red);
  const float inv = rsqrtf(ss / (float)H + eps);
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const int vi = threadIdx.x + i * NT;
    if (vi < nvec) {
      float wv[8], o[8];
      unpack8(*reinterpret_cast<const u32x4*>(w + vi * 8), wv);
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = wv[e] * bf2f(f2bf(v[i][e] * inv));
      *reinterpret_cast<u32x4*>(orow + vi * 8) = pack8(o);
    }
  }
}

// LayerNorm of a row held in registers (fp32 statistics, two passes): NV vectors of 8 columns a thread, W waves a row.
// Encoder rows are 384 to 1024 wide: with a block a row, 48 to 128 of 256 threads had columns, behind two block-wide
// reductions; one wave a row (up to 2048 columns) takes 11.1 us for 13762 x 1024 (before: 20.1) and 8.6 for 12805 x 384
// (17.1, launch included). Wider rows stay a block each: 3000 x 4096 takes 11.0 us so, 12.1 in one wave.
template <int W>
__device__ __forceinline__ float row_sum(float v) {
  if constexpr (W == 1) return wave_sum(v);
  __shared__ float red[W];
  return block_sum(v, red);
}
template <int NV, int W>
__device__ __forceinline__ void ln_row(float (&v)[NV][8], int nvec, int lane, const bf16_t* __restrict__ g,
                                       const bf16_t* __restrict__ b, bf16_t* orow, int H, float eps) {
  u32x4 gr[NV], br[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int vi = min(lane + 64 * W * i, nvec - 1);
    gr[i] = *reinterpret_cast<const u32x4*>(g + vi * 8);
    br[i] = *reinterpret_cast<const u32x4*>(b + vi * 8);
  }
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i)
    if (lane + 64 * W * i < nvec)
#pragma unroll
      for (int e = 0; e < 8; ++e) s += v[i][e];
  const float mean = row_sum<W>(s) / (float)H;
  float sq = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i)
    if (lane + 64 * W * i < nvec)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float d = v[i][e] - mean;
        sq += d * d;
      }
  const float inv = rsqrtf(row_sum<W>(sq) / (float)H + eps);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int vi = lane + 64 * W * i;
    if (vi < nvec) {
      float gv[8], bv[8], o[8];
      unpack8(gr[i], gv);
      unpack8(br[i], bv);
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = (v[i][e] - mean) * inv * gv[e] + bv[e];
      *reinterpret_cast<u32x4*>(orow + vi * 8) = pack8(o);
    }
  }
}

// y = LN(x [+ resid]) * g + b, 4 / W rows a block
template <int NV, int W>
__global__ __launch_bounds__(NT) void layernorm_kernel(const bf16_t* x, int ldx, const bf16_t* resid, int ldr,
                                                       const bf16_t* __restrict__ g, const bf16_t* __restrict__ b,
                                                       bf16_t* out, int ldo, int rows, int H, float eps) {
  const int lane = threadIdx.x & (64 * W - 1), row = blockIdx.x * (NT / 64 / W) + threadIdx.x / (64 * W);
  if (row >= rows) return;  // (whole rows: never part of a block that reduces together)
  const int nvec = H >> 3;
  u32x4 xv[NV], rv[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int vi = min(lane + 64 * W * i, nvec - 1);
    xv[i] = *reinterpret_cast<const u32x4*>(x + (size_t)row * ldx + vi * 8);
    if (resid) rv[i] = *reinterpret_cast<const u32x4*>(resid + (size_t)row * ldr + vi * 8);
  }
  float v[NV][8];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    unpack8(xv[i], v[i]);
    if (resid) {
      float r8[8];
      unpack8(rv[i], r8);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[i][e] += r8[e];
    }
  }
  ln_row<NV, W>(v, nvec, lane, g, b, out + (size_t)row * ldo, H, eps);
}

// y = LN(sum_s P[s] + bias + resid) * g + b from the fp32 split-K slabs P[s][rows][H] of the product that precedes the norm
// (slab S_stride floats apart), 4 / W rows a block: the sum that a reduction launch and its bf16 result would have carried.
template <int NV, int W>
__global__ __launch_bounds__(NT) void layernorm_slabs_kernel(const float* __restrict__ P, int S, size_t slab,
                                                             const bf16_t* __restrict__ bias, const bf16_t* resid, int ldr,
                                                             const bf16_t* __restrict__ g, const bf16_t* __restrict__ b,
                                                             bf16_t* out, int ldo, int rows, int H, float eps) {
  const int lane = threadIdx.x & (64 * W - 1), row = blockIdx.x * (NT / 64 / W) + threadIdx.x / (64 * W);
  if (row >= rows) return;
  const int nvec = H >> 3;
  float v[NV][8];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int vi = min(lane + 64 * W * i, nvec - 1);
    float r8[8], b8[8];
    unpack8(*reinterpret_cast<const u32x4*>(resid + (size_t)row * ldr + vi * 8), r8);
    unpack8(*reinterpret_cast<const u32x4*>(bias + vi * 8), b8);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[i][e] = 0.f;
    const float* p = P + (size_t)row * H + vi * 8;
    int s = 0;
    for (; s + 4 <= S; s += 4) {  // four slabs' loads in flight
      f32x4 t[4][2];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        t[u][0] = *reinterpret_cast<const f32x4*>(p + (s + u) * slab);
        t[u][1] = *reinterpret_cast<const f32x4*>(p + (s + u) * slab + 4);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int e = 0; e < 8; ++e) v[i][e] += t[u][e >> 2][e & 3];
    }
    for (; s < S; ++s)
#pragma unroll
      for (int e = 0; e < 8; ++e) v[i][e] += p[s * slab + e];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[i][e] += b8[e] + r8[e];
  }
  ln_row<NV, W>(v, nvec, lane, g, b, out + (size_t)row * ldo, H, eps);
}

// token embedding gather: out[t] = table[ids[t]]
// carry (optional, asynchronous decode): carry[t] >= 0 takes the token id from prev[carry[t]] (the
// previous decode step's sampled tokens, still on the device) instead of ids[t]; the resolved id is
// written back to ids[t] so the step's inputs stay self-describing.
// NORM: and xn[t] = rmsnorm(out[t]) * w as rmsnorm_kernel has it, from the row in registers: the first layer's input, a launch
// of its own before (four Llama layers 4096 wide, 11 sequences of 2500 tokens in fp8: 406.9 -> 404.3 us a step).
template <bool NORM>
__global__ __launch_bounds__(NT) void embed_kernel(int* __restrict__ ids, const bf16_t* __restrict__ table,
                                                   bf16_t* out, int H, int vocab, const int* __restrict__ carry,
                                                   const int* __restrict__ prev, const bf16_t* __restrict__ w, bf16_t* xn,
                                                   float eps) {
  const int t = blockIdx.x;
  int id = ids[t];
  if (carry != nullptr) {
    const int c = carry[t];
    if (c >= 0) {
      id = prev[c];
      __syncthreads();  // every lane has read ids[t] before lane 0 overwrites it
      if (threadIdx.x == 0) ids[t] = id;
    }
  }
  id = id < 0 ? 0 : (id >= vocab ? vocab - 1 : id);
  const u32x4* src = reinterpret_cast<const u32x4*>(table + (size_t)id * H);
  u32x4* dst = reinterpret_cast<u32x4*>(out + (size_t)t * H);
  if constexpr (!NORM) {
    for (int i = threadIdx.x; i < (H >> 3); i += NT) dst[i] = src[i];
  } else {
    __shared__ float red[NT / 64];
    constexpr int MAXV = 4;  // as rmsnorm_kernel
    u32x4 x[MAXV], g[MAXV];
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < MAXV; ++i) {
      const int vi = threadIdx.x + i * NT;
      if (vi < (H >> 3)) {
        x[i] = src[vi];
        g[i] = reinterpret_cast<const u32x4*>(w)[vi];
      }
    }
#pragma unroll
    for (int i = 0; i < MAXV; ++i) {
      const int vi = threadIdx.x + i * NT;
      if (vi < (H >> 3)) {
        dst[vi] = x[i];
        float v[8];
        unpack8(x[i], v);
#pragma unroll
        for (int e = 0; e < 8; ++e) ss += v[e] * v[e];
      }
    }
    ss = block_sum(ss, red);
    const float inv = rsqrtf(ss / (float)H + eps);
#pragma unroll
    for (int i = 0; i < MAXV; ++i) {
      const int vi = threadIdx.x + i * NT;
      if (vi < (H >> 3)) {
        float v[8], wv[8], o[8];
        unpack8(x[i], v);
        unpack8(g[i], wv);
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = wv[e] * bf2f(f2bf(v[e] * inv));
        reinterpret_cast<u32x4*>(xn + (size_t)t * H)[vi] = pack8(o);
      }
    }
  }
}

// BERT / XLM-R embeddings: LN(word[id] + pos[pos_id] + type[type_id]) (+ optional GPT-2 style no-LN), 4 / W rows a block
template <int NV, int W>
__global__ __launch_bounds__(NT) void embed_ln_kernel(const int* __restrict__ ids, const int* __restrict__ pos_ids,
                                                      const bf16_t* __restrict__ word, const bf16_t* __restrict__ pos,
                                                      const bf16_t* __restrict__ type, const bf16_t* __restrict__ g,
                                                      const bf16_t* __restrict__ b, bf16_t* out, int rows, int H, float eps,
                                                      int do_ln) {
  const int lane = threadIdx.x & (64 * W - 1), t = blockIdx.x * (NT / 64 / W) + threadIdx.x / (64 * W);
  if (t >= rows) return;
  const bf16_t* wr = word + (size_t)ids[t] * H;
  const bf16_t* pr = pos + (size_t)pos_ids[t] * H;
  const int nvec = H >> 3;
  u32x4 wv[NV], pv[NV], tv[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int vi = min(lane + 64 * W * i, nvec - 1);
    wv[i] = *reinterpret_cast<const u32x4*>(wr + vi * 8);
    pv[i] = *reinterpret_cast<const u32x4*>(pr + vi * 8);
    if (type) tv[i] = *reinterpret_cast<const u32x4*>(type + vi * 8);
  }
  float v[NV][8];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    float p[8];
    unpack8(wv[i], v[i]);
    unpack8(pv[i], p);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[i][e] += p[e];
    if (type) {
      unpack8(tv[i], p);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[i][e] += p[e];
    }
  }
  bf16_t* orow = out + (size_t)t * H;
  if (do_ln) return ln_row<NV, W>(v, nvec, lane, g, b, orow, H, eps);
#pragma unroll
  for (int i = 0; i < NV; ++i)
    if (lane + 64 * W * i < nvec) *reinterpret_cast<u32x4*>(orow + (lane + 64 * W * i) * 8) = pack8(v[i]);
}

// f(NV, W) as constants for a row of H <= 8192 columns
template <typename F>
hipError_t by_row(int H, F f) {
  using std::integral_constant;
  if (H <= 512) f(integral_constant<int, 1>{}, integral_constant<int, 1>{});
  else if (H <= 1024) f(integral_constant<int, 2>{}, integral_constant<int, 1>{});
  else if (H <= 2048) f(integral_constant<int, 4>{}, integral_constant<int, 1>{});
  // two vectors a thread, since one of its four would load again what another has (14000 x 3072
  // 38.4 -> 29.1 us, 2000 x 4096 10.0 -> 8.6)
  else if (H <= 4096) f(integral_constant<int, 2>{}, integral_constant<int, 4>{});
  else f(integral_constant<int, 4>{}, integral_constant<int, 4>{});
  return hipGetLastError();
}

// Fused RoPE (rotate_half layout, HF bf16 rounding replicated) + paged KV write.
// qkv row layout: [Hq*D | Hkv*D | Hkv*D]. q is rotated in place, k rotated and
// written to k_cache, v copied to v_cache. Cache layout [nblocks][Hkv][BS][D].
// cos/sin tables: [max_pos][D/2] fp32 holding bf16-rounded values.
// slot < 0 means "do not cache" (padding token).
__global__ __launch_bounds__(NT) void rope_kv_kernel(bf16_t* qkv, int ld, const int* __restrict__ positions,
                                                     const float* __restrict__ cos_t, const float* __restrict__ sin_t,
                                                     const int* __restrict__ slots, bf16_t* kc, bf16_t* vc, int Hq,
                                                     int Hkv, int D, int BS, int apply_rope) {
  const int t = blockIdx.x;
  const int pos = positions[t];
  const int slot = slots ? slots[t] : -1;
  bf16_t* row = qkv + (size_t)t * ld;
  const int half = D >> 1;
  const int vpr = half >> 3;  // 8-wide vectors per half head
  const float* ct = cos_t + (size_t)pos * half;
  const float* st = sin_t + (size_t)pos * half;
  const int nrot = (Hq + Hkv) * vpr;
  for (int i = threadIdx.x; i < nrot; i += NT) {
    const int h = i / vpr, v = i % vpr;
    bf16_t* hp = row + h * D;
    float x1[8], x2[8], o1[8], o2[8];
    unpack8(*reinterpret_cast<const u32x4*>(hp + v * 8), x1);
    unpack8(*reinterpret_cast<const u32x4*>(hp + half + v * 8), x2);
    if (apply_rope) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float c = ct[v * 8 + e], s = st[v * 8 + e];
        // q*cos + rotate_half(q)*sin, each op rounded to bf16 like torch bf16 math
        o1[e] = bf2f(f2bf(bf2f(f2bf(x1[e] * c)) + bf2f(f2bf(-x2[e] * s))));
        o2[e] = bf2f(f2bf(bf2f(f2bf(x2[e] * c)) + bf2f(f2bf(x1[e] * s))));
      }
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) { o1[e] = x1[e]; o2[e] = x2[e]; }
    }
    const u32x4 p1 = pack8(o1), p2 = pack8(o2);
    if (h < Hq) {
      *reinterpret_cast<u32x4*>(hp + v * 8) = p1;
      *reinterpret_cast<u32x4*>(hp + half + v * 8) = p2;
    } else if (slot >= 0) {
      const int kh = h - Hq;
      bf16_t* dst = kc + (((size_t)(slot / BS) * Hkv + kh) * BS + (slot % BS)) * D;
      *reinterpret_cast<u32x4*>(dst + v * 8) = p1;
      *reinterpret_cast<u32x4*>(dst + half + v * 8) = p2;
      // keep the rotated k in qkv too (encoder-style consumers / debugging)
      *reinterpret_cast<u32x4*>(hp + v * 8) = p1;
      *reinterpret_cast<u32x4*>(hp + half + v * 8) = p2;
    } else {
      *reinterpret_cast<u32x4*>(hp + v * 8) = p1;
      *reinterpret_cast<u32x4*>(hp + half + v * 8) = p2;
    }
  }
  if (slot >= 0) {
    const int vpd = D >> 3;
    for (int i = threadIdx.x; i < Hkv * vpd; i += NT) {
      const int kh = i / vpd, v = i % vpd;
      const bf16_t* src = row + (Hq + Hkv + kh) * D + v * 8;
      bf16_t* dst = vc + (((size_t)(slot / BS) * Hkv + kh) * BS + (slot % BS)) * D + v * 8;
      *reinterpret_cast<u32x4*>(dst) = *reinterpret_cast<const u32x4*>(src);
    }
  }
}

// out[t, j] = silu(x[t, j]) * x[t, I + j]   (unpacked [gate | up] rows)
__global__ __launch_bounds__(NT) void silu_mul_kernel(const bf16_t* x, int ldx, bf16_t* out, int ldo, int I) {
  const int t = blockIdx.x;
  for (int v = threadIdx.x; v < (I >> 3); v += NT) {
    float g[8], u[8], o[8];
    unpack8(*reinterpret_cast<const u32x4*>(x + (size_t)t * ldx + v * 8), g);
    unpack8(*reinterpret_cast<const u32x4*>(x + (size_t)t * ldx + I + v * 8), u);
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = silu(g[e]) * u[e];
    *reinterpret_cast<u32x4*>(out + (size_t)t * ldo + v * 8) = pack8(o);
  }
}

// gather rows: out[i] = x[idx[i]]   (last-token selection before lm_head)
__global__ __launch_bounds__(NT) void gather_rows_kernel(const bf16_t* x, int ldx, const int* __restrict__ idx,
                                                         bf16_t* out, int ldo, int H) {
  const int i = blockIdx.x;
  const bf16_t* src = x + (size_t)idx[i] * ldx;
  for (int v = threadIdx.x; v < (H >> 3); v += NT)
    *reinterpret_cast<u32x4*>(out + (size_t)i * ldo + v * 8) = *reinterpret_cast<const u32x4*>(src + v * 8);
}


// ---- consumers of the split-K decode GEMM (gemm_part.hip): they sum the S fp32 partial slabs
// P[S][M][ldp] while doing their own row work, so the reduction needs no extra launch.

// h = bf16(h + bf16(sum_s P[s][row]))  (HF: bf16 linear output, then the bf16 residual add), written
// back to h; out = rmsnorm(h) * w exactly as rmsnorm_kernel. One block of 512 threads per row.
// ROUNDED = false: h = bf16(h + sum_s P[s][row]), the rounding of a product whose epilogue adds the residual: where a prompt's
// step may take either form, the one with slabs loses nothing (300 rows, four Llama layers 4096 wide: error of the last values
// against 64 bits 7.11e-3 with the sum rounded first, 6.80e-3 without and 6.79e-3 from the epilogue).
// idx: only the rows idx[i], to out[i], and h stays as it is (behind a prompt's last layer nothing reads it): the norm of all 300 rows
// and a gather behind it before (with the launch saved in front: 300 tokens 856 -> 846 us, 2048 wide, bound by the host, 400 466 -> 449).
constexpr int PNT = 512;
template <bool ROUNDED>
__global__ __launch_bounds__(PNT) void add_partials_rmsnorm_kernel(const float* __restrict__ P, int S, int M,
                                                                   bf16_t* h, int ldh,
                                                                   const bf16_t* __restrict__ w, bf16_t* out,
                                                                   int ldo, int H, float eps, const int* __restrict__ idx) {
  __shared__ float red[PNT / 64];
  const int row = idx ? idx[blockIdx.x] : blockIdx.x;
  bf16_t* hr = h + (size_t)row * ldh;
  constexpr int MAXV = 2;  // up to 2 x 8 x 512 = 8192 columns in registers
  float v[MAXV][8];
  const int nvec = H >> 3;
  float ss = 0.f;
  // every independent load in flight together (one memory round trip, not three): the first PSU
  // slabs, the residual row and the norm weights
  f32x4 pv[MAXV][PSU][2];
  u32x4 hv[MAXV], gv[MAXV];
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const int vi = min((int)threadIdx.x + i * PNT, nvec - 1);
    if (i * PNT < nvec) {  // block-uniform
      load_slabs8(P + (size_t)row * H + vi * 8, S, (size_t)M * H, pv[i]);
      hv[i] = *reinterpret_cast<const u32x4*>(hr + vi * 8);
      gv[i] = *reinterpret_cast<const u32x4*>(w + vi * 8);
    }
  }
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const int vi = threadIdx.x + i * PNT;
    if (vi < nvec) {
      float a[8];
      add_slabs8(pv[i], P + (size_t)row * H + vi * 8, S, (size_t)M * H, a);
      unpack8(hv[i], v[i]);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[i][e] = bf2f(f2bf(v[i][e] + (ROUNDED ? bf2f(f2bf(a[e])) : a[e])));
      if (!idx) *reinterpret_cast<u32x4*>(hr + vi * 8) = pack8(v[i]);
#pragma unroll
      for (int e = 0; e < 8; ++e) ss += v[i][e] * v[i][e];
    }
  }
  ss = block_sum(ss, red);
  const float inv = rsqrtf(ss / (float)H + eps);
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const int vi = threadIdx.x + i * PNT;
    if (vi < nvec) {
      float wv[8], o[8];
      unpack8(gv[i], wv);
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = wv[e] * bf2f(f2bf(v[i][e] * inv));
      *reinterpret_cast<u32x4*>(out + (size_t)blockIdx.x * ldo + vi * 8) = pack8(o);
    }
  }
}

// rope_kv_kernel fed by qkv partial slabs: qkv = bf16(sum_s P[s][t]) (the bf16 linear output), then
// the same rotate_half RoPE (HF bf16 op rounding) and paged-KV write. Rotated q goes to q_out
// (row stride ldq); k / v go to the cache only. grid = (T, HG): head groups split over blocks.

__global__ __launch_bounds__(NT) void rope_kv_partials_kernel(const float* __restrict__ P, int S, int T, int ldp,
                                                              bf16_t* q_out, int ldq,
                                                              const int* __restrict__ positions,
                                                              const float* __restrict__ cos_t,
                                                              const float* __restrict__ sin_t,
                                                              const int* __restrict__ slots, bf16_t* kc, bf16_t* vc,
                                                              int Hq, int Hkv, int D, int BS) {
  const int t = blockIdx.x, hg = blockIdx.y, ngroups = gridDim.y;
  const int pos = positions[t];
  const int slot = slots ? slots[t] : -1;
  const size_t slab = (size_t)T * ldp;
  const float* prow = P + (size_t)t * ldp;
  const int half = D >> 1;
  const int vpr = half >> 3;
  const float* ct = cos_t + (size_t)pos * half;
  const float* st = sin_t + (size_t)pos * half;
  const int nh = Hq + 2 * Hkv;
  for (int i = threadIdx.x + hg * NT; i < nh * vpr; i += NT * ngroups) {
    const int hd = i / vpr, v = i % vpr;
    float x1[8], x2[8];
    sum_partials8(prow + hd * D + v * 8, S, slab, x1);
    sum_partials8(prow + hd * D + half + v * 8, S, slab, x2);
    if (hd >= Hq + Hkv) {  // v head: straight to the cache
      if (slot >= 0) {
        bf16_t* dst = vc + (((size_t)(slot / BS) * Hkv + (hd - Hq - Hkv)) * BS + (slot % BS)) * D;
        *reinterpret_cast<u32x4*>(dst + v * 8) = pack8(x1);
        *reinterpret_cast<u32x4*>(dst + half + v * 8) = pack8(x2);
      }
      continue;
    }
    float o1[8], o2[8];
    rope8(x1, x2, ct + v * 8, st + v * 8, o1, o2);
    if (hd < Hq) {
      bf16_t* qp = q_out + (size_t)t * ldq + hd * D;
      *reinterpret_cast<u32x4*>(qp + v * 8) = pack8(o1);
      *reinterpret_cast<u32x4*>(qp + half + v * 8) = pack8(o2);
    } else if (slot >= 0) {
      bf16_t* dst = kc + (((size_t)(slot / BS) * Hkv + (hd - Hq)) * BS + (slot % BS)) * D;
      *reinterpret_cast<u32x4*>(dst + v * 8) = pack8(o1);
      *reinterpret_cast<u32x4*>(dst + half + v * 8) = pack8(o2);
    }
  }
}

}  // namespace

RAGK_API int ragk_rmsnorm(const void* x, int ldx, void* resid, int ldr, const void* w, void* out, int ldo, int rows,
                          int H, float eps, hipStream_t st) {
  if (rows <= 0) return 0;
  if (H % 8 || H > 8 * NT * 4) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(rmsnorm_kernel, dim3(rows), dim3(NT), 0, st, (const bf16_t*)x, ldx, (bf16_t*)resid, ldr,
                     (const bf16_t*)w, (bf16_t*)out, ldo, H, eps, (const int*)nullptr);
  return (int)hipGetLastError();
}

// out[i] = rmsnorm(x[rows[i]]) * w
RAGK_API int ragk_rmsnorm_rows(const void* x, int ldx, const int* rows, const void* w, void* out, int ldo, int n, int H, float eps,
                               hipStream_t st) {
  if (n <= 0) return 0;
  if (H % 8 || H > 8 * NT * 4 || !rows) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(rmsnorm_kernel, dim3(n), dim3(NT), 0, st, (const bf16_t*)x, ldx, (bf16_t*)nullptr, 0, (const bf16_t*)w,
                     (bf16_t*)out, ldo, H, eps, rows);
  return (int)hipGetLastError();
}

RAGK_API int ragk_layernorm(const void* x, int ldx, const void* resid, int ldr, const void* g, const void* b,
                            void* out, int ldo, int rows, int H, float eps, hipStream_t st) {
  if (rows <= 0) return 0;
  if (H % 8 || H > 8 * NT * 4) return (int)hipErrorInvalidValue;
  return (int)by_row(H, [&](auto nv, auto w) {
    constexpr int R = NT / 64 / decltype(w)::value;
    hipLaunchKernelGGL((layernorm_kernel<decltype(nv)::value, decltype(w)::value>), dim3((rows + R - 1) / R), dim3(NT), 0, st,
                       (const bf16_t*)x, ldx, (const bf16_t*)resid, ldr, (const bf16_t*)g, (const bf16_t*)b, (bf16_t*)out, ldo,
                       rows, H, eps);
  });
}

// P: S slabs of rows x H floats, one after the other; bias [H]; resid bf16 rows.
RAGK_API int ragk_layernorm_slabs(const float* P, int S, const void* bias, const void* resid, int ldr, const void* g,
                                  const void* b, void* out, int ldo, int rows, int H, float eps, hipStream_t st) {
  if (rows <= 0) return 0;
  if (H % 8 || H > 8 * NT * 4 || S < 1) return (int)hipErrorInvalidValue;
  return (int)by_row(H, [&](auto nv, auto w) {
    constexpr int R = NT / 64 / decltype(w)::value;
    hipLaunchKernelGGL((layernorm_slabs_kernel<decltype(nv)::value, decltype(w)::value>), dim3((rows + R - 1) / R), dim3(NT), 0,
                       st, P, S, (size_t)rows * H, (const bf16_t*)bias, (const bf16_t*)resid, ldr, (const bf16_t*)g,
                       (const bf16_t*)b, (bf16_t*)out, ldo, rows, H, eps);
  });
}

RAGK_API int ragk_embed(const int* ids, const void* table, void* out, int T, int H, int vocab, hipStream_t st) {
  if (T <= 0) return 0;
  if (H % 8) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(embed_kernel<false>, dim3(T), dim3(NT), 0, st, const_cast<int*>(ids), (const bf16_t*)table,
                     (bf16_t*)out, H, vocab, (const int*)nullptr, (const int*)nullptr, (const bf16_t*)nullptr, (bf16_t*)nullptr, 0.f);
  return (int)hipGetLastError();
}

// Embedding gather whose token ids may come from the previous step's device-side sampler output:
// carry[t] >= 0 -> id = prev[carry[t]] (also stored to ids[t]); carry[t] < 0 -> ids[t].
RAGK_API int ragk_embed_carry(int* ids, const int* carry, const int* prev, const void* table, void* out, int T,
                              int H, int vocab, hipStream_t st) {
  if (T <= 0) return 0;
  if (H % 8 || !carry || !prev) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(embed_kernel<false>, dim3(T), dim3(NT), 0, st, ids, (const bf16_t*)table, (bf16_t*)out, H, vocab,
                     carry, prev, (const bf16_t*)nullptr, (bf16_t*)nullptr, 0.f);
  return (int)hipGetLastError();
}

// Both (carry null: ids as they are), and xn = rmsnorm(out) * w.
RAGK_API int ragk_embed_rmsnorm(int* ids, const int* carry, const int* prev, const void* table, void* out, const void* w, void* xn,
                                int T, int H, int vocab, float eps, hipStream_t st) {
  if (T <= 0) return 0;
  if (H % 8 || H > 8 * NT * 4 || (carry && !prev) || !w || !xn) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(embed_kernel<true>, dim3(T), dim3(NT), 0, st, ids, (const bf16_t*)table, (bf16_t*)out, H, vocab, carry, prev,
                     (const bf16_t*)w, (bf16_t*)xn, eps);
  return (int)hipGetLastError();
}

RAGK_API int ragk_embed_ln(const int* ids, const int* pos_ids, const void* word, const void* pos, const void* type,
                           const void* g, const void* b, void* out, int T, int H, float eps, int do_ln,
                           hipStream_t st) {
  if (T <= 0) return 0;
  if (H % 8 || H > 8 * NT * 4) return (int)hipErrorInvalidValue;
  return (int)by_row(H, [&](auto nv, auto w) {
    constexpr int R = NT / 64 / decltype(w)::value;
    hipLaunchKernelGGL((embed_ln_kernel<decltype(nv)::value, decltype(w)::value>), dim3((T + R - 1) / R), dim3(NT), 0, st, ids,
                       pos_ids, (const bf16_t*)word, (const bf16_t*)pos, (const bf16_t*)type, (const bf16_t*)g,
                       (const bf16_t*)b, (bf16_t*)out, T, H, eps, do_ln);
  });
}

RAGK_API int ragk_rope_kv(void* qkv, int ld, const int* positions, const float* cos_t, const float* sin_t,
                          const int* slots, void* kc, void* vc, int T, int Hq, int Hkv, int D, int BS,
                          int apply_rope, hipStream_t st) {
  if (T <= 0) return 0;
  if (D % 16) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(rope_kv_kernel, dim3(T), dim3(NT), 0, st, (bf16_t*)qkv, ld, positions, cos_t, sin_t, slots,
                     (bf16_t*)kc, (bf16_t*)vc, Hq, Hkv, D, BS, apply_rope);
  return (int)hipGetLastError();
}

RAGK_API int ragk_silu_mul(const void* x, int ldx, void* out, int ldo, int T, int I, hipStream_t st) {
  if (T <= 0) return 0;
  if (I % 8) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(silu_mul_kernel, dim3(T), dim3(NT), 0, st, (const bf16_t*)x, ldx, (bf16_t*)out, ldo, I);
  return (int)hipGetLastError();
}

RAGK_API int ragk_gather_rows(const void* x, int ldx, const int* idx, void* out, int ldo, int n, int H,
                              hipStream_t st) {
  if (n <= 0) return 0;
  if (H % 8) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(gather_rows_kernel, dim3(n), dim3(NT), 0, st, (const bf16_t*)x, ldx, idx, (bf16_t*)out, ldo, H);
  return (int)hipGetLastError();
}

// idx null: all M rows, n = M. A selection without rows has no address either, so that one alone does not say which of the two is meant.
RAGK_API int ragk_add_partials_rmsnorm(const float* P, int S, int M, void* h, int ldh, const void* w, void* out,
                                       int ldo, int H, float eps, int rounded, const int* idx, int n, hipStream_t st) {
  if (!idx && n != M) return (int)hipErrorInvalidValue;
  if (M <= 0 || n <= 0) return 0;
  if (H % 8 || H > 8 * PNT * 2 || S < 1) return (int)hipErrorInvalidValue;
  const auto kernel = rounded ? add_partials_rmsnorm_kernel<true> : add_partials_rmsnorm_kernel<false>;
  hipLaunchKernelGGL(kernel, dim3(idx ? n : M), dim3(PNT), 0, st, P, S, M, (bf16_t*)h, ldh, (const bf16_t*)w, (bf16_t*)out, ldo, H,
                     eps, idx);
  return (int)hipGetLastError();
}

// P: [S][T][ldp] fp32 qkv partials (ldp >= (Hq + 2 Hkv) * D); q_out: rotated q [T][ldq] bf16.
RAGK_API int ragk_rope_kv_partials(const float* P, int S, int T, int ldp, void* q_out, int ldq,
                                   const int* positions, const float* cos_t, const float* sin_t, const int* slots,
                                   void* kc, void* vc, int Hq, int Hkv, int D, int BS, hipStream_t st) {
  if (T <= 0) return 0;
  if (D % 16 || S < 1) return (int)hipErrorInvalidValue;
  // head groups per row: enough blocks to spread the slab reads over the CUs at decode batch sizes,
  // at least one wave of (head, 8-column) items per block
  const int items = (Hq + 2 * Hkv) * (D / 16);
  const int groups = std::max(1, std::min((items + 63) / 64, std::max(4, (512 + T - 1) / T)));
  hipLaunchKernelGGL(rope_kv_partials_kernel, dim3(T, groups), dim3(NT), 0, st, P, S, T, ldp, (bf16_t*)q_out,
                     ldq, positions, cos_t, sin_t, slots, (bf16_t*)kc, (bf16_t*)vc, Hq, Hkv, D, BS);
  return (int)hipGetLastError();
}
