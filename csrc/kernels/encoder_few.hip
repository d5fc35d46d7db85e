// A sentence encoder over one sequence of at most 32 rows (a question): four launches a layer instead of seven.
//
// A query of 14 tokens is 21 MB of weights (4 us) behind a chain of dependent launches of 2.4 to 4 us each, most of which is
// launch, first loads and the last store. Here every launch is a product whose blocks first make its input rows themselves:
//   qkv    rows = norm of the rows before (of the token embeddings in layer 0)
//   out    rows = attention of the qkv rows, all heads in every block
//   up     rows = norm
//   down   rows as they lie
// A block is 16 output columns: it requests its weights (and whatever else does not depend on the rows), then works on the rows
// while they travel, keeps the rows in LDS as bf16 and multiplies: 16 waves share the rows, then K, and meet in LDS. Repeating the
// rows' work in each of 24 to 256 blocks costs reads from L2 (21 KB a block for 14 fp32 rows of 384) and 0.6 us, the launch it
// saves 2.4 to 4. Sums of a product, its bias and its residual reach the norm behind it in fp32; block 0 writes the norm's rows
// out, as the residual of the product after next.
// Six layers of 384 columns, 14 rows: 220 us a call in seven launches a layer, 111 in these, 108.7 of it the chain on the device and
// 88 the host's launches beside 31 of checks (119 a call where the host is not ahead). With the rows' loads in front of the weights,
// column groups known when compiling, no spare K-steps and 64 bytes of arguments 96 and 68; 30 rows 142 -> 128; 24 layers of 1024, 14 rows 691 ->
// 630. A launch on the device is 1.4 us behind the one before, 1.3 to 2 for the rows' (or the down projection's operands') trip to
// memory and 1 through LDS for the sum. Past 16384 values of rows the repeated work costs more than it saves (ops/native.py
// encoder_few_ok).
#include "attn_tiles.h"
#include "encoder.h"
#include <type_traits>
using namespace ragk;

namespace {

constexpr int FEW_W = 16;  // waves

enum FewPro : int { ROWS, EMBED, NORM, ATTEND };  // (named: it is part of the kernels' names, which host and device have to agree on)

// 64 bytes: the host pays for a launch by the lines of its arguments (3.3 us for one, 3.8 from two on; one struct for all launches
// had 248 bytes), and 25 of them are what a call of six layers is on its side.
struct FewArgs {
  const void* x;          // ROWS: bf16 [T][K]; NORM: fp32 [T][K]; ATTEND: bf16 qkv [T][3 K]
  const bf16_t *w, *bias;  // [N][K], [N]
  void* out;              // ROWS and ATTEND: fp32 [T][N], else bf16
  const bf16_t *p, *q;    // ROWS and ATTEND: residual [T][N]; EMBED, NORM: gain and shift
  bf16_t* h;              // EMBED, NORM: the rows for the residual of the product after next
  unsigned sizes;         // T, K / 128, N / 16 in 6, 10 and 16 bits
  float f;                // ATTEND: scale in log2 units; EMBED, NORM: eps
  __host__ __device__ int T() const { return sizes & 63; }
  __host__ __device__ int K() const { return (sizes >> 6 & 1023) * 128; }
  __host__ __device__ int N() const { return (sizes >> 16) * 16; }
};
static_assert(sizeof(FewArgs) == 64, "one line of arguments");
struct EmbedArgs : FewArgs {
  const bf16_t *word, *places, *type;
  const int* ids_dev;  // token ids on the device, or (null) by value
  int ids[FEW_T];
  int first_pos;
};

// One row in a wave: lane l holds columns 2 l + 128 j and the one after, j < NJ = K / 128 (known when compiling: behind a branch a
// column group each, the first one's load was waited for before the others went out). norm.hip's formula and order of roundings.
template <int NJ>
__device__ __forceinline__ void few_norm(float (&v)[2 * NJ], float eps, const unsigned (&gr)[NJ], const unsigned (&br)[NJ],
                                         unsigned (&o)[NJ]) {
  constexpr int K = 128 * NJ;
  float s = 0.f, sq = 0.f;
#pragma unroll
  for (int j = 0; j < NJ; ++j) s += v[2 * j] + v[2 * j + 1];
  const float mean = wave_sum(s) / (float)K;
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const float d0 = v[2 * j] - mean, d1 = v[2 * j + 1] - mean;
    sq += d0 * d0 + d1 * d1;
  }
  const float inv = rsqrtf(wave_sum(sq) / (float)K + eps);
#pragma unroll
  for (int j = 0; j < NJ; ++j)
    o[j] = pk2bf((v[2 * j] - mean) * inv * __uint_as_float(gr[j] << 16) + __uint_as_float(br[j] << 16),
                 (v[2 * j + 1] - mean) * inv * __uint_as_float(gr[j] & 0xffff0000u) + __uint_as_float(br[j] & 0xffff0000u));
}

template <int NJ>
__device__ __forceinline__ void few_pairs(const bf16_t* p, int lane, unsigned (&r)[NJ]) {
#pragma unroll
  for (int j = 0; j < NJ; ++j) r[j] = *reinterpret_cast<const unsigned*>(p + 2 * lane + 128 * j);
}

template <int NJ>
__device__ __forceinline__ void few_row(const float* x, int row, int lane, float (&v)[2 * NJ]) {
  const float2* p = reinterpret_cast<const float2*>(x + (size_t)row * 128 * NJ) + lane;
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const float2 t = p[64 * j];
    v[2 * j] = t.x;
    v[2 * j + 1] = t.y;
  }
}
template <int NJ>
__device__ __forceinline__ void few_row(const EmbedArgs& a, int row, int lane, float (&v)[2 * NJ]) {
  constexpr int K = 128 * NJ;
  unsigned wv[NJ], pv[NJ], tv[NJ];
  few_pairs(a.word + (size_t)(a.ids_dev ? a.ids_dev[row] : a.ids[row]) * K, lane, wv);
  few_pairs(a.places + (size_t)(a.first_pos + row) * K, lane, pv);
  if (a.type) few_pairs(a.type, lane, tv);
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    v[2 * j] = __uint_as_float(wv[j] << 16) + __uint_as_float(pv[j] << 16);
    v[2 * j + 1] = __uint_as_float(wv[j] & 0xffff0000u) + __uint_as_float(pv[j] & 0xffff0000u);
    if (a.type) {
      v[2 * j] += __uint_as_float(tv[j] << 16);
      v[2 * j + 1] += __uint_as_float(tv[j] & 0xffff0000u);
    }
  }
}

// One head of all rows: operands as loaded, then softmax(q k^T) v into the LDS rows. Scores transposed as in attention.hip: a
// lane holds keys 16 kt + 4 fh + r of query 16 qt + fr; the values' fragment takes the keys in that order.
template <int MT, int D>
struct FewHead {
  bf16x8 q[MT][D / 32], k[MT][D / 32], v[D / 16];
  __device__ __forceinline__ void load(const bf16_t* qkv, int K, int T, int hd, int fr, int fh) {
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const bf16_t* p = qkv + (size_t)min(16 * t + fr, T - 1) * 3 * K + hd * D + 8 * fh;
#pragma unroll
      for (int s = 0; s < D / 32; ++s) {
        q[t][s] = *reinterpret_cast<const bf16x8*>(p + 32 * s);
        k[t][s] = *reinterpret_cast<const bf16x8*>(p + K + 32 * s);
      }
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const bf16_t* p = qkv + (size_t)min(16 * (j >> 2) + 4 * fh + (j & 3), T - 1) * 3 * K + 2 * K + hd * D + fr;
#pragma unroll
      for (int dt = 0; dt < D / 16; ++dt) v[dt][j] = j < 4 * MT ? (short)p[16 * dt] : (short)0;
    }
  }
  __device__ __forceinline__ void attend(char* rows, int rowb, int T, int hd, int fr, int fh, float c) {
#pragma unroll
    for (int qt = 0; qt < MT; ++qt) {
      f32x4 s[2];
      float mx = -INFINITY;
#pragma unroll
      for (int kt = 0; kt < MT; ++kt) {
        s[kt] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < D / 32; ++ks) s[kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k[kt][ks], q[qt][ks], s[kt], 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int key = 16 * kt + 4 * fh + r;
          if (key >= T) s[kt][r] = -INFINITY;
          mx = fmaxf(mx, s[kt][r]);
        }
      }
      mx = max_xor32(max_xor16(mx)) * c;
      const float m = mx == -INFINITY ? 0.f : mx;
      float l = 0.f;
      if (MT == 1) s[1] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kt = 0; kt < MT; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          s[kt][r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kt][r], c, -m));
          l += s[kt][r];
        }
      l += __shfl_xor(l, 16, 64);
      l += __shfl_xor(l, 32, 64);
      const float inv = l > 0.f ? 1.f / l : 0.f;
      const bf16x8 p = pack_p(s[0], s[1]);
#pragma unroll
      for (int dt = 0; dt < D / 16; ++dt) {
        f32x4 o = (f32x4){0.f, 0.f, 0.f, 0.f};
        o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v[dt], p, o, 0, 0, 0);
        *reinterpret_cast<uint2*>(rows + (16 * qt + fr) * rowb + (hd * D + 16 * dt + 4 * fh) * 2) =
            make_uint2(pk2bf(o[0] * inv, o[1] * inv), pk2bf(o[2] * inv, o[3] * inv));
      }
    }
  }
};

// MT = 16-row tiles; NP = K-steps of 32 that a wave requests at once (it takes every 16th). D: head size (ATTEND), K / 128 (EMBED, NORM).
template <int PRO, int EPI, int MT, int NP, int D>
__global__ __launch_bounds__(FEW_W * 64) void few_kernel(std::conditional_t<PRO == EMBED, EmbedArgs, FewArgs> a) {
  const int T = a.T(), K = PRO == EMBED || PRO == NORM ? 128 * D : a.K(), N = a.N();
  extern __shared__ __attribute__((aligned(16))) char smem[];
  f32x4(*red)[MT][64] = reinterpret_cast<f32x4(*)[MT][64]>(smem);  // [wave][tile][lane]
  char* rows = smem + FEW_W * MT * 1024;
  const int rowb = K * 2 + 16;  // rows 16 bytes apart in the banks
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int fr = lane & 15, fh = lane >> 4, n0 = blockIdx.x * 16, nk = K / 32;

  // ---- requests, the rows ahead of what waits for them: loads come back in order, and with the weights in front a row waited for
  // 20 KB of them (indices clamped, so that few requests stand behind a branch, where the compiler would wait for all)
  constexpr bool MAKES = PRO == EMBED || PRO == NORM;
  constexpr int NJ = MAKES ? D : 1;
  float v[MT][2 * NJ];
  unsigned gr[NJ], br[NJ];
  FewHead<MT, PRO == ATTEND ? D : 32> head;
  if constexpr (MAKES) {
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      if (i && wid + FEW_W * i >= T) break;
      const int row = min(wid + FEW_W * i, T - 1);
      if constexpr (PRO == EMBED) few_row<NJ>(a, row, lane, v[i]);
      else few_row<NJ>(reinterpret_cast<const float*>(a.x), row, lane, v[i]);
    }
    few_pairs(a.p, lane, gr);
    few_pairs(a.q, lane, br);
  }
  if constexpr (PRO == ATTEND) head.load(reinterpret_cast<const bf16_t*>(a.x), K, T, min(wid, K / D - 1), fr, fh);
  __builtin_amdgcn_sched_barrier(0);
  const bf16_t* wp = a.w + (size_t)(n0 + fr) * K + 8 * fh;
  bf16x8 wf[NP], xf[MT][NP];
  auto request = [&](int base) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int s = min(base + wid + FEW_W * i, nk - 1);
      wf[i] = *reinterpret_cast<const bf16x8*>(wp + 32 * s);
      if constexpr (PRO == ROWS) {
#pragma unroll
        for (int t = 0; t < MT; ++t)
          xf[t][i] = *reinterpret_cast<const bf16x8*>(reinterpret_cast<const bf16_t*>(a.x) + (size_t)min(16 * t + fr, T - 1) * K +
                                                      8 * fh + 32 * s);
      }
    }
  };
  request(0);
  const int orow = threadIdx.x >> 4, ocol = n0 + (threadIdx.x & 15);  // this thread's output
  const bool mine = orow < T && orow < 16 * MT;
  const bf16_t bias = a.bias[ocol];
  bf16_t resid = 0;
  if constexpr (EPI == EPI_BIAS_RESID) resid = a.p[(size_t)min(orow, T - 1) * N + ocol];
  __builtin_amdgcn_sched_barrier(0);

  // ---- the rows
  if constexpr (MAKES) {
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int row = wid + FEW_W * i;
      if (i && row >= T) break;  // (the first one's norm in front of a branch: 24 layers of 1024, 14 rows 636 -> 630)
      unsigned o[NJ];
      few_norm(v[i], a.f, gr, br, o);
      if (row < T) {
#pragma unroll
        for (int j = 0; j < NJ; ++j) *reinterpret_cast<unsigned*>(rows + row * rowb + 4 * lane + 256 * j) = o[j];
        if (blockIdx.x == 0)
#pragma unroll
          for (int j = 0; j < NJ; ++j) *reinterpret_cast<unsigned*>(a.h + (size_t)row * K + 2 * lane + 128 * j) = o[j];
      }
    }
  }
  if constexpr (PRO == ATTEND) {
    const int heads = K / D;
    for (int hd = wid; hd < heads; hd += FEW_W) {
      if (hd != wid) head.load(reinterpret_cast<const bf16_t*>(a.x), K, T, hd, fr, fh);
      head.attend(rows, rowb, T, hd, fr, fh, a.f);
    }
  }
  if constexpr (PRO != ROWS) __syncthreads();

  // ---- the product (rows past the last are whatever LDS held: their outputs are not stored)
  f32x4 acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
  for (int base = 0; base < nk; base += FEW_W * NP) {
    if (base) request(base);
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int s = base + wid + FEW_W * i;
      if (s < nk)
#pragma unroll
        for (int t = 0; t < MT; ++t) {
          bf16x8 x;
          if constexpr (PRO == ROWS) x = xf[t][i];
          else x = *reinterpret_cast<const bf16x8*>(rows + (16 * t + fr) * rowb + 64 * s + 16 * fh);
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, wf[i], acc[t], 0, 0, 0);
        }
    }
  }
#pragma unroll
  for (int t = 0; t < MT; ++t) red[wid][t][lane] = acc[t];
  __syncthreads();
  if (mine) {
    const int t = orow >> 4, ln = 16 * ((orow & 15) >> 2) + (threadIdx.x & 15), r = orow & 3;
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < FEW_W; ++w) v += red[w][t][ln][r];
    v += EPI == EPI_BIAS_RESID ? bf2f(bias) + bf2f(resid) : bf2f(bias);
    if constexpr (EPI == EPI_BIAS_GELU) v = gelu_erf(v);
    if constexpr (EPI == EPI_BIAS_RESID) reinterpret_cast<float*>(a.out)[(size_t)orow * N + ocol] = v;
    else reinterpret_cast<bf16_t*>(a.out)[(size_t)orow * N + ocol] = f2bf(v);
  }
}

template <int PRO, int EPI, int MT, int NP, int D>
int few_launch(const std::conditional_t<PRO == EMBED, EmbedArgs, FewArgs>& a, hipStream_t st) {
  const int lds = FEW_W * MT * 1024 + (PRO == ROWS ? 0 : 16 * MT * (a.K() * 2 + 16));
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&few_kernel<PRO, EPI, MT, NP, D>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize,
                                                     FEW_W * MT * 1024 + (PRO == ROWS ? 0 : 16 * MT * (FEW_H * 2 + 16)));
  if (attr != hipSuccess) return (int)attr;
  hipLaunchKernelGGL((few_kernel<PRO, EPI, MT, NP, D>), dim3(a.N() / 16), dim3(FEW_W * 64), lds, st, a);
  return (int)hipGetLastError();
}

template <int PRO, int EPI, int NP, int D>
int few_rows(const std::conditional_t<PRO == EMBED, EmbedArgs, FewArgs>& a, hipStream_t st) {
  return a.T() <= 16 ? few_launch<PRO, EPI, 1, NP, D>(a, st) : few_launch<PRO, EPI, 2, NP, D>(a, st);
}
// EMBED, NORM: rows of K = 128 NJ columns
template <int PRO, int EPI, int NJ = FEW_H / 128>
int few_made(const std::conditional_t<PRO == EMBED, EmbedArgs, FewArgs>& a, hipStream_t st) {
  if (a.K() == 128 * NJ) return few_rows<PRO, EPI, NJ <= 4 ? 1 : 2, NJ>(a, st);
  if constexpr (NJ > 1) return few_made<PRO, EPI, NJ - 1>(a, st);
  else return (int)hipErrorInvalidValue;
}
template <int EPI, int D>
int few_attend(const FewArgs& a, hipStream_t st) {
  if (a.K() > FEW_H) return (int)hipErrorInvalidValue;
  return a.K() <= 512 ? few_rows<ATTEND, EPI, 1, D>(a, st) : few_rows<ATTEND, EPI, 2, D>(a, st);
}
// As many K-steps at once as a wave has (of K = 1536 three): a spare one is the last again, and its loads take their time (with
// four, the chain of six such layers 101.1 us for 96.4 at 14 rows, 135.4 for 128.4 at 30).
template <int EPI>
int few_plain(const FewArgs& a, hipStream_t st) {
  switch ((a.K() + 511) / 512) {
    case 1: return few_rows<ROWS, EPI, 1, 1>(a, st);
    case 2: return few_rows<ROWS, EPI, 2, 1>(a, st);
    case 3: return few_rows<ROWS, EPI, 3, 1>(a, st);
    case 4: return few_rows<ROWS, EPI, 4, 1>(a, st);
    case 5: case 6: return few_rows<ROWS, EPI, 6, 1>(a, st);
    default: return few_rows<ROWS, EPI, 8, 1>(a, st);
  }
}

constexpr int POOL_W = 8;
// Norm of the rows, then the pooled row as encoder.hip has it (the norm's rows rounded to bf16). A wave takes every eighth row.
template <int NJ>
__global__ __launch_bounds__(POOL_W * 64) void few_pool_kernel(const float* __restrict__ y, const bf16_t* __restrict__ g,
                                                              const bf16_t* __restrict__ b, float* out, int T, float eps, int mode,
                                                              int normalize) {
  constexpr int H = 128 * NJ;
  __shared__ float part[POOL_W][H];
  __shared__ float red[POOL_W];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int first = mode == 2 ? T - 1 : 0, last = mode == 1 ? T : first + 1;
  unsigned gr[NJ], br[NJ];
  few_pairs(g, lane, gr);
  few_pairs(b, lane, br);
  float acc[2 * NJ];
#pragma unroll
  for (int e = 0; e < 2 * NJ; ++e) acc[e] = 0.f;
  constexpr int AT_ONCE = (FEW_T + POOL_W - 1) / POOL_W;  // a wave's rows, requested together
  float v[AT_ONCE][2 * NJ];
#pragma unroll
  for (int i = 0; i < AT_ONCE; ++i) few_row<NJ>(y, min(first + wid + POOL_W * i, last - 1), lane, v[i]);
#pragma unroll
  for (int i = 0; i < AT_ONCE; ++i) {
    if (first + wid + POOL_W * i >= last) continue;
    unsigned o[NJ];
    few_norm(v[i], eps, gr, br, o);
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      acc[2 * j] += __uint_as_float(o[j] << 16);
      acc[2 * j + 1] += __uint_as_float(o[j] & 0xffff0000u);
    }
  }
#pragma unroll
  for (int j = 0; j < NJ; ++j) *reinterpret_cast<float2*>(&part[wid][2 * lane + 128 * j]) = make_float2(acc[2 * j], acc[2 * j + 1]);
  __syncthreads();
  const float inv = mode == 1 ? 1.f / (float)T : 1.f;
  constexpr int NC = (H + POOL_W * 64 - 1) / (POOL_W * 64);
  float c[NC], ss = 0.f;
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const int col = threadIdx.x + POOL_W * 64 * i;
    c[i] = 0.f;
    if (col < H) {
#pragma unroll
      for (int w = 0; w < POOL_W; ++w) c[i] += part[w][col];
      c[i] *= inv;
      ss += c[i] * c[i];
    }
  }
  float scale = 1.f;
  if (normalize) {
    ss = block_sum(ss, red);
    scale = 1.f / fmaxf(sqrtf(ss), 1e-12f);  // torch.nn.functional.normalize eps
  }
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const int col = threadIdx.x + POOL_W * 64 * i;
    if (col < H) out[col] = c[i] * scale;
  }
}

template <int NJ = FEW_H / 128>
int few_pool(const EncoderCall& c, const bf16_t* g, const bf16_t* b, hipStream_t st) {
  if (c.H == 128 * NJ) {
    hipLaunchKernelGGL(few_pool_kernel<NJ>, dim3(1), dim3(POOL_W * 64), 0, st, c.y, g, b, c.out, c.T, c.eps, c.pooling, c.normalize);
    return (int)hipGetLastError();
  }
  if constexpr (NJ > 1) return few_pool<NJ - 1>(c, g, b, st);
  else return (int)hipErrorInvalidValue;
}

}  // namespace

namespace ragk {

// c.few: one sequence of T <= FEW_T rows, H <= FEW_H, head size 32 or 64 (checked again here).
int encoder_few_forward(const EncoderCall& c, hipStream_t st) {
  const int H = c.H, T = c.T, D = c.heads > 0 ? H / c.heads : 0, l1 = c.l1 ? c.l1 : c.n_layers;
  if (c.B != 1 || T < 1 || T > FEW_T || H > FEW_H || H % 128 || c.I % 128 || D * c.heads != H || (D != 32 && D != 64) ||
      c.l0 < 0 || l1 <= c.l0 || c.n_layers < l1 || c.I < 128 || c.I >= 128 * 1024 || (!c.ids && !c.ids_host))
    return (int)hipErrorInvalidValue;
  auto sizes = [&](int K, int N) { return (unsigned)T | (unsigned)(K / 128) << 6 | (unsigned)(N / 16) << 16; };
#define RAGK_TRY(x) \
  if (const int rc = (x)) return rc
  for (int l = c.l0; l < l1; ++l) {
    const void* const* w = c.layers + 12 * l;
    auto b16 = [&](int i) { return (const bf16_t*)w[i]; };
    const float scale = 1.4426950408889634f / sqrtf((float)D);
    // qkv
    if (l == 0) {
      EmbedArgs a{};
      static_cast<FewArgs&>(a) = FewArgs{nullptr, b16(0), b16(1), c.qkv, (const bf16_t*)c.ln_g, (const bf16_t*)c.ln_b, (bf16_t*)c.h,
                                         sizes(H, 3 * H), c.eps};
      a.word = (const bf16_t*)c.word, a.places = (const bf16_t*)c.pos_table, a.type = (const bf16_t*)c.type_row;
      a.ids_dev = c.ids, a.first_pos = c.first_pos;
      if (!c.ids) __builtin_memcpy(a.ids, c.ids_host, (size_t)T * 4);
      RAGK_TRY((few_made<EMBED, EPI_BIAS>(a, st)));
    } else {  // behind the norm that ends the layer before
      const FewArgs a{c.y, b16(0), b16(1), c.qkv, b16(-2), b16(-1), (bf16_t*)c.h, sizes(H, 3 * H), c.eps};
      RAGK_TRY((few_made<NORM, EPI_BIAS>(a, st)));
    }
    // attention and its projection
    const FewArgs out{c.qkv, b16(2), b16(3), c.y, (const bf16_t*)c.h, nullptr, nullptr, sizes(H, H), scale};
    RAGK_TRY(D == 32 ? (few_attend<EPI_BIAS_RESID, 32>(out, st)) : (few_attend<EPI_BIAS_RESID, 64>(out, st)));
    const FewArgs up{c.y, b16(6), b16(7), c.f, b16(4), b16(5), (bf16_t*)c.h, sizes(H, c.I), c.eps};
    RAGK_TRY((few_made<NORM, EPI_BIAS_GELU>(up, st)));
    const FewArgs down{c.f, b16(8), b16(9), c.y, (const bf16_t*)c.h, nullptr, nullptr, sizes(c.I, H), 0.f};
    RAGK_TRY(few_plain<EPI_BIAS_RESID>(down, st));
  }
#undef RAGK_TRY
  if (l1 < c.n_layers) return 0;
  const void* const* w = c.layers + 12 * (c.n_layers - 1);
  return few_pool(c, (const bf16_t*)w[10], (const bf16_t*)w[11], st);
}

}  // namespace ragk
