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
// Six layers of 384 columns, 14 rows: 220 -> 111 us a call, 25 launches of 4.4 instead of 44 (with eight waves a block, two rows a
// wave, 119); 24 layers of 1024, 14 rows: 752 -> 686 (726). What is left of a launch is its start, one trip to memory for the rows
// and one through LDS for the sum (a down projection alone, without rows to make, takes as long as the others). Past 16384 values
// of rows the repeated work costs more than it saves (ops/native.py encoder_few_ok).
#include "attn_tiles.h"
#include "encoder.h"
using namespace ragk;

namespace {

constexpr int FEW_W = 16;  // waves

enum { ROWS, EMBED, NORM, ATTEND };

struct FewArgs {
  const void* x;          // ROWS: bf16 [T][K]; NORM: fp32 [T][K]; ATTEND: bf16 qkv [T][3 K]
  const bf16_t *g, *b;    // EMBED, NORM: gain and shift
  bf16_t* h;              // ... and where the rows go (null: nowhere)
  const bf16_t *word, *places, *type;  // EMBED
  const int* ids_dev;     // token ids on the device, or (null) by value
  int ids[FEW_T];
  int first_pos;
  float scale_log2;       // ATTEND
  const bf16_t *w, *bias, *resid;  // [N][K], [N], ROWS and ATTEND: [T][N]
  void* out;              // ROWS and ATTEND: fp32 [T][N], else bf16
  int T, N, K;
  float eps;
};

// One row in a wave: lane l holds columns 2 l + 128 j and the one after. norm.hip's formula and order of roundings.
__device__ __forceinline__ void few_norm(float (&v)[16], int nj, int K, float eps, const unsigned (&gr)[8], const unsigned (&br)[8],
                                         unsigned (&o)[8]) {
  float s = 0.f, sq = 0.f;
#pragma unroll
  for (int j = 0; j < 8; ++j)
    if (j < nj) s += v[2 * j] + v[2 * j + 1];
  const float mean = wave_sum(s) / (float)K;
#pragma unroll
  for (int j = 0; j < 8; ++j)
    if (j < nj) {
      const float d0 = v[2 * j] - mean, d1 = v[2 * j + 1] - mean;
      sq += d0 * d0 + d1 * d1;
    }
  const float inv = rsqrtf(wave_sum(sq) / (float)K + eps);
#pragma unroll
  for (int j = 0; j < 8; ++j)
    if (j < nj)
      o[j] = pk2bf((v[2 * j] - mean) * inv * __uint_as_float(gr[j] << 16) + __uint_as_float(br[j] << 16),
                   (v[2 * j + 1] - mean) * inv * __uint_as_float(gr[j] & 0xffff0000u) + __uint_as_float(br[j] & 0xffff0000u));
}

__device__ __forceinline__ void few_pairs(const bf16_t* p, int lane, int nj, unsigned (&r)[8]) {
#pragma unroll
  for (int j = 0; j < 8; ++j)
    if (j < nj) r[j] = *reinterpret_cast<const unsigned*>(p + 2 * lane + 128 * j);
}

template <int PRO>
__device__ __forceinline__ void few_row(const FewArgs& a, int row, int lane, int nj, float (&v)[16]) {
  if constexpr (PRO == NORM) {
    const float2* p = reinterpret_cast<const float2*>(reinterpret_cast<const float*>(a.x) + (size_t)row * a.K) + lane;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (j < nj) {
        const float2 t = p[64 * j];
        v[2 * j] = t.x;
        v[2 * j + 1] = t.y;
      }
  } else {
    unsigned wv[8], pv[8], tv[8];
    few_pairs(a.word + (size_t)(a.ids_dev ? a.ids_dev[row] : a.ids[row]) * a.K, lane, nj, wv);
    few_pairs(a.places + (size_t)(a.first_pos + row) * a.K, lane, nj, pv);
    if (a.type) few_pairs(a.type, lane, nj, tv);
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (j < nj) {
        v[2 * j] = __uint_as_float(wv[j] << 16) + __uint_as_float(pv[j] << 16);
        v[2 * j + 1] = __uint_as_float(wv[j] & 0xffff0000u) + __uint_as_float(pv[j] & 0xffff0000u);
        if (a.type) {
          v[2 * j] += __uint_as_float(tv[j] << 16);
          v[2 * j + 1] += __uint_as_float(tv[j] & 0xffff0000u);
        }
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

// MT = 16-row tiles; NP = K-steps of 32 that a wave requests at once (it takes every 16th). D: head size (ATTEND).
template <int PRO, int EPI, int MT, int NP, int D>
__global__ __launch_bounds__(FEW_W * 64) void few_kernel(FewArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  f32x4(*red)[MT][64] = reinterpret_cast<f32x4(*)[MT][64]>(smem);  // [wave][tile][lane]
  char* rows = smem + FEW_W * MT * 1024;
  const int rowb = a.K * 2 + 16;  // rows 16 bytes apart in the banks
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int fr = lane & 15, fh = lane >> 4, n0 = blockIdx.x * 16, nk = a.K / 32;

  // ---- what does not depend on the rows
  const bf16_t* wp = a.w + (size_t)(n0 + fr) * a.K + 8 * fh;
  bf16x8 wf[NP], xf[MT][NP];
  auto request = [&](int base) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int s = base + wid + FEW_W * i;
      if (s < nk) wf[i] = *reinterpret_cast<const bf16x8*>(wp + 32 * s);
      if constexpr (PRO == ROWS) {
#pragma unroll
        for (int t = 0; t < MT; ++t)
          if (s < nk)
            xf[t][i] = *reinterpret_cast<const bf16x8*>(reinterpret_cast<const bf16_t*>(a.x) +
                                                        (size_t)min(16 * t + fr, a.T - 1) * a.K + 8 * fh + 32 * s);
      }
    }
  };
  request(0);
  const int orow = threadIdx.x >> 4, ocol = n0 + (threadIdx.x & 15);  // this thread's output
  const bool mine = orow < a.T && orow < 16 * MT;
  float add = bf2f(a.bias[ocol]);
  if constexpr (EPI == EPI_BIAS_RESID) {
    if (mine) add += bf2f(a.resid[(size_t)orow * a.N + ocol]);
  }

  // ---- the rows
  if constexpr (PRO == EMBED || PRO == NORM) {
    const int nj = a.K / 128;
    unsigned gr[8], br[8];
    few_pairs(a.g, lane, nj, gr);
    few_pairs(a.b, lane, nj, br);
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int row = wid + FEW_W * i;
      if (row < a.T) {
        float v[16];
        unsigned o[8];
        few_row<PRO>(a, row, lane, nj, v);
        few_norm(v, nj, a.K, a.eps, gr, br, o);
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (j < nj) {
            *reinterpret_cast<unsigned*>(rows + row * rowb + 4 * lane + 256 * j) = o[j];
            if (blockIdx.x == 0) *reinterpret_cast<unsigned*>(a.h + (size_t)row * a.K + 2 * lane + 128 * j) = o[j];
          }
      }
    }
  }
  if constexpr (PRO == ATTEND) {
    const bf16_t* qkv = reinterpret_cast<const bf16_t*>(a.x);
    const int heads = a.K / D;
    for (int hd = wid; hd < heads; hd += FEW_W) {
      FewHead<MT, D> head;
      head.load(qkv, a.K, a.T, hd, fr, fh);
      head.attend(rows, rowb, a.T, hd, fr, fh, a.scale_log2);
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
    v += add;
    if constexpr (EPI == EPI_BIAS_GELU) v = gelu_erf(v);
    if constexpr (EPI == EPI_BIAS_RESID) reinterpret_cast<float*>(a.out)[(size_t)orow * a.N + ocol] = v;
    else reinterpret_cast<bf16_t*>(a.out)[(size_t)orow * a.N + ocol] = f2bf(v);
  }
}

template <int PRO, int EPI, int MT, int NP, int D>
int few_launch(const FewArgs& a, hipStream_t st) {
  const int lds = FEW_W * MT * 1024 + (PRO == ROWS ? 0 : 16 * MT * (a.K * 2 + 16));
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&few_kernel<PRO, EPI, MT, NP, D>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize,
                                                     FEW_W * MT * 1024 + (PRO == ROWS ? 0 : 16 * MT * (FEW_H * 2 + 16)));
  if (attr != hipSuccess) return (int)attr;
  hipLaunchKernelGGL((few_kernel<PRO, EPI, MT, NP, D>), dim3(a.N / 16), dim3(FEW_W * 64), lds, st, a);
  return (int)hipGetLastError();
}

template <int PRO, int EPI, int D = 32>
int few_dispatch(const FewArgs& a, hipStream_t st) {
  if (a.T < 1 || a.T > FEW_T || a.K % 128 || a.K <= 0 || a.N % 16 || (PRO != ROWS && a.K > FEW_H)) return (int)hipErrorInvalidValue;
#define RAGK_FEW(NP) return a.T <= 16 ? few_launch<PRO, EPI, 1, NP, D>(a, st) : few_launch<PRO, EPI, 2, NP, D>(a, st)
  if (a.K <= 512) RAGK_FEW(1);
  if constexpr (PRO != ROWS) RAGK_FEW(2);
  if (a.K <= 1024) RAGK_FEW(2);
  if (a.K <= 2048) RAGK_FEW(4);
  RAGK_FEW(8);
#undef RAGK_FEW
}

constexpr int POOL_W = 8;
// Norm of the rows, then the pooled row as encoder.hip has it (the norm's rows rounded to bf16). A wave takes every eighth row.
__global__ __launch_bounds__(POOL_W * 64) void few_pool_kernel(const float* __restrict__ y, const bf16_t* __restrict__ g,
                                                              const bf16_t* __restrict__ b, float* out, int T, int H, float eps,
                                                              int mode, int normalize) {
  __shared__ float part[POOL_W][FEW_H];
  __shared__ float red[POOL_W];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nj = H / 128;
  const int first = mode == 2 ? T - 1 : 0, last = mode == 1 ? T : first + 1;
  unsigned gr[8], br[8];
  few_pairs(g, lane, nj, gr);
  few_pairs(b, lane, nj, br);
  float acc[16];
#pragma unroll
  for (int e = 0; e < 16; ++e) acc[e] = 0.f;
  FewArgs a{};
  a.x = y;
  a.K = H;
  for (int row = first + wid; row < last; row += POOL_W) {
    float v[16];
    unsigned o[8];
    few_row<NORM>(a, row, lane, nj, v);
    few_norm(v, nj, H, eps, gr, br, o);
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (j < nj) {
        acc[2 * j] += __uint_as_float(o[j] << 16);
        acc[2 * j + 1] += __uint_as_float(o[j] & 0xffff0000u);
      }
  }
#pragma unroll
  for (int j = 0; j < 8; ++j)
    if (j < nj) *reinterpret_cast<float2*>(&part[wid][2 * lane + 128 * j]) = make_float2(acc[2 * j], acc[2 * j + 1]);
  __syncthreads();
  const float inv = mode == 1 ? 1.f / (float)T : 1.f;
  float v[FEW_H / (POOL_W * 64)], ss = 0.f;
#pragma unroll
  for (int i = 0; i < FEW_H / (POOL_W * 64); ++i) {
    const int c = threadIdx.x + POOL_W * 64 * i;
    v[i] = 0.f;
    if (c < H) {
#pragma unroll
      for (int w = 0; w < POOL_W; ++w) v[i] += part[w][c];
      v[i] *= inv;
      ss += v[i] * v[i];
    }
  }
  float scale = 1.f;
  if (normalize) {
    ss = block_sum(ss, red);
    scale = 1.f / fmaxf(sqrtf(ss), 1e-12f);  // torch.nn.functional.normalize eps
  }
#pragma unroll
  for (int i = 0; i < FEW_H / (POOL_W * 64); ++i) {
    const int c = threadIdx.x + POOL_W * 64 * i;
    if (c < H) out[c] = v[i] * scale;
  }
}

}  // namespace

namespace ragk {

// c.few: one sequence of T <= FEW_T rows, H <= FEW_H, head size 32 or 64 (checked again here).
int encoder_few_forward(const EncoderCall& c, hipStream_t st) {
  const int H = c.H, T = c.T, D = c.heads > 0 ? H / c.heads : 0;
  if (c.B != 1 || T < 1 || T > FEW_T || H > FEW_H || H % 128 || c.I % 128 || D * c.heads != H || (D != 32 && D != 64) ||
      c.n_layers < 1 || (!c.ids && !c.ids_host))
    return (int)hipErrorInvalidValue;
#define RAGK_TRY(x) \
  if (const int rc = (x)) return rc
  for (int l = 0; l < c.n_layers; ++l) {
    const void* const* w = c.layers + 12 * l;
    auto b16 = [&](int i) { return (const bf16_t*)w[i]; };
    FewArgs a{};
    a.T = T, a.eps = c.eps, a.scale_log2 = 1.4426950408889634f / sqrtf((float)D);
    // qkv
    a.K = H, a.N = 3 * H, a.h = (bf16_t*)c.h, a.w = b16(0), a.bias = b16(1), a.out = c.qkv;
    if (l == 0) {
      a.g = (const bf16_t*)c.ln_g, a.b = (const bf16_t*)c.ln_b;
      a.word = (const bf16_t*)c.word, a.places = (const bf16_t*)c.pos_table, a.type = (const bf16_t*)c.type_row;
      a.ids_dev = c.ids, a.first_pos = c.first_pos;
      if (!c.ids) __builtin_memcpy(a.ids, c.ids_host, (size_t)T * 4);
      RAGK_TRY((few_dispatch<EMBED, EPI_BIAS>(a, st)));
    } else {
      a.x = c.y, a.g = b16(-2), a.b = b16(-1);  // the norm that ends the layer before
      RAGK_TRY((few_dispatch<NORM, EPI_BIAS>(a, st)));
    }
    // attention and its projection
    a.x = c.qkv, a.N = H, a.w = b16(2), a.bias = b16(3), a.resid = (const bf16_t*)c.h, a.out = c.y;
    RAGK_TRY(D == 32 ? (few_dispatch<ATTEND, EPI_BIAS_RESID, 32>(a, st)) : (few_dispatch<ATTEND, EPI_BIAS_RESID, 64>(a, st)));
    // up
    a.x = c.y, a.g = b16(4), a.b = b16(5), a.N = c.I, a.w = b16(6), a.bias = b16(7), a.out = c.f;
    RAGK_TRY((few_dispatch<NORM, EPI_BIAS_GELU>(a, st)));
    // down
    a.x = c.f, a.K = c.I, a.N = H, a.w = b16(8), a.bias = b16(9), a.out = c.y;
    RAGK_TRY((few_dispatch<ROWS, EPI_BIAS_RESID>(a, st)));
  }
#undef RAGK_TRY
  const void* const* w = c.layers + 12 * (c.n_layers - 1);
  hipLaunchKernelGGL(few_pool_kernel, dim3(1), dim3(POOL_W * 64), 0, st, c.y, (const bf16_t*)w[10], (const bf16_t*)w[11], c.out, T, H,
                     c.eps, c.pooling, c.normalize);
  return (int)hipGetLastError();
}

}  // namespace ragk
