// Attention with shaped scores over the paged cache (K pages [blocks][G][64][DK], V pages [blocks][G][64][DV]),
// or over packed key / value rows of the step (row_attn_*: keys of a sequence in consecutive rows):
//
//   s_ij = softcap * tanh(q_i . k_j * scale / softcap) + table[h][min(i - j, far)]
//   j visible to i:  j <= i  and  (window == 0 or i - j < window or j < keep)
//   out_i = gate_ih * sum_j exp(s_ij) v_j / (sink + sum_j exp(s_ij)),  sink in {0, 1}
//   gate_ih: none, one sigmoid per head, or one per head and value element
//
// Positions are the tokens' own in the sequence, so the kept first tokens enter with their true distances.
// Scores, softmax and the bias are fp32.
//
//  * kv_store     : k, and v mixed with the first mixing layer's values of the same token, into the pages.
//  * attn_rows    : one wave per (token, query head), plain fp32 arithmetic. Any head size; the fp32 path.
//  * attn_prefill : MFMA flash attention over 64-key pages, 4 waves = GB query heads of one KV head x (4 / GB)
//                   groups of 32 query rows. Only pages with a visible key are visited: the pages of the kept first
//                   tokens, then those of the window. The bias table row of each head sits in LDS.
//  * attn_decode  : one query per sequence. Takes the projection as fp32 split-K slabs, so the slab sum, the bias
//                   add, the value mix and the cache append need no launch of their own; the pages of a
//                   sequence are split over partitions (attn_merge joins them) when batch x KV heads is small.
//
// The MFMA kernels keep the softmax weights at 16 significant bits for P.V (bf16 high + low part, two products).
#include "attn_tiles.h"
#include "seq_common.h"
#include <type_traits>
using namespace ragk;

namespace {

struct ShapedArgs {
  const void* q; int ldq;      // projection rows; head h at h * DK, gates at off_g
  const void* kc; const void* vc;
  const int* block_tables; int bt_stride;
  const int* cu_q;             // [S + 1]; null: one token per sequence
  const int* kv_lens;          // [S]
  const float* table;          // [H][far + 1] or null
  void* out; int ldo;
  int T, S, H, G, DK, DV;
  int off_g;                   // column of the gates, -1: no gate
  int gate_vec;                // 1: a gate per head and value element, 0: one per head
  int window, keep, far, sink;
  float scale, softcap;
  // keys: entry e of a sequence's page list starts at kc + e * k_unit + kv head * k_head, rows k_row apart. Paged:
  // e = block table entry; packed rows: e = key_off[seq] + first position of the page.
  const int* key_off;          // [S] row of position 0 of each sequence (may be negative), null: paged
  long long k_unit, v_unit;
  int k_head, k_row, v_head, v_row;
  __device__ __forceinline__ int entry(const int* bt, int seq, int page) const {
    return key_off ? key_off[seq] + page * 64 : bt[page];
  }
};

template <typename T>
__global__ __launch_bounds__(256) void kv_store_kernel(const T* __restrict__ row, int ld, int off_k, int off_v, int G, int DK,
                                                       int DV, const int* __restrict__ slots, T* kc, T* vc,
                                                       const T* __restrict__ v_first, int ldf,
                                                       const float* __restrict__ lam) {
  const int t = blockIdx.x, slot = slots[t];
  if (slot < 0) return;
  const int blk = slot >> 6, off = slot & 63;
  const T* r = row + (size_t)t * ld;
  const int nk = G * DK / 8, nv = G * DV / 8;
  for (int i = threadIdx.x; i < nk + nv; i += 256) {
    float f[8];
    if (i < nk) {
      const int g = i / (DK / 8), c = (i % (DK / 8)) * 8;
      ld8(r + off_k + i * 8, f);
      st8(kc + (((size_t)blk * G + g) * 64 + off) * DK + c, f);
    } else {
      const int j = i - nk, g = j / (DV / 8), c = (j % (DV / 8)) * 8;
      ld8(r + off_v + j * 8, f);
      if (v_first != nullptr) {
        const float lm = lam[0];
        float w[8];
        ld8(v_first + (size_t)t * ldf + j * 8, w);
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = (1.f - lm) * f[e] + lm * w[e];
      }
      st8(vc + (((size_t)blk * G + g) * 64 + off) * DV + c, f);
    }
  }
}

// NC: value columns per lane, sizes up to 64 NC
template <typename T, int NC>
__global__ __launch_bounds__(64) void attn_rows_kernel(ShapedArgs a) {
  __shared__ float sq[64 * NC], sp[64];
  const int t = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
  const int s = a.cu_q ? seq_of(a.cu_q, a.S, t) : t;
  const int q0 = a.cu_q ? a.cu_q[s] : t, q1 = a.cu_q ? a.cu_q[s + 1] : t + 1;
  const int L = a.kv_lens[s], i = L - (q1 - q0) + (t - q0);
  const int g = h / (a.H / a.G);
  const T* qr = (const T*)a.q + (size_t)t * a.ldq;
  for (int d = lane; d < a.DK; d += 64) sq[d] = ld1(qr + h * a.DK + d);
  __syncthreads();
  const int* bt = a.block_tables + (size_t)s * a.bt_stride;
  const int n_pages = i / 64 + 1;
  const int keep_pages = a.window > 0 ? min(n_pages, (a.keep + 63) / 64) : n_pages;
  const int first_win = a.window > 0 ? max(keep_pages, max(0, i - a.window + 1) / 64) : n_pages;
  const int n_it = keep_pages + max(0, n_pages - first_win);
  float m = a.sink ? 0.f : -INFINITY, l = a.sink ? 1.f : 0.f;
  float acc[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) acc[c] = 0.f;
  for (int it = 0; it < n_it; ++it) {
    const int pg = it < keep_pages ? it : first_win + it - keep_pages;
    const int e0 = a.entry(bt, s, pg), j = pg * 64 + lane;
    const T* kr = (const T*)a.kc + e0 * a.k_unit + (size_t)g * a.k_head + (size_t)lane * a.k_row;
    const bool ok = j <= i && (a.window <= 0 || i - j < a.window || j < a.keep);
    float x = 0.f;
    if (ok) {
      for (int d = 0; d < a.DK; d += 8) {
        float f[8];
        ld8(kr + d, f);
#pragma unroll
        for (int e = 0; e < 8; ++e) x = fmaf(sq[d + e], f[e], x);
      }
      x *= a.scale;
      if (a.softcap > 0.f) x = a.softcap * tanhf(x / a.softcap);
      if (a.table) x += a.table[(size_t)h * (a.far + 1) + min(i - j, a.far)];
    } else {
      x = -INFINITY;
    }
    const float mn = fmaxf(m, wave_max(x));
    if (mn == -INFINITY) continue;  // nothing visible yet (uniform over the wave)
    const float alpha = expf(m - mn);
    const float p = expf(x - mn);
    m = mn;
    l = l * alpha + wave_sum(p);
    __syncthreads();
    sp[lane] = p;
    __syncthreads();
    const T* vb = (const T*)a.vc + e0 * a.v_unit + (size_t)g * a.v_head;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int d = lane + 64 * c;
      if (d < a.DV) {
        acc[c] *= alpha;
        const int nj = min(64, i + 1 - pg * 64);
        for (int k = 0; k < nj; ++k) acc[c] = fmaf(sp[k], ld1(vb + (size_t)k * a.v_row + d), acc[c]);
      }
    }
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
  float gate = 1.f;
  if (a.off_g >= 0 && !a.gate_vec) gate = 1.f / (1.f + expf(-ld1(qr + a.off_g + h)));
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int d = lane + 64 * c;
    if (d < a.DV && a.off_g >= 0 && a.gate_vec) gate = 1.f / (1.f + expf(-ld1(qr + a.off_g + h * a.DV + d)));
    if (d < a.DV) st1((T*)a.out + (size_t)t * a.ldo + h * a.DV + d, acc[c] * inv * gate);
  }
}

// ---- visited pages of a query range [qmin, qmax]: the kept first pages, then the window's ----
struct Pages {
  int n_keep, first, n;  // iteration it -> page it < n_keep ? it : first + it - n_keep
  __device__ __forceinline__ int page(int it) const { return it < n_keep ? it : first + it - n_keep; }
};
__device__ __forceinline__ Pages visited(int qmin, int qmax, int window, int keep) {
  const int n_pages = qmax / KT + 1;
  if (window <= 0) return Pages{n_pages, n_pages, n_pages};
  const int nk = min(n_pages, (keep + KT - 1) / KT);
  const int f = max(nk, max(0, qmin - window + 1) / KT);
  return Pages{nk, f, nk + max(0, n_pages - f)};
}

// softcapped score in log2 units: cap2 * tanh(x / cap) = cap2 - 2 cap2 / (1 + 2^(x * c1)); c1 = 2 scale log2e / cap
struct Shape {
  float c1, cap2, c;  // cap2 > 0: soft-capped; else s = x * c
  __device__ __forceinline__ float sigma(float x) const {  // 1 / (1 + 2^(x * c1))
    return __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(x * c1));
  }
};
// tanh(y) / y as a polynomial in y^2, |error of tanh| < 1.4e-7 for |y| <= TANH_R (least-maximum fit): cheaper than the
// exponential and the reciprocal, which on this ALU take four issue slots each
constexpr float TANH_R = 0.5f;
constexpr float TANH_C[4] = {0.999997676f, -0.333206551f, 0.131451449f, -0.0433724665f};

constexpr float LOG2E = 1.4426950408889634f;
__device__ __forceinline__ Shape make_shape(float scale, float softcap) {
  return Shape{softcap > 0.f ? 2.f * scale * LOG2E / softcap : 0.f, softcap > 0.f ? softcap * LOG2E : 0.f, scale * LOG2E};
}

struct ShapedPrefill {
  ShapedArgs a;
  const int* tiles; int n_hg, gb;  // work list (seq, first query); head groups; heads per block
  int sb_stride;                   // floats per head of the LDS bias table, 0: none
};

// PLAIN: no soft cap, bias, kept first tokens or zero score, and a positive scale: the maxima run over the raw products.
// BOUNDED: every score is known to stay within a range whose exponentials fp32 holds (soft cap + largest bias), so
// the sums need no running maximum: the weights are 2^s, and the extra zero score adds exactly 1.
enum PrefillMode { GENERAL, BOUNDED, PLAIN };
// Bound by the score arithmetic (vector unit) with the products behind it: 4 waves a block, a wave 32 queries of one head,
// 32x32x16 products of keys x queries. A lane pair holds one query, so its maximum, its rescale and its position arithmetic
// are one per lane, and a key fragment feeds twice the products of a 16x16x32 one. The values are read transposed at pair
// granularity (vswz32: with the 16-column swizzle half of those reads met in a bank, 64.1 against 61.9 us below). A block's
// end asks for all its output gates together. Before (16x16x32 products, gates one by one), now, a launch, us:
//   one gate a value, plain scores: 24 heads, 1777 tokens 70.0 -> 61.9, 2 x 700 29.6 -> 25.1, 300 17.6 -> 15.2
//   soft cap, bias, window, zero score: 5 x 1900 120.8 -> 113.2, 5000 334.9 -> 323.1, 3 x 400 25.3 -> 24.2
// Layouts as in attn_prefill_v3_kernel (attention.hip).
template <int DK, int DV, PrefillMode MODE>
__global__ __launch_bounds__(256, (DK <= 128 && DV <= 128) ? 2 : 1) void attn_shaped_prefill_kernel(ShapedPrefill pa) {
  using CK = Cfg<DK>;
  using CV = Cfg<DV>;
  constexpr int QS = DK / 16, DB = DV / 32;  // products over a key row, 32-wide blocks of a value row
  const ShapedArgs& a = pa.a;
  extern __shared__ __attribute__((aligned(16))) char smem[];  // [buf][K | V], page list, bias tables
  int* s_bt = reinterpret_cast<int*>(smem + 2 * (CK::TILEB + CV::TILEB));
  float* s_bias = reinterpret_cast<float*>(s_bt + MAX_BT);

  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int wid_u = __builtin_amdgcn_readfirstlane(wid);
  const int tix = (int)blockIdx.x / pa.n_hg, hg = (int)blockIdx.x - tix * pa.n_hg;
  const int seq = pa.tiles[2 * tix], q_start = pa.tiles[2 * tix + 1];
  const int G = a.H / a.G, gb = pa.gb, per_kv = G / gb;
  const int kvh = hg / per_kv, h0 = kvh * G + (hg % per_kv) * gb, hb = wid_u % gb, hq = h0 + hb;
  const int pbase = q_start + (wid_u / gb) * 32;
  const int q_off = a.cu_q[seq], q_len = a.cu_q[seq + 1] - q_off, kv_len = a.kv_lens[seq];
  const int ctx0 = kv_len - q_len;
  const int qt_rows = 32 * (4 / gb);
  const int keep = MODE == PLAIN ? 0 : a.keep, sink = MODE == PLAIN ? 0 : a.sink;
  const Pages pg = visited(ctx0 + q_start, ctx0 + min(q_start + qt_rows, q_len) - 1, a.window, keep);
  const int wave_pmin = ctx0 + pbase, wave_pmax = ctx0 + min(pbase + 31, q_len - 1);
  const int l32 = lane & 31, h = lane >> 5, i16 = lane & 15;  // this lane's query, half of the keys / columns
  const int qpos = ctx0 + pbase + l32, qi = pbase + l32;

  bf16x8 qf[QS];
  {
    const bf16_t* qp = (const bf16_t*)a.q + (size_t)(q_off + min(qi, q_len - 1)) * a.ldq + hq * DK + 8 * h;
#pragma unroll
    for (int s = 0; s < QS; ++s) qf[s] = *reinterpret_cast<const bf16x8*>(qp + 16 * s);
  }
  f32x16 o[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[db][e] = 0.f;
  // the extra zero score: running max 0, one unit in the sum (one of a query's two lanes holds it)
  float m_i = sink ? 0.f : -INFINITY, l_i = sink && h == 0 ? 1.f : 0.f;
  const int* bt = a.block_tables + (size_t)seq * a.bt_stride;
  for (int i = threadIdx.x; i < pg.n; i += 256) s_bt[i] = a.entry(bt, seq, pg.page(i));
  if (MODE != PLAIN && a.table && pa.sb_stride)
    for (int b = 0; b < gb; ++b)
      for (int i = threadIdx.x; i <= a.far; i += 256)
        s_bias[b * pa.sb_stride + i] = a.table[(size_t)(h0 + b) * (a.far + 1) + i] * LOG2E;
  __syncthreads();
  const float* tb = MODE != PLAIN && a.table ? a.table + (size_t)hq * (a.far + 1) : nullptr;
  const float* s_tb = s_bias + hb * pa.sb_stride;  // the same row in LDS, in log2 units
  const float far_bias = tb ? tb[a.far] * LOG2E : 0.f;
  const Shape shape = make_shape(a.scale, a.softcap);
  const bool capped = MODE != PLAIN && shape.cap2 > 0.f;
  const int win = a.window > 0 ? a.window : 0x7fffffff;
  // the polynomial in the raw product x: s = x (q0 + x^2 (q1 + ...)), good while |x| <= x_lim
  const float yx = capped ? a.scale / a.softcap : 0.f, yx2 = yx * yx, x_lim = capped ? TANH_R / yx : 0.f;
  const float q0 = shape.cap2 * yx * TANH_C[0], q1 = shape.cap2 * yx * yx2 * TANH_C[1];
  const float q2 = shape.cap2 * yx * yx2 * yx2 * TANH_C[2], q3 = shape.cap2 * yx * yx2 * yx2 * yx2 * TANH_C[3];

  // a page's rows by LDS-DMA, each wave a quarter of the 1-KiB pieces; per-lane source offsets are fixed
  constexpr int KP = CK::PIECES / 4, VP = CV::PIECES / 4;
  int koff[KP], voff[VP];
#pragma unroll
  for (int i = 0; i < KP; ++i) {
    const int row = (wid_u + 4 * i) * CK::RPP + lane / CK::NC, ph = lane % CK::NC;
    koff[i] = row * a.k_row * 2 + 16 * (ph ^ kswz<DK>(row));
  }
#pragma unroll
  for (int i = 0; i < VP; ++i) {
    const int row = (wid_u + 4 * i) * CV::RPP + lane / CV::NC, ph = lane % CV::NC;
    voff[i] = row * a.v_row * 2 + 16 * (ph ^ vswz32<DV>(row));
  }
  const unsigned lds0 = lds_addr(smem);
  auto stage = [&](int entry, int buf) {
    const int e0 = __builtin_amdgcn_readfirstlane(entry);
    const i32x4 srd_k = make_srd((const bf16_t*)a.kc + e0 * a.k_unit + kvh * a.k_head, (63 * a.k_row + DK) * 2);
    const i32x4 srd_v = make_srd((const bf16_t*)a.vc + e0 * a.v_unit + kvh * a.v_head, (63 * a.v_row + DV) * 2);
    const unsigned l = lds0 + buf * (CK::TILEB + CV::TILEB);
#pragma unroll
    for (int i = 0; i < KP; ++i) blds16_asm(srd_k, koff[i], 0, l + (wid_u + 4 * i) * 1024);
#pragma unroll
    for (int i = 0; i < VP; ++i) blds16_asm(srd_v, voff[i], 0, l + CK::TILEB + (wid_u + 4 * i) * 1024);
  };
  // fragment reads: the swizzles of key rows 32 kb + l32 and of value rows 16 ks + 4 h + .. do not depend on kb and ks
  int kat[QS], vat[DB][2];
#pragma unroll
  for (int s = 0; s < QS; ++s) kat[s] = l32 * CK::ROWB + 16 * ((2 * s + h) ^ kswz<DK>(l32));
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int r = 4 * h + (i16 >> 2) + 8 * u, chunk = 2 * (2 * db + ((lane >> 4) & 1)) + ((i16 >> 1) & 1);
      vat[db][u] = CK::TILEB + r * CV::ROWB + 16 * (chunk ^ vswz32<DV>(r)) + 8 * (i16 & 1);
    }
#pragma unroll
  for (int s = 0; s < QS; ++s) asm volatile("" : "+v"(qf[s]));  // waited for outside the loop
  stage(s_bt[0], 0);  // pg.n >= 1: a query always sees its own page
  wait_vmcnt0();
  __syncthreads();

  for (int it = 0; it < pg.n; ++it) {
    const int cur = it & 1, k0 = pg.page(it) * KT;
    const char* page = smem + cur * (CK::TILEB + CV::TILEB);
    const bool active = k0 <= wave_pmax && (wave_pmin - (k0 + KT - 1) < win || k0 < keep);
    const int next = s_bt[min(it + 1, pg.n - 1)];
    f32x16 s[2];
    if (active) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int e = 0; e < 16; ++e) s[kb][e] = 0.f;
#pragma unroll
      for (int ks = 0; ks < QS; ++ks)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
          const bf16x8 kf = *reinterpret_cast<const bf16x8*>(page + kat[ks] + kb * 32 * CK::ROWB);
          s[kb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[ks], s[kb], 0, 0, 0);
        }
    }
    if (it + 1 < pg.n) stage(next, cur ^ 1);  // DMA of the next page behind the QK^T products
    if (active) {
      const bool all_visible = k0 + KT - 1 <= wave_pmin && (wave_pmax - k0 < win || k0 + KT <= keep);
      const bool far_only = !tb || wave_pmin - (k0 + KT - 1) >= a.far;  // one bias for the whole page
      // scores in log2 units, with the page-wide bias; wave-uniform branches around whole pages of elements
      const float base = far_only ? far_bias : 0.f;
      const int d0 = qpos - k0 - 4 * h;  // distance of this lane's key 0; element e of block kb is key 32 kb + 8 (e / 4) + e % 4
#define RAGK_SCORES(kb, e)  _Pragma("unroll") for (int kb = 0; kb < 2; ++kb) _Pragma("unroll") for (int e = 0; e < 16; ++e)
      if (capped) {
        float ax = 0.f;
        RAGK_SCORES(kb, e) ax = fmaxf(ax, fabsf(s[kb][e]));
        if (!__builtin_amdgcn_ballot_w64(!(ax <= x_lim))) {
          RAGK_SCORES(kb, e) {
            const float x = s[kb][e], z = x * x;
            const float q = __builtin_fmaf(z, __builtin_fmaf(z, __builtin_fmaf(z, q3, q2), q1), q0);
            s[kb][e] = __builtin_fmaf(x, q, base);
          }
        } else {
          RAGK_SCORES(kb, e) s[kb][e] = __builtin_fmaf(-2.f * shape.cap2, shape.sigma(s[kb][e]), base + shape.cap2);
        }
      } else if constexpr (MODE != PLAIN) {
        RAGK_SCORES(kb, e) s[kb][e] = __builtin_fmaf(s[kb][e], shape.c, base);
      }
      if (!far_only) {
        if (pa.sb_stride) {
          RAGK_SCORES(kb, e) s[kb][e] += s_tb[max(0, min(d0 - 32 * kb - 8 * (e >> 2) - (e & 3), a.far))];
        } else {
          RAGK_SCORES(kb, e)
            s[kb][e] = __builtin_fmaf(tb[max(0, min(d0 - 32 * kb - 8 * (e >> 2) - (e & 3), a.far))], LOG2E, s[kb][e]);
        }
      }
      if (!all_visible) {
        RAGK_SCORES(kb, e) {
          const int d = d0 - 32 * kb - 8 * (e >> 2) - (e & 3);
          const bool ok = (d >= 0) & ((d < win) | (qpos - d < keep));
          s[kb][e] = ok ? s[kb][e] : -INFINITY;
        }
      }
      float ls[2] = {0.f, 0.f};
      if constexpr (MODE == BOUNDED) {
        RAGK_SCORES(kb, e) {
          s[kb][e] = __builtin_amdgcn_exp2f(s[kb][e]);
          ls[kb] += s[kb][e];
        }
        l_i += ls[0] + ls[1];
      } else {
        float mx = -INFINITY;
        RAGK_SCORES(kb, e) mx = fmaxf(mx, s[kb][e]);
        mx = max_xor32(mx);
        if constexpr (MODE == PLAIN) mx *= shape.c;
        float alpha = 1.f;
        if (mx > m_i + RESCALE_LOG2) {
          alpha = m_i == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_i - mx);
          m_i = mx;
        }
        const float mref = m_i == -INFINITY ? 0.f : m_i;
        RAGK_SCORES(kb, e) {
          s[kb][e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kb][e], MODE == PLAIN ? shape.c : 1.f, -mref));
          ls[kb] += s[kb][e];
        }
        l_i = l_i * alpha + (ls[0] + ls[1]);
        if (__builtin_amdgcn_ballot_w64(alpha != 1.f)) {
#pragma unroll
          for (int db = 0; db < DB; ++db) o[db] *= alpha;
        }
      }
#undef RAGK_SCORES
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {  // 16 keys: elements 8 (ks % 2) .. of block ks / 2, and the value rows in their order
        const int kb = ks >> 1, e0 = 8 * (ks & 1);
        bf16x8 hi, lo;
        split_p((f32x4){s[kb][e0], s[kb][e0 + 1], s[kb][e0 + 2], s[kb][e0 + 3]},
                (f32x4){s[kb][e0 + 4], s[kb][e0 + 5], s[kb][e0 + 6], s[kb][e0 + 7]}, hi, lo);
#pragma unroll
        for (int db = 0; db < DB; ++db) {
          const bf16x4 v0 = tr_read(page + vat[db][0] + ks * 16 * CV::ROWB), v1 = tr_read(page + vat[db][1] + ks * 16 * CV::ROWB);
          const bf16x8 vf = (bf16x8){v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
          o[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, hi, o[db], 0, 0, 0);
          o[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, lo, o[db], 0, 0, 0);
        }
      }
    }
    wait_vmcnt0();
    __syncthreads();
  }

  l_i += __shfl_xor(l_i, 32, 64);
  float inv = l_i > 0.f ? 1.f / l_i : 0.f;
  // element 4 b + r of block db is column 32 db + 8 b + 4 h + r
  const bf16_t* gq = (const bf16_t*)a.q + (size_t)(q_off + min(qi, q_len - 1)) * a.ldq + a.off_g;
  const bool gv = a.off_g >= 0 && a.gate_vec;
  bf16x4 gate[DB][4];
  if (gv) {  // all of them together: one by one, where they are used, each was a trip to memory, 16 at the end of a block
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int b = 0; b < 4; ++b) gate[db][b] = *reinterpret_cast<const bf16x4*>(gq + hq * DV + 32 * db + 8 * b + 4 * h);
  } else if (a.off_g >= 0) {
    inv *= __builtin_amdgcn_rcpf(1.f + __expf(-bf2f(gq[hq])));
  }
  if (qi >= q_len) return;
  bf16_t* op = (bf16_t*)a.out + (size_t)(q_off + qi) * a.ldo + hq * DV + 4 * h;
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      f32x4 v = (f32x4){o[db][4 * b], o[db][4 * b + 1], o[db][4 * b + 2], o[db][4 * b + 3]} * inv;
      if (gv) {
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] *= __builtin_amdgcn_rcpf(1.f + __expf(-bf2f_s(gate[db][b][r])));
      }
      *reinterpret_cast<uint2*>(op + 32 * db + 8 * b) = make_uint2(pk2bf(v[0], v[1]), pk2bf(v[2], v[3]));
    }
}

// ---- decode ----
struct ShapedDecode {
  const float* P; int S; int ldp; size_t slab;  // projection slabs [S][B][ldp]
  const bf16_t* bias;                            // [ldp] or null
  bf16_t* kc; bf16_t* vc;
  const int* block_tables; int bt_stride, bt_cols;
  const int* kv_lens; const int* slots;
  const float* table;
  const float* v_first; const float* lam;        // [B][G * DV] values to mix in, or null
  float* v_own;                                  // [B][G * DV] own values out, or null
  bf16_t* out; int ldo;
  float* part_o; float* part_ml;                 // [B][H][max_parts][DV], [B][H][max_parts][2]
  int B, H, G, off_k, off_v, off_g;
  int window, keep, far, sink, min_tiles, max_parts;
  float scale, softcap;
};

__device__ __forceinline__ float slab_gate(const ShapedDecode& a, int b, int h) {
  if (a.off_g < 0) return 1.f;
  float g = a.bias ? bf2f(a.bias[a.off_g + h]) : 0.f;
  const float* P = a.P + (size_t)b * a.ldp + a.off_g + h;
  for (int s0 = 0; s0 < a.S; s0 += PSU) {  // a round of loads, then their sum in order
    float p[PSU];
#pragma unroll
    for (int u = 0; u < PSU; ++u) p[u] = P[min(s0 + u, a.S - 1) * a.slab];
#pragma unroll
    for (int u = 0; u < PSU; ++u)
      if (s0 + u < a.S) g += p[u];
  }
  return __builtin_amdgcn_rcpf(1.f + __expf(-g));
}
static_assert(KT == DEC_TILE, "a page");
constexpr int DEC_UPT = KT / DEC_U;  // units of a page
// units that a new token at `pos` visits (the last page's second half may lie past it)
__device__ __forceinline__ int units(const Pages& pg, int pos) { return pg.n * DEC_UPT - (pos % KT < DEC_U ? 1 : 0); }
// units per partition: the visited ones spread over all partitions, at least min_tiles pages each
__device__ __forceinline__ int part_units(int n, const ShapedDecode& a) {
  return decode_share(n, a.min_tiles, a.max_parts);
}

constexpr int DEC_HEADS = 16;  // query heads per decode block (one MFMA column each)

// grid: (KV heads x groups of 16 query heads, batch, max_parts), 4 waves; a wave takes every 4th unit. What bounds it, its two trips
// to memory ahead of the stream, units of half a page and the next one behind the present one: as attn_decode_block (attention.hip).
// Us with the join, before and now: 17 rows of 2400 tokens, 32 heads over 8, 43.8 -> 40.3; 1 of 5000 14.6 -> 11.3; 25 of 4700 97.7
// -> 83.3 (5.9 TB/s); 16 heads over 4: 4 of 1000 14.9 -> 9.9, 20 of 2400 35.3 -> 22.9, 50 of 1250 39.8 -> 28.7.
template <int DK, int DV>
__global__ __launch_bounds__(256, (DK <= 128 && DV <= 128) ? 2 : 1) void attn_shaped_decode_kernel(ShapedDecode a) {
  using CK = Cfg<DK>;
  using CV = Cfg<DV>;
  constexpr int KB = DEC_U / 16, VPC = CV::PIECES / DEC_UPT;  // key blocks of a unit, 1-KiB pieces of its values
  constexpr int OS = DV + 4;                                   // floats between the combined rows
  constexpr int ROWS = DEC_HEADS * (OS + 2) * 4, PW = CV::TILEB / DEC_UPT > ROWS ? CV::TILEB / DEC_UPT : ROWS;  // LDS of a wave
  __shared__ __attribute__((aligned(16))) char smem[4 * PW + DEC_HEADS * DK * 2];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int wid_u = __builtin_amdgcn_readfirstlane(wid);
  const int part = blockIdx.z, b = blockIdx.y;
  const int Gq = a.H / a.G, chunks = (Gq + DEC_HEADS - 1) / DEC_HEADS;
  const int kvh = blockIdx.x / chunks, hc = blockIdx.x % chunks;
  const int h0 = kvh * Gq + hc * DEC_HEADS, nh = min(DEC_HEADS, Gq - hc * DEC_HEADS);
  PageRow<2> table(a.block_tables + (size_t)b * a.bt_stride, a.bt_cols, lane);
  const int pos = ld_uniform(a.kv_lens + b) - 1;
  const Pages pg = visited(pos, pos, a.window, a.keep);
  const int n = units(pg, pos), pt = part_units(n, a);
  const int it0 = part * pt;
  if (it0 >= n) return;  // block-uniform, before any barrier
  const int it1 = min(it0 + pt, n), nparts = (n + pt - 1) / pt;
  const int fr = lane & 15, fh = lane >> 4;
  table.wait();
  char* sV = smem + wid_u * PW;
  bf16_t* s_q = reinterpret_cast<bf16_t*>(smem + 4 * PW);

  bf16x8 kf[KB][CK::KS];
  u32x4 vr[VPC];
  constexpr int VP = CV::RPP < CV::RB * CV::GR ? CV::RB * CV::GR / CV::RPP : 1;  // pieces until the swizzle repeats
  const unsigned k_lane = (fr * DK + 8 * fh) * 2;
  unsigned v_lane[VP];
#pragma unroll
  for (int i = 0; i < VP; ++i)
    v_lane[i] = lane / CV::NC * CV::ROWB + 16 * ((lane % CV::NC) ^ vswz<DV>(i * CV::RPP + lane / CV::NC));
  auto first_key = [&](int it) {  // (row of the cache pages, all heads of a page behind each other)
    return ((size_t)table(pg.page(it / DEC_UPT)) * a.G + kvh) * KT + it % DEC_UPT * DEC_U;
  };
  auto request_k = [&](int it) {
    const char* kb = reinterpret_cast<const char*>(a.kc + first_key(it) * DK);
#pragma unroll
    for (int t = 0; t < KB; ++t)
#pragma unroll
      for (int s = 0; s < CK::KS; ++s) kf[t][s] = *reinterpret_cast<const bf16x8*>(kb + (16 * t * DK + 32 * s) * 2 + k_lane);
  };
  auto request_v = [&](int it) {
    const char* vb = reinterpret_cast<const char*>(a.vc + first_key(it) * DV);
#pragma unroll
    for (int i = 0; i < VPC; ++i) vr[i] = *reinterpret_cast<const u32x4*>(vb + i * 1024 + v_lane[i % VP]);
  };

  // Projection rows, four columns a thread: the heads' queries, then (in the block that takes the last unit) the new token's k and v
  const bool append = it1 == n;  // block-uniform
  const int n_q = nh * DK / 4, n_all = n_q + (append ? (DK + DV) / 4 : 0);
  f32x4 x[PSU], first;
  uint2 bias;
  auto column = [&](int i) {
    const int j = i - n_q;
    return j < 0 ? h0 * DK + 4 * i : j < DK / 4 ? a.off_k + kvh * DK + 4 * j : a.off_v + kvh * DV + 4 * min(j - DK / 4, DV / 4 - 1);
  };
  auto slab = [&](int i, int u) {
    return *reinterpret_cast<const f32x4*>(a.P + (size_t)u * a.slab + (size_t)b * a.ldp + column(i));
  };
  auto value = [&](int i) {  // place of a value item among the tokens' values
    return ((size_t)b * a.G + kvh) * DV + 4 * max(0, min(i - n_q - DK / 4, DV / 4 - 1));
  };
  const float lm = a.v_first ? a.lam[0] : 0.f;
  auto request_item = [&](int i) {
#pragma unroll
    for (int u = 0; u < PSU; ++u) x[u] = slab(i, min(u, a.S - 1));
    bias = a.bias ? *reinterpret_cast<const uint2*>(a.bias + column(i)) : make_uint2(0u, 0u);
    first = a.v_first ? *reinterpret_cast<const f32x4*>(a.v_first + value(i)) : (f32x4){0.f, 0.f, 0.f, 0.f};
  };
  auto finish_item = [&](int i) {
    f32x4 f = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < PSU; ++u)
      if (u < a.S) f += x[u];
    for (int u = PSU; u < a.S; ++u) f += slab(i, u);
    if (a.bias)
      f += (f32x4){__uint_as_float(bias.x << 16), __uint_as_float(bias.x & 0xffff0000u), __uint_as_float(bias.y << 16),
                   __uint_as_float(bias.y & 0xffff0000u)};
    const f32x4 own = f;
    if (a.v_first && i >= n_q + DK / 4) f = (1.f - lm) * f + lm * first;
    const uint2 r = make_uint2(pk2bf(f[0], f[1]), pk2bf(f[2], f[3]));
    asm volatile("" ::"v"(r.x), "v"(r.y), "v"(first));  // every load is used on every path
    if (i < n_q) {
      *reinterpret_cast<uint2*>(s_q + 4 * i) = r;
    } else if (i < n_all) {
      const int slot = ld_uniform(a.slots + b), j = i - n_q;
      const size_t row = ((size_t)(slot >> 6) * a.G + kvh) * KT + (slot & 63);
      if (j < DK / 4) {
        *reinterpret_cast<uint2*>(a.kc + row * DK + 4 * j) = r;
      } else {
        if (a.v_own) *reinterpret_cast<f32x4*>(a.v_own + value(i)) = own;
        *reinterpret_cast<uint2*>(a.vc + row * DV + 4 * (j - DK / 4)) = r;
      }
    }
  };
  const float* tb = a.table ? a.table + (size_t)(h0 + min(fr, nh - 1)) * (a.far + 1) : nullptr;
  const float far_bias = tb ? tb[a.far] * LOG2E : 0.f;
  // (requested whether the wave has a unit or not, and in this order: attn_decode_block)
  const int first_it = min(it0 + wid_u, it1 - 1);
  request_item(threadIdx.x);
  __builtin_amdgcn_sched_barrier(0);
  request_k(first_it);
  __builtin_amdgcn_sched_barrier(0);
  request_v(first_it);
  __builtin_amdgcn_sched_barrier(0);
  finish_item(threadIdx.x);
  for (int i0 = 256; i0 < n_all; i0 += 256) {  // block-uniform
    request_item(i0 + threadIdx.x);
    finish_item(i0 + threadIdx.x);
  }
  if (append) {
    __syncthreads();  // q in LDS; the appended row visible to the whole block
    if (it0 + wid_u == n - 1) {  // this wave's first unit is the one that was appended to
      request_k(first_it);
      __builtin_amdgcn_sched_barrier(0);
      request_v(first_it);
    }
  } else {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // no LDS access moves to either side
  }
  bf16x8 qf[CK::KS];
#pragma unroll
  for (int s = 0; s < CK::KS; ++s) {
    qf[s] = *reinterpret_cast<const bf16x8*>(s_q + min(fr, nh - 1) * DK + 32 * s + 8 * fh);
    if (fr >= nh) qf[s] = (bf16x8){0, 0, 0, 0, 0, 0, 0, 0};
  }

  const Shape shape = make_shape(a.scale, a.softcap);
  const bool capped = shape.cap2 > 0.f;
  const int win = a.window > 0 ? a.window : 0x7fffffff;
  f32x4 o[CV::DT];
#pragma unroll
  for (int dt = 0; dt < CV::DT; ++dt) o[dt] = (f32x4){0.f, 0.f, 0.f, 0.f};
  float m_i = -INFINITY, l_i = 0.f;
  auto unit = [&](int it, auto more_t) {
    constexpr bool MORE = decltype(more_t)::value;
    const int k0 = pg.page(it / DEC_UPT) * KT + it % DEC_UPT * DEC_U;
    f32x4 s4[KB];
#pragma unroll
    for (int t = 0; t < KB; ++t) {
      s4[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < CK::KS; ++s) s4[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[t][s], qf[s], s4[t], 0, 0, 0);
    }
    const int d0 = pos - k0 - 4 * fh;  // distance of this lane's key 0
    const bool far_only = !tb || pos - (k0 + DEC_U - 1) >= a.far;
    f32x4 near[KB];  // biases of keys nearer than the table's end (ahead of the next unit: loads return in order)
#pragma unroll
    for (int t = 0; t < KB; ++t) near[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
    if (!far_only) {
#pragma unroll
      for (int t = 0; t < KB; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) near[t][r] = tb[max(0, min(d0 - 16 * t - r, a.far))] * LOG2E;
#pragma unroll
      for (int t = 0; t < KB; ++t) asm volatile("" ::"v"(near[t]));
    }
    if constexpr (MORE) {
      __builtin_amdgcn_sched_barrier(0);
      request_k(it + 4);
      __builtin_amdgcn_sched_barrier(0);
    }
    const float base = (capped ? shape.cap2 : 0.f) + (far_only ? far_bias : 0.f);
    if (capped) {
#pragma unroll
      for (int t = 0; t < KB; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) s4[t][r] = __builtin_fmaf(-2.f * shape.cap2, shape.sigma(s4[t][r]), base);
    } else {
#pragma unroll
      for (int t = 0; t < KB; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) s4[t][r] = __builtin_fmaf(s4[t][r], shape.c, base);
    }
    if (!far_only) {
#pragma unroll
      for (int t = 0; t < KB; ++t) s4[t] += near[t];
    }
    if (!(k0 + DEC_U - 1 <= pos && (pos - k0 < win || k0 + DEC_U <= a.keep))) {
#pragma unroll
      for (int t = 0; t < KB; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int d = d0 - 16 * t - r;
          const bool ok = (d >= 0) & ((d < win) | (pos - d < a.keep));
          s4[t][r] = ok ? s4[t][r] : -INFINITY;
        }
    }
    float mx = -INFINITY;
#pragma unroll
    for (int t = 0; t < KB; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) mx = fmaxf(mx, s4[t][r]);
    mx = max_xor32(max_xor16(mx));
    const float m_new = fmaxf(m_i, mx), m_use = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = __builtin_amdgcn_exp2f(m_i - m_use);
    float ls = 0.f;
#pragma unroll
    for (int t = 0; t < KB; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float p = __builtin_amdgcn_exp2f(s4[t][r] - m_use);
        s4[t][r] = p;
        ls += p;
      }
    l_i = l_i * alpha + ls;
    m_i = m_new;
#pragma unroll
    for (int dt = 0; dt < CV::DT; ++dt) o[dt] *= alpha;
    bf16x8 hi, lo;
    split_p(s4[0], s4[1], hi, lo);
#pragma unroll
    for (int i = 0; i < VPC; ++i) *reinterpret_cast<u32x4*>(sV + i * 1024 + lane * 16) = vr[i];
    if constexpr (MORE) request_v(it + 4);
#pragma unroll
    for (int dt = 0; dt < CV::DT; ++dt) {
      const bf16x8 vf = load_vt<DV>(sV, dt, 0, lane);
      o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, hi, o[dt], 0, 0, 0);
      o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, lo, o[dt], 0, 0, 0);
    }
  };
  int it = it0 + wid_u;
  if (it < it1) {
    for (; it + 4 < it1; it += 4) unit(it, std::true_type{});
    unit(it, std::false_type{});
  }

  // combine the 4 waves: each puts its rows and their statistics where its values lay
  float* so = reinterpret_cast<float*>(smem);
  l_i += __shfl_xor(l_i, 16, 64);
  l_i += __shfl_xor(l_i, 32, 64);
  if (fr < nh) {
    float* w = so + wid_u * (PW / 4);
#pragma unroll
    for (int dt = 0; dt < CV::DT; ++dt) *reinterpret_cast<f32x4*>(w + fr * OS + 16 * dt + 4 * fh) = o[dt];
    if (fh == 0) *reinterpret_cast<float2*>(w + DEC_HEADS * OS + 2 * fr) = make_float2(m_i, l_i);
  }
  __syncthreads();
  for (int e = threadIdx.x; e < nh * (DV / 4); e += 256) {
    const int g = e / (DV / 4), d = e % (DV / 4) * 4, h = h0 + g;
    float2 ml[4];
    f32x4 ov[4];
    float M = nparts == 1 && a.sink ? 0.f : -INFINITY;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      ml[w] = *reinterpret_cast<const float2*>(so + w * (PW / 4) + DEC_HEADS * OS + 2 * g);
      ov[w] = *reinterpret_cast<const f32x4*>(so + w * (PW / 4) + g * OS + d);
      M = fmaxf(M, ml[w].x);
    }
    const float Mu = M == -INFINITY ? 0.f : M;
    float L = nparts == 1 && a.sink ? __builtin_amdgcn_exp2f(-Mu) : 0.f;
    f32x4 O = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float sc = __builtin_amdgcn_exp2f(ml[w].x - Mu);
      L += ml[w].y * sc;
      O += ov[w] * sc;
    }
    if (nparts == 1) {
      const float gate = slab_gate(a, b, h);
      if (!(L > 0.f)) O = (f32x4){0.f, 0.f, 0.f, 0.f}, L = 1.f;
      *reinterpret_cast<u32x2_a2*>(a.out + (size_t)b * a.ldo + h * DV + d) =
          (u32x2_a2){pk2bf(O[0] / L * gate, O[1] / L * gate), pk2bf(O[2] / L * gate, O[3] / L * gate)};
    } else {
      const size_t pi = ((size_t)b * a.H + h) * a.max_parts + part;
      *reinterpret_cast<f32x4_a4*>(a.part_o + pi * DV + d) = O;
      if (d == 0) *reinterpret_cast<f32x2_a4*>(a.part_ml + pi * 2) = (f32x2_a4){M, L};
    }
  }
}

// join the partitions of one (head, sequence), add the extra zero score, apply the gate; DV threads, at least a wave
__global__ void attn_shaped_merge_kernel(ShapedDecode a, int DV) {
  const int h = blockIdx.x, b = blockIdx.y, d = min((int)threadIdx.x, DV - 1);
  const size_t p0 = ((size_t)b * a.H + h) * a.max_parts;
  const float gate = slab_gate(a, b, h);
  int nparts = 0;
  const float2 r = join_parts(
      a.part_ml + p0 * 2, a.part_o + p0 * DV, DV, a.max_parts, d, a.sink,
      [&] {
        const int pos = a.kv_lens[b] - 1;
        const int n = units(visited(pos, pos, a.window, a.keep), pos), pt = part_units(n, a);
        return nparts = (n + pt - 1) / pt;
      },
      [](float x) { return __builtin_amdgcn_exp2f(x); });
  if (nparts == 1 || (int)threadIdx.x >= DV) return;  // one: written by the decode kernel
  a.out[(size_t)b * a.ldo + h * DV + d] = f2bf(r.y > 0.f ? r.x / r.y * gate : 0.f);
}

template <int DK, int DV, PrefillMode MODE>
int launch_prefill_mode(const ShapedPrefill& pa, int n_tiles, int lds, hipStream_t st) {
  (void)hipFuncSetAttribute((const void*)attn_shaped_prefill_kernel<DK, DV, MODE>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            lds);
  hipLaunchKernelGGL((attn_shaped_prefill_kernel<DK, DV, MODE>), dim3(n_tiles * pa.n_hg), dim3(256), lds, st, pa);
  return (int)hipGetLastError();
}
template <int DK, int DV>
int launch_prefill(ShapedPrefill pa, int n_tiles, int bounded, hipStream_t st) {
  constexpr int base = 2 * (Cfg<DK>::TILEB + Cfg<DV>::TILEB) + MAX_BT * 4;
  constexpr int room = ((DK <= 128 && DV <= 128) ? 80 * 1024 : 160 * 1024) - base;
  const ShapedArgs& a = pa.a;
  int extra = a.table ? pa.gb * (a.far + 1) * 4 : 0;
  if (extra > room) extra = 0;  // a very long table is read through the caches
  pa.sb_stride = extra ? a.far + 1 : 0;
  const int lds = base + (extra + 15) / 16 * 16;
  if (bounded) return launch_prefill_mode<DK, DV, BOUNDED>(pa, n_tiles, lds, st);
  if (!a.table && !a.keep && !a.sink && !(a.softcap > 0.f) && a.scale > 0.f)
    return launch_prefill_mode<DK, DV, PLAIN>(pa, n_tiles, lds, st);
  return launch_prefill_mode<DK, DV, GENERAL>(pa, n_tiles, lds, st);
}

template <int DK, int DV>
int launch_decode(const ShapedDecode& a, hipStream_t st) {
  const int chunks = (a.H / a.G + DEC_HEADS - 1) / DEC_HEADS;
  hipLaunchKernelGGL((attn_shaped_decode_kernel<DK, DV>), dim3(a.G * chunks, a.B, a.max_parts), dim3(256), 0, st, a);
  if (a.max_parts > 1)
    hipLaunchKernelGGL(attn_shaped_merge_kernel, dim3(a.H, a.B), dim3(DV < 64 ? 64 : DV), 0, st, a, DV);
  return (int)hipGetLastError();
}

#define RAGK_SHAPED_DISPATCH(FN, ...)                                  \
  do {                                                                 \
    if (DK == 32 && DV == 32) return FN<32, 32>(__VA_ARGS__);          \
    if (DK == 32 && DV == 64) return FN<32, 64>(__VA_ARGS__);          \
    if (DK == 32 && DV == 128) return FN<32, 128>(__VA_ARGS__);        \
    if (DK == 32 && DV == 256) return FN<32, 256>(__VA_ARGS__);        \
    if (DK == 64 && DV == 32) return FN<64, 32>(__VA_ARGS__);          \
    if (DK == 64 && DV == 64) return FN<64, 64>(__VA_ARGS__);          \
    if (DK == 64 && DV == 128) return FN<64, 128>(__VA_ARGS__);        \
    if (DK == 64 && DV == 256) return FN<64, 256>(__VA_ARGS__);        \
    if (DK == 128 && DV == 32) return FN<128, 32>(__VA_ARGS__);        \
    if (DK == 128 && DV == 64) return FN<128, 64>(__VA_ARGS__);        \
    if (DK == 128 && DV == 128) return FN<128, 128>(__VA_ARGS__);      \
    if (DK == 128 && DV == 256) return FN<128, 256>(__VA_ARGS__);      \
    if (DK == 256 && DV == 32) return FN<256, 32>(__VA_ARGS__);        \
    if (DK == 256 && DV == 64) return FN<256, 64>(__VA_ARGS__);        \
    if (DK == 256 && DV == 128) return FN<256, 128>(__VA_ARGS__);      \
    if (DK == 256 && DV == 256) return FN<256, 256>(__VA_ARGS__);      \
    return (int)hipErrorInvalidValue;                                  \
  } while (0)

}  // namespace

namespace {
ShapedArgs paged_args(const void* q, int ldq, const void* kc, const void* vc, const int* bt, int bt_stride, const int* cu_q,
                      const int* kv_lens, const float* table, void* out, int ldo, int T, int S, int H, int G, int DK,
                      int DV, int off_g, int window, int keep, int far, int sink, float scale, float softcap) {
  return ShapedArgs{q, ldq, kc, vc, bt, bt_stride, cu_q, kv_lens, table, out, ldo, T, S, H, G, DK, DV, off_g, 0, window,
                    keep, far, sink, scale, softcap, nullptr, (long long)G * 64 * DK, (long long)G * 64 * DV, 64 * DK, DK,
                    64 * DV, DV};
}
// packed rows [keys][ldk]: keys at column h * DK, values at off_v + h * DV; one gate per value element
ShapedArgs rows_args(const void* q, int ldq, const void* kv, int ldk, int off_v, size_t elem, const int* key_off,
                     const int* cu_q, const int* kv_lens, void* out, int ldo, int T, int S, int H, int DK, int DV, int off_g,
                     int window, float scale) {
  return ShapedArgs{q, ldq, kv, (const char*)kv + off_v * elem, nullptr, 0, cu_q, kv_lens, nullptr, out, ldo, T, S, H, H, DK,
                    DV, off_g, 1, window, 0, 0, 0, scale, 0.f, key_off, ldk, ldk, DK, ldk, DV, ldk};
}
template <typename T>
void launch_rows(const ShapedArgs& a, hipStream_t st) {
  if (a.DK <= 256 && a.DV <= 256) hipLaunchKernelGGL((attn_rows_kernel<T, 4>), dim3(a.T, a.H), dim3(64), 0, st, a);
  else hipLaunchKernelGGL((attn_rows_kernel<T, 16>), dim3(a.T, a.H), dim3(64), 0, st, a);
}
int dispatch_prefill(int DK, int DV, const ShapedPrefill& pa, int n_tiles, int bounded, hipStream_t st) {
  RAGK_SHAPED_DISPATCH(launch_prefill, pa, n_tiles, bounded, st);
}
}  // namespace

// bf16. tiles: [n_tiles][2] (sequence, first query) of 128 / gb query rows each; gb in {1, 2, 4} divides H / G.
// bounded: the caller knows that (softcap + largest |bias|) * log2e < 80 (every 2^score and the sum over any context fit).
RAGK_API int ragk_shaped_attn_prefill(const void* q, int ldq, const void* kc, const void* vc, const int* block_tables,
                                      int bt_stride, const int* cu_q, const int* kv_lens, const int* tiles, int n_tiles,
                                      int gb, const float* table, void* out, int ldo, int H, int G, int DK, int DV,
                                      int off_g, int window, int keep, int far, int sink, int bounded, float scale,
                                      float softcap, hipStream_t st) {
  if (n_tiles <= 0) return 0;
  if (H % G || (gb != 1 && gb != 2 && gb != 4) || (H / G) % gb || bt_stride > MAX_BT || ldq % 8 || ldo % 4 || !cu_q ||
      window < 0 || keep < 0 || far < 0 || (bounded && !(softcap > 0.f)))
    return (int)hipErrorInvalidValue;
  const ShapedArgs a = paged_args(q, ldq, kc, vc, block_tables, bt_stride, cu_q, kv_lens, table, out, ldo, 0, 0, H, G, DK,
                                  DV, off_g, window, keep, far, sink, scale, softcap);
  const ShapedPrefill pa{a, tiles, H / gb, gb, 0};
  return dispatch_prefill(DK, DV, pa, n_tiles, bounded, st);
}

// The same kernel over packed key / value rows kv [rows][ldk] (bf16): H heads of their own, position p of sequence s in
// row key_off[s] + p. Whole 64-row groups are read: every group that starts at a key must lie inside the rows.
RAGK_API int ragk_row_attn_prefill(const void* q, int ldq, const void* kv, int ldk, int off_v, const int* key_off,
                                   const int* cu_q, const int* kv_lens, const int* tiles, int n_tiles, void* out, int ldo,
                                   int H, int DK, int DV, int off_g, int window, int max_pages, float scale,
                                   hipStream_t st) {
  if (n_tiles <= 0) return 0;
  if (max_pages > MAX_BT || ldq % 8 || ldk % 8 || off_v % 8 || ldo % 4 || off_g % 4 || !cu_q || !key_off || window < 0 ||
      H < 1 || off_v < H * DK || off_v + H * DV > ldk)
    return (int)hipErrorInvalidValue;
  const ShapedPrefill pa{rows_args(q, ldq, kv, ldk, off_v, 2, key_off, cu_q, kv_lens, out, ldo, 0, 0, H, DK, DV, off_g,
                                   window, scale),
                         tiles, H, 1, 0};
  return dispatch_prefill(DK, DV, pa, n_tiles, 0, st);
}

// plain fp32 arithmetic over the same packed rows (fp32 when f32, else bf16); any head size up to 256
RAGK_API int ragk_row_attn_rows(const void* q, int ldq, const void* kv, int ldk, int off_v, const int* key_off,
                                const int* cu_q, const int* kv_lens, void* out, int ldo, int T, int S, int H, int DK,
                                int DV, int off_g, int window, float scale, int f32, hipStream_t st) {
  if (T <= 0) return 0;
  if (DK % 8 || DK > 256 || DV > 256 || H > 65535 || ldk % 8 || off_v % 8 || !cu_q || !key_off)
    return (int)hipErrorInvalidValue;
  const ShapedArgs a = rows_args(q, ldq, kv, ldk, off_v, f32 ? 4 : 2, key_off, cu_q, kv_lens, out, ldo, T, S, H, DK, DV,
                                 off_g, window, scale);
  if (f32) launch_rows<float>(a, st);
  else launch_rows<bf16_t>(a, st);
  return (int)hipGetLastError();
}

// bf16 caches, fp32 slabs P [S][B][ldp] (+ bias). The new token's k / v go to `slots`; out [B][ldo].
RAGK_API int ragk_shaped_attn_decode(const float* P, int S, int ldp, const void* bias, void* kc, void* vc,
                                     const int* block_tables, int bt_stride, int bt_cols, const int* kv_lens,
                                     const int* slots, const float* table, const float* v_first, const float* lam, float* v_own, void* out,
                                     int ldo, float* part_o, float* part_ml, int B, int H, int G, int DK, int DV,
                                     int off_k, int off_v, int off_g, int window, int keep, int far, int sink,
                                     int min_tiles, int max_parts, float scale, float softcap, hipStream_t st) {
  if (B <= 0) return 0;
  if (S < 1 || H % G || ldp % 8 || off_k % 8 || off_v % 8 || min_tiles < 1 || max_parts < 1 || (v_first && !lam) ||
      (max_parts > 1 && (!part_o || !part_ml)) || B > 65535 || window < 0 || keep < 0 || far < 0)
    return (int)hipErrorInvalidValue;
  const ShapedDecode a{P, S, ldp, (size_t)B * ldp, (const bf16_t*)bias, (bf16_t*)kc, (bf16_t*)vc, block_tables, bt_stride,
                       bt_cols, kv_lens, slots, table, v_first, lam, v_own, (bf16_t*)out, ldo, part_o, part_ml, B, H, G, off_k,
                       off_v, off_g, window, keep, far, sink, min_tiles, max_parts, scale, softcap};
  RAGK_SHAPED_DISPATCH(launch_decode, a, st);
}

// row: projection rows [T][ld] (fp32 when f32). v_first: [T][ldf] own values of the first mixing layer, or null.
RAGK_API int ragk_shaped_kv_store(const void* row, int ld, int off_k, int off_v, int T, int G, int DK, int DV,
                                  const int* slots, void* kc, void* vc, const void* v_first, int ldf, const float* lam,
                                  int f32, hipStream_t st) {
  if (T <= 0) return 0;
  if (DK % 8 || DV % 8 || ld % 8 || off_k % 8 || off_v % 8 || ldf % 8 || (v_first && !lam))
    return (int)hipErrorInvalidValue;
  if (f32)
    hipLaunchKernelGGL(kv_store_kernel<float>, dim3(T), dim3(256), 0, st, (const float*)row, ld, off_k, off_v, G, DK, DV,
                       slots, (float*)kc, (float*)vc, (const float*)v_first, ldf, lam);
  else
    hipLaunchKernelGGL(kv_store_kernel<bf16_t>, dim3(T), dim3(256), 0, st, (const bf16_t*)row, ld, off_k, off_v, G, DK, DV,
                       slots, (bf16_t*)kc, (bf16_t*)vc, (const bf16_t*)v_first, ldf, lam);
  return (int)hipGetLastError();
}

RAGK_API int ragk_shaped_attn_rows(const void* q, int ldq, const void* kc, const void* vc, const int* block_tables,
                                   int bt_stride, const int* cu_q, const int* kv_lens, const float* table, void* out,
                                   int ldo, int T, int S, int H, int G, int DK, int DV, int off_g, int window, int keep,
                                   int far, int sink, float scale, float softcap, int f32, hipStream_t st) {
  if (T <= 0) return 0;
  if (DK % 8 || DK > 1024 || DV > 1024 || H % G || H > 65535) return (int)hipErrorInvalidValue;
  const ShapedArgs a = paged_args(q, ldq, kc, vc, block_tables, bt_stride, cu_q, kv_lens, table, out, ldo, T, S, H, G, DK,
                                  DV, off_g, window, keep, far, sink, scale, softcap);
  if (f32) launch_rows<float>(a, st);
  else launch_rows<bf16_t>(a, st);
  return (int)hipGetLastError();
}
