// Flash attention for gfx950 (MFMA 16x16x32 bf16, 64-key tiles, online softmax).
//
// Layout trick ("swapped" products, so no P transpose is ever needed):
//   S^T = K . Q^T   A = K rows from LDS (ds_read_b128, XOR swizzled), B = Q^T
//                   fragments held in VGPRs. C-layout: col = query (lane&15),
//                   row = key (4*(lane>>4)+r)  -> the softmax over keys of one
//                   query is lane-local + 2 shuffles (xor 16, 32).
//   O^T = V^T . P^T A = V^T read with ds_read_b64_tr_b16 (hardware transpose) from
//                   a row-major LDS V tile, B = P^T taken directly from the S^T
//                   accumulators of the same lane (k-slot order permuted to match).
//
// Kernels
//  * attn_prefill<D, GB, CAUSAL, PAGED>: varlen packed queries. PAGED reads K/V
//    from the paged cache [nblocks][Hkv][64][D] through block tables (prefill with
//    any prior context: chunked prefill / prefix reuse); !PAGED reads K/V straight
//    from a packed qkv buffer (bidirectional encoders). One block = 4 waves =
//    GB query heads sharing one KV head x (4/GB) groups of 32 query rows.
//  * attn_decode<D, G>: one query token per sequence, split-K over the context
//    (flash-decoding). Each wave streams its own 32-key units, the next one
//    requested behind the present one (K to VGPRs, V through VGPRs into a
//    wave-private LDS tile for the transposed read); 4 waves combine in LDS;
//    partitions merged by attn_decode_reduce.
//
// Replaces reference ops K5/K6 (causal GQA attention in transformers' Llama SDPA path,
// [dep] modeling_llama.py:191-215) and E3 (XLM-R/BERT bidirectional attention).
#include "attn_tiles.h"
#include <type_traits>
using namespace ragk;

namespace {

// ------------------------------------------------------------------------------------
// Prefill / encoder attention
// ------------------------------------------------------------------------------------
struct PrefillArgs {
  const bf16_t* q;  int q_stride;          // token row stride (elements); head h at +h*D
  const bf16_t* k;  const bf16_t* v;       // PAGED: caches; else packed K/V base pointers
  int kv_stride;                           // !PAGED: token row stride of k/v
  const int* block_tables; int bt_stride;  // PAGED
  const int* cu_q;                         // [S+1] query token offsets
  const int* cu_kv;                        // [S+1] kv token offsets (!PAGED)
  const int* kv_lens;                      // [S] total context length per sequence
  const int* tiles;                        // [n][2] = (seq, q_start)
  bf16_t* out; int out_stride;
  int Hq, Hkv;
  float scale_log2;
  unsigned kv_bytes;                       // PAGED: bytes of one cache (K or V) if < 4 GiB, else 0
  int n_hg;                                // > 0: 1-D grid of n_tiles x n_hg, head group fastest
};

// Prefill block -> (tile index, head group). 1-D grid, head group fastest (n_hg > 0, the default): the
// workgroups dispatch in the tile list's order -- heaviest causal tiles first -- across EVERY head (a 2-D
// grid dispatches head 0's whole list before head 1's, so the last heads' longest tiles start late and
// set the tail), and the round-robin XCD placement of consecutive workgroups keeps each head group on
// one XCD when n_hg is a multiple of 8 (its K/V tiles are re-read from that XCD's L2 by every query tile).
__device__ inline void prefill_block(const PrefillArgs& a, int& tile, int& hg) {
  if (a.n_hg > 0) {
    tile = (int)blockIdx.x / a.n_hg;
    hg = (int)blockIdx.x - tile * a.n_hg;
  } else {
    tile = blockIdx.x;
    hg = blockIdx.y;
  }
}

__device__ unsigned long long* g_attn_dbg = nullptr;  // stamp build only

// PRIO: wave priority around the MFMA clusters (0 none, 1 QK^T and PV, 2 PV only). Two waves share
// each SIMD (2 blocks per CU); raising the priority of the wave that is issuing MFMAs lets the
// other wave's softmax VALU fill around them instead of delaying them.
// BUF (PAGED only, cache < 4 GiB): K/V tiles staged by buffer_load ... lds with the per-lane byte
// offsets (row, swizzled chunk) computed once and the tile's cache offset in an SGPR, instead of
// 64-bit address math per piece per tile (the stamp build put the DMA issue at ~490 of ~4300 wave
// cycles per tile).
template <int D, int GB, bool CAUSAL, bool PAGED, bool STAMP = false, int NWV = 4, int PRIO = 0,
          bool BUF = false>
__global__ __launch_bounds__(NWV * 64, 8 / NWV) void attn_prefill_kernel(PrefillArgs a) {
  unsigned long long stp[6] = {0, 0, 0, 0, 0, 0};
  using C = Cfg<D>;
  constexpr int NTH = NWV * 64;
  constexpr int QT = 32 * (NWV / GB);  // query positions per block
  __shared__ __attribute__((aligned(16))) char smem[4 * C::TILEB];  // [buf][K|V]

  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int wid_u = __builtin_amdgcn_readfirstlane(wid);
  int tix, hg;
  prefill_block(a, tix, hg);
  const int seq = a.tiles[2 * tix], q_start = a.tiles[2 * tix + 1];
  const int G = a.Hq / a.Hkv;
  const int groups_per_kv = G / GB;
  const int kvh = hg / groups_per_kv;
  const int gsub = hg % groups_per_kv;
  const int hq = kvh * G + gsub * GB + (wid % GB);
  const int pbase = q_start + (wid / GB) * 32;

  const int q_off = a.cu_q[seq];
  const int q_len = a.cu_q[seq + 1] - q_off;
  const int kv_len = a.kv_lens[seq];
  const int ctx0 = kv_len - q_len;  // absolute position of query 0

  const int blk_qmax = min(q_start + QT, q_len) - 1;
  const int n_keys = CAUSAL ? min(kv_len, ctx0 + blk_qmax + 1) : kv_len;
  const int n_kt = (n_keys + KT - 1) / KT;
  const int wave_qmax = min(pbase + 31, q_len - 1);
  const int wave_pmax = ctx0 + wave_qmax;

  const int fr = lane & 15, fh = lane >> 4;

  // Q^T fragments (B operand), 2 query sub-tiles of 16
  bf16x8 qf[2][C::KS];
#pragma unroll
  for (int qt = 0; qt < 2; ++qt) {
    int qi = pbase + 16 * qt + fr;
    qi = qi < q_len ? qi : q_len - 1;
    const bf16_t* qp = a.q + (size_t)(q_off + qi) * a.q_stride + hq * D + 8 * fh;
#pragma unroll
    for (int s = 0; s < C::KS; ++s) qf[qt][s] = *reinterpret_cast<const bf16x8*>(qp + 32 * s);
  }

  f32x4 o[C::DT][2];
#pragma unroll
  for (int dt = 0; dt < C::DT; ++dt)
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) o[dt][qt] = (f32x4){0.f, 0.f, 0.f, 0.f};
  float m_i[2] = {-INFINITY, -INFINITY}, l_i[2] = {0.f, 0.f};

  const int kv_off = PAGED ? 0 : a.cu_kv[seq];
  const int* bt = PAGED ? a.block_tables + (size_t)seq * a.bt_stride : nullptr;

  // the sequence's block-table row, cached in LDS once (a global load per tile sat on the DMA
  // issue path: ~1.2k of ~5.7k wave cycles per tile in the stamp build, tools/attn_stamps.py)
  __shared__ int s_bt[PAGED ? MAX_BT : 1];
  if constexpr (PAGED) {
    for (int i = threadIdx.x; i < n_kt; i += NTH) s_bt[i] = bt[i];
    __syncthreads();
  }
  int bt_next = PAGED && n_kt > 0 ? s_bt[0] : 0;  // block of the tile staged next

  static_assert(!BUF || (PAGED && C::PIECES % NWV == 0), "buffer staging: paged caches, whole pieces per wave");
  constexpr int BPW = BUF ? C::PIECES / NWV : 1;
  int koff[BPW], voff[BPW];
  i32x4 srd_k, srd_v;
  if constexpr (BUF) {
#pragma unroll
    for (int i = 0; i < BPW; ++i) {
      const int p = wid_u + NWV * i;
      const int row = p * C::RPP + lane / C::NC, ph = lane % C::NC;
      koff[i] = row * C::ROWB + 16 * (ph ^ kswz<D>(row));
      voff[i] = row * C::ROWB + 16 * (ph ^ vswz<D>(row));
    }
    srd_k = make_srd(a.k, a.kv_bytes);
    srd_v = make_srd(a.v, a.kv_bytes);
  }
  auto stage = [&](int kt, int buf) {
    char* sK = smem + buf * 2 * C::TILEB;
    char* sV = sK + C::TILEB;
    if constexpr (BUF) {
      // unsigned: a cache of 2-4 GiB has tile offsets past INT_MAX (soffset is an unsigned 32-bit add)
      const int soff = __builtin_amdgcn_readfirstlane((int)((unsigned)(bt_next * a.Hkv + kvh) * (unsigned)(KT * D * 2)));
#pragma unroll
      for (int i = 0; i < BPW; ++i) {
        const int p = wid_u + NWV * i;
        blds16(srd_k, koff[i], soff, sK + p * 1024);
        blds16(srd_v, voff[i], soff, sV + p * 1024);
      }
    } else if constexpr (PAGED) {
      const size_t base = ((size_t)bt_next * a.Hkv + kvh) * KT * D;
      const bf16_t* kb = a.k + base;
      const bf16_t* vb = a.v + base;
      stage_kv<D, false, false, NWV>(sK, wid_u, NWV, lane, [&](int r) { return kb + (size_t)r * D; });
      stage_kv<D, true, false, NWV>(sV, wid_u, NWV, lane, [&](int r) { return vb + (size_t)r * D; });
    } else {
      const int k0 = kt * KT;
      auto rowp = [&](const bf16_t* base, int r) {
        int tok = k0 + r;
        tok = tok < kv_len ? tok : kv_len - 1;
        return base + (size_t)(kv_off + tok) * a.kv_stride + kvh * D;
      };
      stage_kv<D, false, false, NWV>(sK, wid_u, NWV, lane, [&](int r) { return rowp(a.k, r); });
      stage_kv<D, true, false, NWV>(sV, wid_u, NWV, lane, [&](int r) { return rowp(a.v, r); });
    }
  };

  if (n_kt > 0) stage(0, 0);
  if constexpr (PAGED) bt_next = n_kt > 1 ? s_bt[1] : 0;
  wait_vmcnt0();
  __syncthreads();

  for (int kt = 0; kt < n_kt; ++kt) {
    unsigned long long t0 = 0, t1 = 0, t2 = 0, t3 = 0, t4 = 0;
    if constexpr (STAMP) t0 = __builtin_amdgcn_s_memtime();
    const int cur = kt & 1;
    const char* sK = smem + cur * 2 * C::TILEB;
    const char* sV = sK + C::TILEB;
    const int k0 = kt * KT;
    const bool active = !CAUSAL || k0 <= wave_pmax;
    // ---- S^T = K Q^T ----
    f32x4 s[4][2];
    if (active) {
      if constexpr (PRIO == 1) __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        s[t][0] = (f32x4){0.f, 0.f, 0.f, 0.f};
        s[t][1] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < C::KS; ++ks) {
          const bf16x8 kf = load_k<D>(sK, t, ks, lane);
          s[t][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[0][ks], s[t][0], 0, 0, 0);
          s[t][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[1][ks], s[t][1], 0, 0, 0);
        }
      }
      if constexpr (PRIO == 1) __builtin_amdgcn_s_setprio(0);
    }
    if constexpr (STAMP) t1 = __builtin_amdgcn_s_memtime();
    // next tile's DMA issued behind the QK^T MFMAs (async-STAGE split: the issue overlaps the MFMA
    // pipe instead of delaying it); every wave stages its pieces, active or not
    if (kt + 1 < n_kt) stage(kt + 1, cur ^ 1);
    if constexpr (PAGED) bt_next = kt + 2 < n_kt ? s_bt[kt + 2] : 0;  // consumed next iteration
    if constexpr (STAMP) t2 = t3 = t4 = __builtin_amdgcn_s_memtime();
    if (active) {
      // ---- online softmax (per query column, lane-local + xor 16/32) ----
      // Max on the raw scores (scale > 0 keeps the order); the log2 scale is folded into one FMA
      // per element. Deferred rescale: the reference max m_i only moves when the tile max exceeds
      // it by more than RESCALE_LOG2 (p stays <= 2^RESCALE_LOG2, exact in fp32 / bf16 P), so the
      // O *= alpha pass (DT*2*4 multiplies per lane) runs on a few early tiles instead of every tile.
      const bool need_mask = CAUSAL ? (k0 + KT - 1 > ctx0 + pbase) || (k0 + KT > kv_len) : (k0 + KT > kv_len);
      const float c = a.scale_log2;
      float alpha[2];
      // one wave-uniform branch per tile (the masked body only runs on diagonal / ragged tiles)
      auto softmax = [&](auto mask_tag, const int qt) {
        constexpr bool MASK = decltype(mask_tag)::value;
        const int qpos = ctx0 + pbase + 16 * qt + fr;
        float mx = -INFINITY;
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            float x = s[t][qt][r];
            if constexpr (MASK) {
              const int kj = k0 + 16 * t + 4 * fh + r;
              const bool ok = kj < kv_len && (!CAUSAL || kj <= qpos);
              x = ok ? x : -INFINITY;
              s[t][qt][r] = x;
            }
            mx = fmaxf(mx, x);
          }
        mx = max_xor16(mx);
        mx = max_xor32(mx);
        const float mxs = mx * c;
        alpha[qt] = 1.f;
        if (mxs > m_i[qt] + RESCALE_LOG2) {
          alpha[qt] = m_i[qt] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_i[qt] - mxs);
          m_i[qt] = mxs;
        }
        const float mref = m_i[qt] == -INFINITY ? 0.f : m_i[qt];
        float ls = 0.f;
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[t][qt][r], c, -mref));
            s[t][qt][r] = p;
            ls += p;
          }
        l_i[qt] = l_i[qt] * alpha[qt] + ls;
      };
      if (need_mask) {
        softmax(std::true_type{}, 0);
        softmax(std::true_type{}, 1);
      } else {
        softmax(std::false_type{}, 0);
        softmax(std::false_type{}, 1);
      }
      if (__builtin_amdgcn_ballot_w64(alpha[0] != 1.f || alpha[1] != 1.f)) {
#pragma unroll
        for (int dt = 0; dt < C::DT; ++dt)
#pragma unroll
          for (int qt = 0; qt < 2; ++qt) o[dt][qt] *= alpha[qt];
      }
      // ---- O^T += V^T P^T ----
      bf16x8 pb[2][2];
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int qt = 0; qt < 2; ++qt) pb[ks][qt] = pack_p(s[2 * ks][qt], s[2 * ks + 1][qt]);
      if constexpr (STAMP) t3 = __builtin_amdgcn_s_memtime();
      if constexpr (PRIO != 0) __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int dt = 0; dt < C::DT; ++dt)
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
          const bf16x8 vf = load_vt<D>(sV, dt, ks, lane);
          o[dt][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pb[ks][0], o[dt][0], 0, 0, 0);
          o[dt][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pb[ks][1], o[dt][1], 0, 0, 0);
        }
      if constexpr (PRIO != 0) __builtin_amdgcn_s_setprio(0);
      if constexpr (STAMP) t4 = __builtin_amdgcn_s_memtime();
    }
    wait_vmcnt0();
    __syncthreads();
    if constexpr (STAMP) {
      const unsigned long long t5 = __builtin_amdgcn_s_memtime();
      stp[0] += t2 - t1;  // DMA issue of the next tile
      stp[1] += t1 - t0;  // QK^T (K reads + 32 MFMA issue)
      stp[2] += t3 - t2;  // softmax (+ waiting for the QK^T results)
      stp[3] += t4 - t3;  // PV (V tr-reads + 32 MFMA issue)
      stp[4] += t5 - t4;  // vmcnt(0) + barrier
      stp[5] += 1;
    }
  }
  if constexpr (STAMP) {
    if (lane == 0 && g_attn_dbg) {
      unsigned long long* d = g_attn_dbg + ((size_t)(blockIdx.y * gridDim.x + blockIdx.x) * 4 + wid) * 6;
#pragma unroll
      for (int i = 0; i < 6; ++i) d[i] = stp[i];
    }
  }

  // ---- finalize: O = O^T / l, store 4 consecutive d (8 B) per (dt, qt) ----
#pragma unroll
  for (int qt = 0; qt < 2; ++qt) {
    float l = l_i[qt];
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    const float inv = l > 0.f ? 1.f / l : 0.f;
    const int qi = pbase + 16 * qt + fr;
    if (qi < q_len) {
      bf16_t* op = a.out + (size_t)(q_off + qi) * a.out_stride + hq * D + 4 * fh;
#pragma unroll
      for (int dt = 0; dt < C::DT; ++dt) {
        const f32x4 v = o[dt][qt] * inv;
        const unsigned lo = pk2bf(v[0], v[1]);
        const unsigned hi = pk2bf(v[2], v[3]);
        *reinterpret_cast<uint2*>(op + 16 * dt) = make_uint2(lo, hi);
      }
    }
  }
}

// ------------------------------------------------------------------------------------
// Encoder attention (bidirectional, K / V rows beside each other in a packed qkv buffer; D 32 and 64).
// A 64-key tile of 32 queries is 32 exponentials a lane (8 clocks of a SIMD each, measured) and some 125 other vector instructions
// (fma, sum, maximum, conversion), against 8 D of 32x32x16 MFMA clocks: the vector unit bounds it. So a wave takes one column
// block of 32 queries, a lane pair each: the maximum is one lane swap a tile, the sum stays in the lane until the end. 32x32x16
// products hold the issue port 8 of their 32 clocks (16x16x32: 8 of 16); K / V addresses are scalar and a tile's buffer is known
// when compiling. Four waves a SIMD share the two units: the vector one is busy 75 % of the time, the matrix one 46 %.
// 12 sequences of 13764 rows, 16 heads of 64: 110 -> 93 us (0.73 us a tile and wave), 64 sequences of 1344 rows 659, one sequence
// of 1330 25 -> 23; 256 of up to 60 rows, 12 heads of 32: 17.1 -> 16.5. Wave priorities around the products changed nothing;
// looking for the maximum only where a sum outgrows 2^8 takes 20 instructions off, but the scores computed again beside it cost
// the fourth wave (94 us). Other head sizes, grouped heads and unaligned rows stay on attn_prefill_kernel.
// Layouts as in attn_prefill_v3_kernel; V rows are swizzled by pairs of 32-B granules (a transposed read takes four rows of two
// granules from each half of the banks).
template <int D>
__global__ __launch_bounds__(256, 3) void attn_encoder_kernel(PrefillArgs a) {
  using C = Cfg<D>;
  constexpr int KS = D / 16, DB = D / 32, PPW = C::PIECES / 4;  // MFMA steps over d, 32-wide blocks of d, DMA pieces a wave
  __shared__ __attribute__((aligned(16))) char smem[4 * C::TILEB];  // [buf][K | V]
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 31, h = lane >> 5, i16 = lane & 15;
  int tix, head;
  prefill_block(a, tix, head);
  const int seq = a.tiles[2 * tix], q_start = a.tiles[2 * tix + 1];
  const int q_off = a.cu_q[seq], q_len = a.cu_q[seq + 1] - q_off;
  const int kv_len = a.kv_lens[seq], n_kt = (kv_len + KT - 1) / KT;
  const int qi = q_start + wid * 32 + n;  // this lane's query

  bf16x8 qf[KS];
  {
    const bf16_t* qp = a.q + (size_t)(q_off + min(qi, q_len - 1)) * a.q_stride + head * D + 8 * h;
#pragma unroll
    for (int s = 0; s < KS; ++s) qf[s] = *reinterpret_cast<const bf16x8*>(qp + 16 * s);
  }
  // waited for here: left to the compiler, its waits stand at the uses, inside the loop, and wait for the tile's DMAs too
#pragma unroll
  for (int s = 0; s < KS; ++s) asm volatile("" : "+v"(qf[s]));

  // per-lane source offsets of the wave's pieces, from the tile's first row
  const int ldb = a.kv_stride * 2;
  int prow[PPW], koff[PPW], voff[PPW], kch[PPW], vch[PPW];
#pragma unroll
  for (int i = 0; i < PPW; ++i) {
    const int row = (wid * PPW + i) * C::RPP + lane / C::NC, ph = lane % C::NC;
    prow[i] = row;
    kch[i] = 16 * (ph ^ kswz<D>(row));
    vch[i] = 16 * (ph ^ vswz32<D>(row));
    koff[i] = row * ldb + kch[i];
    voff[i] = row * ldb + vch[i];
  }
  const size_t kv0 = (size_t)a.cu_kv[seq] * a.kv_stride + head * D;
  const unsigned lds0 = __builtin_amdgcn_readfirstlane(lds_addr(smem));
  auto stage = [&](int kt) {
    const size_t at = kv0 + (size_t)kt * KT * a.kv_stride;
    const i32x4 srd_k = make_srd(a.k + at, 0x7fffffffu), srd_v = make_srd(a.v + at, 0x7fffffffu);
    if ((kt + 1) * KT > kv_len) {  // rows past the end read the last one: their scores are masked
      const int last = kv_len - 1 - kt * KT;
#pragma unroll
      for (int i = 0; i < PPW; ++i) {
        koff[i] = min(prow[i], last) * ldb + kch[i];
        voff[i] = min(prow[i], last) * ldb + vch[i];
      }
    }
    const unsigned dst = lds0 + (kt & 1) * 2 * C::TILEB + wid * PPW * 1024;
#pragma unroll
    for (int i = 0; i < PPW; ++i) {
      blds16_asm(srd_k, koff[i], 0, dst + i * 1024);
      blds16_asm(srd_v, voff[i], 0, dst + C::TILEB + i * 1024);
    }
  };

  // fragment reads: the swizzles of rows 32 kb + n and 16 ks + 4 h + .. do not depend on kb and ks
  int kat[KS], vat[DB][2];
#pragma unroll
  for (int s = 0; s < KS; ++s) kat[s] = n * C::ROWB + 16 * ((2 * s + h) ^ kswz<D>(n));
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int row = 4 * h + (i16 >> 2) + 8 * u, chunk = 2 * (2 * db + ((lane >> 4) & 1)) + ((i16 >> 1) & 1);
      vat[db][u] = C::TILEB + row * C::ROWB + 16 * (chunk ^ vswz32<D>(row)) + 8 * (i16 & 1);
    }

  f32x16 o[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[db][e] = 0.f;
  // mref: the maximum that the exponents are taken against (0 while every score was -inf), move: the score that moves it
  float l_i = 0.f, mref = 0.f, move = -INFINITY;
  bool none = true;
  const float c = a.scale_log2;

  auto tile_step = [&](int kt, auto buf_tag) __attribute__((always_inline)) {
    const char* tile = smem + decltype(buf_tag)::value * 2 * C::TILEB;
    if (kt + 1 < n_kt) stage(kt + 1);  // into the buffer that every wave has read out
    f32x16 s[2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int e = 0; e < 16; ++e) s[kb][e] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        const bf16x8 kf = *reinterpret_cast<const bf16x8*>(tile + kat[ks] + kb * 32 * C::ROWB);
        s[kb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[ks], s[kb], 0, 0, 0);
      }
    // softmax as in attn_prefill_kernel: maximum of the raw scores, deferred rescale
    if ((kt + 1) * KT > kv_len) {
      const int left = kv_len - kt * KT - 4 * h;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int e = 0; e < 16; ++e)
          if (32 * kb + 8 * (e >> 2) + (e & 3) >= left) s[kb][e] = -INFINITY;
    }
    float mx = s[0][0];
#pragma unroll
    for (int e = 1; e < 32; ++e) mx = fmaxf(mx, s[e >> 4][e & 15]);
    const float mxs = max_xor32(mx) * c;
    if (__builtin_amdgcn_ballot_w64(mxs > move)) {
      if (mxs > move) {
        const float alpha = none ? 0.f : __builtin_amdgcn_exp2f(mref - mxs);
        none = false;
        mref = mxs;
        move = mxs + RESCALE_LOG2;
        l_i *= alpha;
#pragma unroll
        for (int db = 0; db < DB; ++db) o[db] *= alpha;
      }
    }
    float ls[2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kb][e], c, -mref));
        s[kb][e] = p;
        ls[kb] = e ? ls[kb] + p : p;
      }
    l_i += ls[0] + ls[1];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      u32x4 pw;
#pragma unroll
      for (int j = 0; j < 4; ++j) pw[j] = pk2bf(s[ks >> 1][8 * (ks & 1) + 2 * j], s[ks >> 1][8 * (ks & 1) + 2 * j + 1]);
      const bf16x8 pb = __builtin_bit_cast(bf16x8, pw);
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        const bf16x4 v0 = tr_read(tile + vat[db][0] + ks * 16 * C::ROWB), v1 = tr_read(tile + vat[db][1] + ks * 16 * C::ROWB);
        const bf16x8 vf = (bf16x8){v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
        o[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pb, o[db], 0, 0, 0);
      }
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };
  if (n_kt > 0) stage(0);
  asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  for (int kt = 0; kt < n_kt; kt += 2) {  // the buffer of a tile is known when compiling: no address arithmetic
    tile_step(kt, std::integral_constant<int, 0>{});
    if (kt + 1 < n_kt) tile_step(kt + 1, std::integral_constant<int, 1>{});
  }

  l_i += __shfl_xor(l_i, 32, 64);
  const float inv = l_i > 0.f ? 1.f / l_i : 0.f;
  if (qi < q_len) {
    bf16_t* op = a.out + (size_t)(q_off + qi) * a.out_stride + head * D + 4 * h;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int b = 0; b < 4; ++b)
        *reinterpret_cast<uint2*>(op + 32 * db + 8 * b) =
            make_uint2(pk2bf(o[db][4 * b] * inv, o[db][4 * b + 1] * inv), pk2bf(o[db][4 * b + 2] * inv, o[db][4 * b + 3] * inv));
  }
}

template <typename F, int... Is>
__device__ __forceinline__ void pp_static_for_impl(F&& f, std::integer_sequence<int, Is...>) {
  (f(std::integral_constant<int, Is>{}), ...);
}
// f(integral_constant<int, i>) for i = 0..N-1 (compile-time slot indices of a fully unrolled loop)
template <int N, typename F>
__device__ __forceinline__ void pp_static_for(F&& f) {
  pp_static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// ------------------------------------------------------------------------------------
// Software-pipelined prefill attention, one wave per SIMD (Llama config: D 128, 4 query heads per
// KV head, causal, paged cache < 4 GiB). attn_prefill_kernel runs two waves per SIMD, each in
// lockstep phases QK^T -> softmax -> PV: the stamps put a wave at ~4.3k cycles per 64-key tile for
// 1024 cycles of its own 16x16x32 MFMAs (~48 % matrix-pipe use), and a barrier-alternated 8-wave
// variant (attn_prefill_pp_kernel) was slower still -- the two waves of a SIMD share one vector
// issue port, and a 16x16x32 MFMA holds it 8 of its 16 cycles. Here:
//   * 32x32x16 MFMAs (the issue port is held 8 of 32 cycles per MFMA, MI355X_MICROARCH.md cycle
//     constants), 32 per tile per wave, and ONE wave per SIMD (4-wave block, one block per CU);
//   * iteration t issues PV(t-1) then QK^T(t+1) on the matrix pipe while the same wave's VALU runs the
//     online softmax of tile t between them: 32 slots, one MFMA each, the LDS fragment of slot i + 2
//     and a softmax chunk (max in slots 0..3, row statistics in 4, one element's fma / exp / add per
//     slot from 5 on: at most one transcendental per MFMA gap). Every MFMA is an ordered volatile asm
//     and each chunk's inputs / results are pinned, so neither the IR passes nor the scheduler can
//     regroup the stream; S is double-buffered (tile loop unrolled by two), P is single-buffered
//     (P(t-1)[ks] is dead before P(t)[ks] is packed);
//   * K / V ring of 4 slots, K staged 3 and V 2 tiles ahead, so iteration t's last two slots can read
//     the first PV fragments of iteration t + 1; LDS-DMA as inline asm (the intrinsic made the
//     waitcnt pass drain vmcnt(0) before every later ds_read); one vmcnt + barrier per tile.
// Diagonal / ragged tiles (masked softmax), the first tile (no PV) and the last (no QK) run the same
// MFMA stream with its halves guarded and the whole softmax after it.
// Layouts (v_mfma_f32_32x32x16_bf16, lane l, h = l >> 5): A[i = l & 31][k = 8h + j], B[k = 8h + j][n = l & 31],
// C[8b + 4h + r][l & 31] in acc[4b + r]. S^T = K Q^T: lane holds query pbase + (l & 31), keys
// 32 kb + 8b + 4h + r. P^T fragment of key step ks (16 keys) = acc S[ks / 2][8 (ks % 2) + j] (keys
// 16 ks + 8 (j / 4) + 4h + j % 4), so V^T is read with the same key order: ds_read_b64_tr_b16 of rows
// 16 ks + 4h + (i >> 2) and + 8 (i = l & 15) gives lane l the d column 32 db + 16 ((l >> 4) & 1) + i.
constexpr int V3_NS = 4;
constexpr int V3_PF = 4, V3_RING = 8;  // ring size divides the 32 slots (continuity across iterations)

// MFMA through the builtin (the compiler's hazard recognizer then covers every MFMA-result read: as
// inline asm the compiler treated the results as ready and could copy an accumulator before the MFMA
// retired). The slot order is kept by a scheduling barrier after every slot. Callers never chain two
// on the same accumulator back to back (PV db-minor, QK^T alternating key blocks).
__device__ __forceinline__ void mfma32_v(f32x16& acc, const bf16x8& a, const bf16x8& b) {
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
}
__device__ __forceinline__ void mfma32_v0(f32x16& acc, const bf16x8& a, const bf16x8& b) {
  const f32x16 z = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, z, 0, 0, 0);
}
// Empty volatile asm on a value: the computation of x cannot move across the pin (inputs pinned at
// the start of a slot's VALU chunk, results at its end: the chunk stays between its two MFMAs).
template <typename T>
__device__ __forceinline__ void pin(T& x) {
  asm volatile("" : "+v"(x));
}
__device__ __forceinline__ void pin_s(int& x) { asm volatile("" : "+s"(x)); }
// The asm MFMAs are opaque to the compiler's hazard recognizer: a VALU read of an MFMA result needs
// the XDL-write -> VALU-read wait states (18 for a 16-pass op), and a VALU write read by an MFMA a few.
__device__ __forceinline__ void mfma_result_wait() {}
// NW = 4: 32 query rows, the tile's first or (blockIdx.y) second half.
// NW = 8: two groups of 4 waves (query rows q_start + [0, 32) and + [32, 64)) share every K / V tile,
// so each SIMD runs two of these streams and one wave's dependency stalls are the other's issue slots.
// DIAG (stamp builds only, wrong results): 1 = no softmax chunks in the fast slots, 2 = no fragment reads
// PRIO_B: static s_setprio 1 for waves 4-7 over the tile loop (MI355X_MICROARCH.md "Two waves per SIMD"
// item 4: the second-dispatched half loses every arbitration otherwise).
// WIDE: the output tile goes through LDS and out as whole 256-B rows (16-B stores, 4 rows per wave
// instruction) instead of 16 8-B stores per lane into 32 different rows (MI355X_MICROARCH.md: the
// attention epilogue store tail is store-issue bound).
template <int NW = 4, bool STAMP = false, int DIAG = 0, int PRIO_B = 0, bool WIDE = false>
__global__ __launch_bounds__(NW * 64, NW / 4) void attn_prefill_v3_kernel(PrefillArgs a) {
  constexpr int D = 128;
  using C = Cfg<D>;
  __shared__ __attribute__((aligned(16))) char smem[2 * V3_NS * C::TILEB];  // [K slots][V slots] 128 KB
  __shared__ int s_bt[MAX_BT];

  constexpr int PPW = 16 / NW;  // DMA pieces per wave per K or V tile
  const int lane = threadIdx.x & 63;
  const int wid_u = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  int tix, hg;
  prefill_block(a, tix, hg);
  const int seq = a.tiles[2 * tix], q_start = a.tiles[2 * tix + 1] + (NW == 4 ? 32 * (int)blockIdx.y : 0);
  const int G = a.Hq / a.Hkv;
  const int groups_per_kv = G / 4;
  const int kvh = hg / groups_per_kv;
  const int hq = kvh * G + (hg % groups_per_kv) * 4 + (wid_u & 3);
  const int pbase = q_start + 32 * (wid_u >> 2);

  const int q_off = a.cu_q[seq];
  const int q_len = a.cu_q[seq + 1] - q_off;
  if (NW == 4 && q_start >= q_len) return;  // block-uniform, before any barrier
  const int kv_len = a.kv_lens[seq];
  const int ctx0 = kv_len - q_len;
  // block-uniform tile counts (every wave runs the same iterations and barriers)
  const int blk_qmax = min(q_start + 8 * NW, q_len) - 1;
  const int n_keys = min(kv_len, ctx0 + blk_qmax + 1);
  const int n_kt = (n_keys + KT - 1) / KT;
  const int h = lane >> 5, l32 = lane & 31;
  // tiles [0, n_fast) need no mask for any wave: every key <= the block's first query position and < kv_len
  const int n_fast = min((ctx0 + q_start + 1) / KT, kv_len / KT);

  // Q^T fragments (B operand): query pbase + l32, d = 16 s + 8 h + [0, 8)
  bf16x8 qf[8];
  {
    int qi = pbase + l32;
    qi = qi < q_len ? qi : q_len - 1;
    const bf16_t* qp = a.q + (size_t)(q_off + qi) * a.q_stride + hq * D + 8 * h;
#pragma unroll
    for (int s = 0; s < 8; ++s) qf[s] = *reinterpret_cast<const bf16x8*>(qp + 16 * s);
  }
  const int* bt = a.block_tables + (size_t)seq * a.bt_stride;
  for (int i = threadIdx.x; i < n_kt; i += NW * 64) s_bt[i] = bt[i];

  // DMA: pieces PPW wid + i (i < PPW) of a 16-piece tile (rows 4 p .. 4 p + 3, one 16-B chunk per lane)
  int koff[PPW], voff[PPW];
#pragma unroll
  for (int i = 0; i < PPW; ++i) {
    const int p = PPW * wid_u + i;
    const int row = p * C::RPP + lane / C::NC, ph = lane % C::NC;
    koff[i] = row * C::ROWB + 16 * (ph ^ kswz<D>(row));
    voff[i] = row * C::ROWB + 16 * (ph ^ vswz<D>(row));
  }
  const i32x4 srd_k = make_srd(a.k, a.kv_bytes);
  const i32x4 srd_v = make_srd(a.v, a.kv_bytes);
  const unsigned lds0 = lds_addr(smem);
  auto tile_soff = [&](int kt) {
    return __builtin_amdgcn_readfirstlane((int)((unsigned)(s_bt[kt] * a.Hkv + kvh) * (unsigned)(KT * D * 2)));
  };
  auto kslot_off = [&](int kt) { return (kt & (V3_NS - 1)) * C::TILEB; };
  auto vslot_off = [&](int kt) { return (V3_NS + (kt & (V3_NS - 1))) * C::TILEB; };
  auto stage_piece = [&](int kt, int soff, bool is_v, int i) {
    blds16_asm(is_v ? srd_v : srd_k, is_v ? voff[i] : koff[i], soff,
               lds0 + (is_v ? vslot_off(kt) : kslot_off(kt)) + (PPW * wid_u + i) * 1024);
  };
  auto stage = [&](int kt, bool is_v) {
    const int soff = tile_soff(kt);
#pragma unroll
    for (int i = 0; i < PPW; ++i) stage_piece(kt, soff, is_v, i);
  };

  // per-lane fragment offsets (bytes within a tile)
  // K (A of QK^T): row 32 kb + l32, chunk (2 s + h) ^ (l & 15) = 16 (h ^ (l & 1)) + 32 (s ^ ((l & 15) >> 1))
  const int kx = (lane & 15) >> 1;
  const int kbase = l32 * 256 + 16 * (h ^ (lane & 1));
  // V^T (A of PV): rows 16 ks + 4h + (i >> 2) [+ 8], chunk (2 (2 db + c16) + ((i >> 1) & 1)) ^ 2 (row & 7)
  const int vi = lane & 15, c16 = (lane >> 4) & 1;
  const int vrow = 4 * h + (vi >> 2);
  const int vbase = vrow * 256 + 16 * ((vi >> 1) & 1) + 8 * (vi & 1);
  const int vx = vrow & 7;
  auto kfrag = [&](int tile_off, int kb, int s) -> bf16x8 {
    return *reinterpret_cast<const bf16x8*>(smem + tile_off + kbase + kb * 32 * 256 + 32 * (s ^ kx));
  };
  auto vfrag = [&](int tile_off, int db, int ks) -> bf16x8 {
    const char* p = smem + tile_off + vbase + ks * 16 * 256 + 32 * ((2 * db + c16) ^ vx);
    const bf16x4 x0 = tr_read(p), x1 = tr_read(p + 8 * 256);
    return (bf16x8){x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
  };

  f32x16 o[4];
#pragma unroll
  for (int db = 0; db < 4; ++db)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[db][e] = 0.f;
  float m_i = -INFINITY, l_i = 0.f;
  f32x16 S0[2], S1[2];
  bf16x8 P[4];
  // fragment of MFMA slot i in ring[i % V3_RING], read V3_PF slots ahead (LDS latency ~100+ cycles: at
  // 2 slots ahead every MFMA waited on its own ds_read)
  bf16x8 ring[V3_RING];
  const float c = a.scale_log2;

  __syncthreads();  // s_bt
#pragma unroll
  for (int kt = 0; kt < 3; ++kt)
    if (kt < n_kt) stage(kt, false);
  stage(0, true);
  if (n_kt > 1) stage(1, true);
  wait_vmcnt0();
  __syncthreads();

  auto pack_p32 = [&](const f32x16& A, int e0) -> bf16x8 {
    return (bf16x8){f2bf_s(A[e0]), f2bf_s(A[e0 + 1]), f2bf_s(A[e0 + 2]), f2bf_s(A[e0 + 3]),
                    f2bf_s(A[e0 + 4]), f2bf_s(A[e0 + 5]), f2bf_s(A[e0 + 6]), f2bf_s(A[e0 + 7])};
  };
  // simple (non-interleaved) pieces for the warm-up tile and the epilogue
  auto qk_simple = [&](int kt, f32x16 (&S)[2]) {
#pragma unroll
    for (int sd = 0; sd < 8; ++sd)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        const bf16x8 f = kfrag(kslot_off(kt), kb, sd);
        if (sd == 0) mfma32_v0(S[kb], f, qf[sd]);
        else mfma32_v(S[kb], f, qf[sd]);
      }
  };
  auto pv_simple = [&](int kt) {
    const int vo = vslot_off(kt);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int db = 0; db < 4; ++db) mfma32_v(o[db], vfrag(vo, db, ks), P[ks]);
  };
  // whole-tile online softmax: this lane's query, 32 of the tile's 64 keys -> P; returns alpha
  auto softmax = [&](auto mask_tag, int k0, f32x16 (&S)[2]) -> float {
    constexpr bool MASK = decltype(mask_tag)::value;
    if constexpr (MASK) {
      const int qpos = ctx0 + pbase + l32;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int kj = k0 + 32 * kb + 8 * (e >> 2) + 4 * h + (e & 3);
          S[kb][e] = (kj < kv_len && kj <= qpos) ? S[kb][e] : -INFINITY;
        }
    }
    float mx = -INFINITY;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int e = 0; e < 16; ++e) mx = fmaxf(mx, S[kb][e]);
    mx = max_xor32(mx);
    const float mxs = mx * c;
    const bool up = mxs > m_i + RESCALE_LOG2;
    const float alpha = up ? (m_i == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_i - mxs)) : 1.f;
    m_i = up ? mxs : m_i;
    const float mref = m_i == -INFINITY ? 0.f : m_i;
    float ls = 0.f;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const float pe = __builtin_amdgcn_exp2f(__builtin_fmaf(S[kb][e], c, -mref));
        S[kb][e] = pe;
        ls += pe;
      }
    l_i = l_i * alpha + ls;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) P[ks] = pack_p32(S[ks >> 1], 8 * (ks & 1));
    return alpha;
  };
  auto rescale = [&](float alpha) {
    if (__builtin_amdgcn_ballot_w64(alpha != 1.f)) {
#pragma unroll
      for (int db = 0; db < 4; ++db) o[db] *= alpha;
    }
  };
  auto barrier = [] {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };

  unsigned long long stp[4] = {0, 0, 0, 0};
  // Fast iteration t (1 <= t < t_end: tile t unmasked, PV(t-1) and QK^T(t+1) exist). MFMA slots
  // 0..15: PV(t-1) (V slot t-1; ks = i / 4, db = i % 4), 16..31: QK^T(t+1) (K slot t+1; kb = i % 2,
  // d-step (i-16) / 2). Slot i reads the fragment of slot i + V3_PF; the last V3_PF slots read the
  // first PV(t) fragments of the next iteration. Softmax(t) of S_cur -> P in chunks. DMA: K(t+3) (slots 6..18),
  // V(t+2) (22..28). Then O *= alpha(t) (rare), vmcnt (this iteration's DMAs stay in flight), barrier.
  // PH = t & 3, a compile-time constant (the loop below is unrolled by the ring's 4 slots): with the slot
  // offsets constant every fragment read folds its tile offset into the ds_read immediate (one v_add per
  // fragment read with runtime offsets; unrolled: 6 x 5.4k 1328 -> 1279 us, one 5.2k prompt 250 -> 229,
  // profiles/attn_prefill_unroll4_ab_r5.log)
  auto fast = [&](auto ph_tag, int t, f32x16 (&S_cur)[2], f32x16 (&S_next)[2]) {
    constexpr int PH = decltype(ph_tag)::value;
    unsigned long long t0 = 0;
    if constexpr (STAMP) t0 = __builtin_amdgcn_s_memtime();
    static_assert(V3_NS == 4 && PH >= 0 && PH < 4, "slot phase");
    constexpr int vo = (V3_NS + ((PH + 3) & 3)) * C::TILEB;  // V(t - 1)
    constexpr int ko = ((PH + 1) & 3) * C::TILEB;            // K(t + 1)
    constexpr int vno = (V3_NS + PH) * C::TILEB;             // V(t)
    const bool st_k = t + 3 < n_kt, st_v = t + 2 < n_kt;
    const int soff_k = tile_soff(st_k ? t + 3 : 0);
    const int soff_v = tile_soff(st_v ? t + 2 : 0);
    float alpha = 1.f, mx = -INFINITY, mref = 0.f, ls = 0.f, pend = 0.f;
    float pv[32];  // the probabilities of this tile (P is packed from here, S_cur is not rewritten)
    pp_static_for<32>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      // MFMA slot i
      if constexpr (i < 16) {
        mfma32_v(o[i % 4], ring[i % V3_RING], P[i / 4]);
      } else {
        constexpr int kb = i % 2, sd = (i - 16) / 2;
        if constexpr (sd == 0) mfma32_v0(S_next[kb], ring[i % V3_RING], qf[sd]);
        else mfma32_v(S_next[kb], ring[i % V3_RING], qf[sd]);
      }
      // fragment for slot i + V3_PF (the per-lane bases x tile offsets are CSE'd: 12 address adds per
      // iteration; the scheduling barrier at the end of the slot keeps each read in its slot)
      constexpr int j = i + V3_PF;
      if constexpr (DIAG != 2) {
        const int ao = j < 16 ? vo : (j < 32 ? ko : vno);
        if constexpr (j < 16) ring[j % V3_RING] = vfrag(ao, j % 4, j / 4);
        else if constexpr (j < 32) ring[j % V3_RING] = kfrag(ao, j % 2, (j - 16) / 2);
        else ring[j % V3_RING] = vfrag(ao, (j - 32) % 4, (j - 32) / 4);
      }
      // softmax chunk: max in slots 0..3, row statistics in 4, one element per slot from 5 on
      if constexpr (DIAG == 1) {
      } else if constexpr (i < 4) {
        // no input pins: a pinned copy of each element cost a v_mov (the sched barrier keeps the slot)
#pragma unroll
        for (int e = 0; e < 8; ++e) mx = fmaxf(mx, S_cur[i / 2][8 * (i % 2) + e]);
        pin(mx);
      } else if constexpr (i == 4) {
        mx = max_xor32(mx);
        const float mxs = mx * c;
        const bool up = mxs > m_i + RESCALE_LOG2;
        alpha = up ? (m_i == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_i - mxs)) : 1.f;
        m_i = up ? mxs : m_i;
        mref = m_i == -INFINITY ? 0.f : m_i;
        pin(alpha);
        pin(m_i);
        pin(mref);
      } else {
        // elements x with 5 + (27 x) / 32 == i: the probability straight from the accumulator, pinned
        // (results only: a pinned copy of an input element cost a v_mov); each is added to the row sum
        // one element later (no exp -> add dependency inside a slot)
        pp_static_for<32>([&](auto xc) {
          constexpr int x = decltype(xc)::value;
          if constexpr (5 + (27 * x) / 32 == i) {
            float pe = __builtin_amdgcn_exp2f(__builtin_fmaf(S_cur[x >> 4][x & 15], c, -mref));
            pin(pe);
            ls += pend;  // the previous element's value: no exp -> add dependency inside a slot
            pend = pe;
            pv[x] = pe;
            if constexpr (x % 8 == 7) {
              P[x / 8] = (bf16x8){f2bf_s(pv[x - 7]), f2bf_s(pv[x - 6]), f2bf_s(pv[x - 5]), f2bf_s(pv[x - 4]),
                                  f2bf_s(pv[x - 3]), f2bf_s(pv[x - 2]), f2bf_s(pv[x - 1]), f2bf_s(pv[x])};
              pin(P[x / 8]);
            }
            pin(ls);
          }
        });
      }
      // DMA pieces: K(t+3) in slots 6, 10, 14, 18; V(t+2) in slots 22, 24, 26, 28 (the first PPW of each)
      if constexpr (i >= 6 && i <= 18 && (i - 6) % 4 == 0 && (i - 6) / 4 < PPW) {
        if (st_k) stage_piece(t + 3, soff_k, false, (i - 6) / 4);
      }
      if constexpr (i >= 22 && i <= 28 && (i - 22) % 2 == 0 && (i - 22) / 2 < PPW) {
        if (st_v) stage_piece(t + 2, soff_v, true, (i - 22) / 2);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    l_i = l_i * alpha + (ls + pend);
    if constexpr (STAMP) {
      const unsigned long long t1 = __builtin_amdgcn_s_memtime();
      stp[0] += t1 - t0;
      t0 = t1;
    }
    rescale(alpha);
    // this iteration's DMAs (PPW per issued tile) stay in flight, the previous iteration's have landed
    if constexpr (PPW == 4) {
      if (st_k && st_v) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
      else if (st_k || st_v) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
      else wait_vmcnt0();
    } else {
      if (st_k && st_v) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
      else if (st_k || st_v) asm volatile("s_waitcnt vmcnt(2)" ::: "memory");
      else wait_vmcnt0();
    }
    barrier();
    if constexpr (STAMP) stp[1] += __builtin_amdgcn_s_memtime() - t0;
  };

  unsigned long long te = 0;
  if constexpr (STAMP) te = __builtin_amdgcn_s_memtime();
  if constexpr (PRIO_B) {
    if (wid_u >= 4) __builtin_amdgcn_s_setprio(1);
  }
  qk_simple(0, S0);  // S(0)
  mfma_result_wait();
  // fast iterations: [1, t_end); warm-up tile 0 when there is at least one
  const int t_end = min(n_fast, n_kt - 1);
  int t = 0;
  if (t_end >= 1) {
    // tile 0 (unmasked, QK^T(1) exists): softmax(0), S(1), DMA K(3) / V(2), the first PV(0) fragments
    softmax(std::false_type{}, 0, S0);
    qk_simple(1, S1);
    mfma_result_wait();
    if (3 < n_kt) stage(3, false);
    if (2 < n_kt) stage(2, true);
#pragma unroll
    for (int j = 0; j < V3_PF; ++j) ring[j] = vfrag(vslot_off(0), j % 4, j / 4);
    barrier();  // (O is zero: no rescale; the prologue DMAs were drained)
    t = 1;
    using P0 = std::integral_constant<int, 0>;
    using P1 = std::integral_constant<int, 1>;
    using P2 = std::integral_constant<int, 2>;
    using P3 = std::integral_constant<int, 3>;
    for (; t + 3 < t_end; t += 4) {  // t = 1 (mod 4) at every trip
      fast(P1{}, t, S1, S0);
      fast(P2{}, t + 1, S0, S1);
      fast(P3{}, t + 2, S1, S0);
      fast(P0{}, t + 3, S0, S1);
    }
    if (t < t_end) {
      fast(P1{}, t, S1, S0);
      ++t;
    }
    if (t < t_end) {
      fast(P2{}, t, S0, S1);
      ++t;
    }
    if (t < t_end) {
      fast(P3{}, t, S1, S0);
      ++t;
    }
    if (t & 1) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) S0[kb] = S1[kb];
    }
  }
  if constexpr (STAMP) {
    const unsigned long long t1 = __builtin_amdgcn_s_memtime();
    stp[2] += t1 - te - stp[0] - stp[1];
    te = t1;
  }
  // epilogue: tiles [t, n_kt) (masked diagonal / ragged ones and the last; at most 3), S(t) in S0, P(t-1)
  // pending. Every tile they touch is staged after V(t + 2) here (the ring holds it), then drained.
  if (t + 2 < n_kt) stage(t + 2, true);
  wait_vmcnt0();
  barrier();
  if (t >= 1) pv_simple(t - 1);
  for (; t < n_kt; ++t) {
    const int k0 = t * KT;
    const bool need_mask = (k0 + KT - 1 > ctx0 + pbase) || (k0 + KT > kv_len);
    mfma_result_wait();  // S(t) and O from the MFMAs just issued
    const float alpha = need_mask ? softmax(std::true_type{}, k0, S0) : softmax(std::false_type{}, k0, S0);
    rescale(alpha);
    pv_simple(t);
    if (t + 1 < n_kt) qk_simple(t + 1, S0);
  }
  if constexpr (STAMP) stp[3] += __builtin_amdgcn_s_memtime() - te;
  if constexpr (STAMP) {
    if (lane == 0 && g_attn_dbg) {
      unsigned long long* d = g_attn_dbg + ((size_t)(blockIdx.y * gridDim.x + blockIdx.x) * NW + wid_u) * 6;
#pragma unroll
      for (int i = 0; i < 4; ++i) d[i] = stp[i];
      d[4] = n_kt;
      d[5] = max(0, min(n_fast, n_kt - 1) - 1);  // fast iterations
    }
  }

  // finalize: O^T[32 db + 8 b + 4 h + r][query] = o[db][4 b + r] / l; {r0, r1} = {l_i, partner's l_i}
  const auto lr = __builtin_amdgcn_permlane32_swap(__float_as_uint(l_i), __float_as_uint(l_i), false, false);
  const float l = __uint_as_float(lr[0]) + __uint_as_float(lr[1]);
  const float inv = l > 0.f ? 1.f / l : 0.f;
  const int qi = pbase + l32;
  if constexpr (WIDE) {
    // every wave is past its last K / V slot read (the loop's barrier count is the same in both groups),
    // so the ring is free: each wave stages its 32 x 128 bf16 tile (8 KiB, rows of 256 B, 16-B chunk c of
    // row r at slot c ^ (r & 15)) and stores whole rows
    __syncthreads();
    char* so = smem + wid_u * 8192;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const int e = 4 * b;
        const int d = 32 * db + 8 * b + 4 * h;  // 4 values: chunk d / 8, half (d / 4) & 1
        const int c = (d >> 3) ^ (l32 & 15);
        *reinterpret_cast<uint2*>(so + l32 * 256 + 16 * c + 8 * ((d >> 2) & 1)) =
            make_uint2(pk2bf(o[db][e] * inv, o[db][e + 1] * inv), pk2bf(o[db][e + 2] * inv, o[db][e + 3] * inv));
      }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the wave's own LDS writes, read back by itself
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int r = 4 * i + (lane >> 4), c = lane & 15;
      const u32x4 v = *reinterpret_cast<const u32x4*>(so + r * 256 + 16 * (c ^ (r & 15)));
      if (pbase + r < q_len)
        *reinterpret_cast<u32x4*>(a.out + (size_t)(q_off + pbase + r) * a.out_stride + hq * D + 8 * c) = v;
    }
    return;
  }
  if (qi < q_len) {
    bf16_t* op = a.out + (size_t)(q_off + qi) * a.out_stride + hq * D + 4 * h;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const int e = 4 * b;
        *reinterpret_cast<uint2*>(op + 32 * db + 8 * b) =
            make_uint2(pk2bf(o[db][e] * inv, o[db][e + 1] * inv), pk2bf(o[db][e + 2] * inv, o[db][e + 3] * inv));
      }
  }
}

// ------------------------------------------------------------------------------------
// Decode attention (one query token per sequence), split-K over context partitions.
// ------------------------------------------------------------------------------------
struct DecodeArgs {
  const bf16_t* q; int q_stride;           // [B] rows, head h at +h*D
  const bf16_t* kc; const bf16_t* vc;      // paged caches
  const int* block_tables; int bt_stride, bt_cols;
  const int* kv_lens;                      // [B]
  float* part_o;                           // [B][Hq][max_parts][D]
  float* part_ml;                          // [B][Hq][max_parts][2]
  bf16_t* out; int out_stride;
  int Hq, Hkv, part_tiles, max_parts;
  float scale_log2;
  // Fused RoPE + KV append (null qkv_p: q is read from `q` and the cache already holds the new token).
  // The qkv projection arrives as fp32 split-K partial slabs P[S][B][ldp] (gemm_part.hip); every
  // block sums + rotates its G query heads itself, and the block owning the last KV tile also sums,
  // rotates and appends the new token's k / v before reading that tile.
  const float* qkv_p; long long p_slab; int ldp, S;
  const int* positions; const int* slots;
  const float* cos_t; const float* sin_t;
};

static_assert(KT == DEC_TILE, "a page");  // DEC_U: what a wave takes at a time where tiles come through registers

// Units per partition of one sequence: its keys spread evenly over all max_parts partitions (never fewer
// than part_tiles tiles per partition). The grid is sized once for max_parts (hipGraph
// capture), so sizing the split from the actual length keeps every launched block busy with the
// same amount of KV: splitting a 5.3k-token context by a fixed 32-tile partition left 1 of 4
// partitions idle and 8 vs 5 tiles per wave on the others.
__device__ __forceinline__ int decode_part_units(int n, const DecodeArgs& a, int unit = DEC_U) {
  return decode_share(n, a.part_tiles, a.max_parts, unit);
}

// LDS of one decode-attention block: one V tile per wave (KL: and one K tile per wave after them), then the
// block's rotated q (G x D bf16).
template <int D, int G, int NW = 4, bool KL = false, int DG = 0>
constexpr int decode_lds_bytes() {
  return NW * Cfg<D>::TILEB * (KL ? 2 : 1) / (!KL && DG == 0 ? KT / DEC_U : 1) + G * D * 2;
}

// The K / V stream bounds it, and for short contexts the trips to memory in front of it. Both lengths and page table are one trip,
// the queries' slabs and the first unit another (four in a row before: length, page, tile, and the slabs behind the tile, since
// vector loads return in order), and a wave's next unit is on its way while it works on one. Units of half a page: few pages
// spread over more waves and blocks, and many end closer together (with whole pages, a wave of two beside three of one). One
// layer, 128-wide heads, us with the join, page by page before / page by page ahead / in units: 11 rows of 2000 tokens, 8 KV heads
// 28.6 / 26.1 / 23.3; 3 of 4000 19.3 / 15.5 / 14.4; 20 of 5000 68.0 / 63.7 / 59.4; 25 of 2400 60 / - / 53.7; 1 of 5267 13.3 / 11.9
// / 10.5; 2 rows of 2000, 4 KV heads 11.3 / 10.7 / 8.4; 32 of 4200 in one partition (KL, whole pages) 96 / 92.5, 5.97 TB/s.
// One split-K partition block of decode attention: partition `part` of KV head `kvh` of sequence `b`.
// NW: waves per block (4; 8 for the batch-32 grid with one partition per sequence: one 8-wave block per
// CU keeps the same KV bytes in flight as two 4-wave blocks and needs no merge launch). A multi-partition
// sequence writes its partition records; attn_decode_reduce_kernel (or, deferred, the o_proj GEMM's
// gemm_part_merge) merges them.
// DG = 1 (diagnostic build, tools/attn_decode_probe.py): the loads of whole pages, one behind the other, without QK^T / softmax /
// PV -- what the access pattern takes without the kernel's units and look-ahead. DG = 2: as 1, but K also arrives by LDS-DMA
// (1 KiB per instruction, into the V buffer: results meaningless) instead of 64-B row pieces.
// KL: K tiles arrive by LDS-DMA too (whole 1 KiB pieces instead of 64-B row pieces per lane: the pure access
// pattern streams 4-5 % faster, tools/attn_decode_probe.py) and the QK^T fragments are read from LDS; a
// wave then holds 32 KB of LDS, so the single-partition grid uses 4-wave blocks (one per CU).
template <int D, int G, bool NT = false, int NW = 4, int DG = 0, bool KL = false>
__device__ __forceinline__ void attn_decode_block(const DecodeArgs& a, int part, int kvh, int b, char* smem) {
  constexpr int NTH = NW * 64;
  constexpr bool REGS = !KL && DG != 2;    // K and V tiles through registers
  constexpr bool AHEAD = REGS && DG == 0;  // ... and requested a tile ahead
  using C = Cfg<D>;
  constexpr int KU = AHEAD ? DEC_U : KT, UPT = KT / KU;  // keys of a unit, units of a page
  constexpr int VB = C::TILEB / UPT, VPC = C::PIECES / UPT;  // bytes and 1-KiB pieces of its values
  static_assert(G <= 16, "at most 16 query heads per KV head");
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int wid_u = __builtin_amdgcn_readfirstlane(wid);
  PageRow<2> table(a.block_tables + (size_t)b * a.bt_stride, a.bt_cols, lane);
  const int kv_len = ld_uniform(a.kv_lens + b), pos = ld_uniform((a.qkv_p ? a.positions : a.kv_lens) + b);
  const int n_kt = (kv_len + KU - 1) / KU;  // (all counts below in units)
  const int pt = decode_part_units(n_kt, a, KU);
  const int kt0 = part * pt;
  if (kt0 >= n_kt) return;  // block-uniform early exit (before any barrier)
  const int kt1 = min(kt0 + pt, n_kt);
  const int nparts = (n_kt + pt - 1) / pt;
  const int fr = lane & 15, fh = lane >> 4;
  table.wait();

  bf16x8 qf[C::KS];
  char* sV = smem + wid_u * VB;
  char* sK = smem + (NW + wid_u) * C::TILEB;  // KL only
  bf16x8 kf[KU / 16][C::KS];
  auto page = [&](int kt) { return (((size_t)table(kt / UPT) * a.Hkv + kvh) * KT + kt % UPT * KU) * D; };
  // (lanes' places as 32-bit offsets from a scalar address: a pair of registers a load otherwise)
  constexpr int VP = C::RPP < C::RB * C::GR ? C::RB * C::GR / C::RPP : 1;  // pieces until the swizzle repeats
  const unsigned k_lane = (fr * D + 8 * fh) * 2;
  unsigned v_lane[VP];
#pragma unroll
  for (int i = 0; i < VP; ++i)
    v_lane[i] = lane / C::NC * C::ROWB + 16 * ((lane % C::NC) ^ vswz<D>(i * C::RPP + lane / C::NC));
  constexpr int KP = C::RPP < 16 ? 16 / C::RPP : 1;  // K pieces likewise
  unsigned kd_lane[KP];
#pragma unroll
  for (int i = 0; i < KP; ++i)
    kd_lane[i] = lane / C::NC * C::ROWB + 16 * ((lane % C::NC) ^ kswz<D>(i * C::RPP + lane / C::NC));
  if constexpr (KL) {  // held: worked out again in front of the loop they cost 0.2 us
#pragma unroll
    for (int i = 0; i < VP; ++i) asm volatile("" : "+v"(v_lane[i]));
#pragma unroll
    for (int i = 0; i < KP; ++i) asm volatile("" : "+v"(kd_lane[i]));
  }
  // (the instruction's offset counts for both addresses: four pieces to a scalar base and an LDS base. With each piece's own bases,
  // the LDS one from vector registers, a tile's 32 requests were 200 instructions more: 256 pairs of 1000 / 2000 tokens 23.6 / 39.4
  // us, now 22.4 / 38.0)
  auto piece = [&](const bf16_t* tile, int i, unsigned at, char* lds) __attribute__((always_inline)) {
    const auto* g = (const __attribute__((address_space(1))) char*)tile + i / 4 * 4096 + at;
    auto* l = (__attribute__((address_space(3))) char*)lds + i / 4 * 4096;
    constexpr int AUX = NT ? 2 : 0;
    switch (i % 4) {
      case 0: __builtin_amdgcn_global_load_lds(g, l, 16, 0, AUX); break;
      case 1: __builtin_amdgcn_global_load_lds(g, l, 16, 1024, AUX); break;
      case 2: __builtin_amdgcn_global_load_lds(g, l, 16, 2048, AUX); break;
      default: __builtin_amdgcn_global_load_lds(g, l, 16, 3072, AUX); break;
    }
  };
  auto request_k = [&](int kt) {
    const bf16_t* kb = a.kc + page(kt);
    if constexpr (KL) {
#pragma unroll
      for (int i = 0; i < C::PIECES; ++i) piece(kb, i, kd_lane[i % KP], sK);
    } else {
#pragma unroll
      for (int t = 0; t < KU / 16; ++t)
#pragma unroll
        for (int s = 0; s < C::KS; ++s) {
          const bf16x8* p = reinterpret_cast<const bf16x8*>(reinterpret_cast<const char*>(kb + 16 * t * D + 32 * s) + k_lane);
          kf[t][s] = NT ? __builtin_nontemporal_load(p) : *p;
        }
    }
  };
  // V: whole 1-KiB pieces, by LDS-DMA (KL) or through registers, so that the tile behind it can be on its way while this one is
  // read from LDS (the compiler drains every load in flight around LDS-DMA pieces, K's with them)
  u32x4 vr[VPC];
  auto request_v = [&](int kt) {
    const bf16_t* vb = a.vc + page(kt);
    if constexpr (!REGS) {
#pragma unroll
      for (int i = 0; i < C::PIECES; ++i) piece(vb, i, v_lane[i % VP], sV);
    } else {
#pragma unroll
      for (int i = 0; i < VPC; ++i) {
        const u32x4* p = reinterpret_cast<const u32x4*>(reinterpret_cast<const char*>(vb) + i * 1024 + v_lane[i % VP]);
        vr[i] = NT ? __builtin_nontemporal_load(p) : *p;
      }
    }
  };
  // Rotating path (qkv_p): q = RoPE(bf16(sum_s P[s][b])) for this KV head's G query heads, staged through LDS; in the block owning
  // the last KV tile the new token's k (rotated) and v are appended meanwhile. Every wave takes whole heads, a rotate_half pair
  // (d, d + D / 2) a lane.
  bf16_t* s_q = reinterpret_cast<bf16_t*>(smem + NW * VB * (KL ? 2 : 1));
  constexpr int PL = D / 2, IPW = 64 / PL;  // pairs of a head, heads of a wave at a time
  const bool rope = a.qkv_p != nullptr, append = rope && kt1 == n_kt;  // block-uniform
  const int n_items = G + (append ? 2 : 0);                            // query heads, then k and v
  const int p = lane % PL, it0 = wid * IPW + lane / PL;
  float x1[PSU], x2[PSU], cs = 0.f, sn = 0.f;
  auto column = [&](int it) {
    it = min(it, G + 1);
    return a.qkv_p + (size_t)b * a.ldp + (size_t)(it < G ? kvh * G + it : (it == G ? a.Hq : a.Hq + a.Hkv) + kvh) * D + p;
  };
  auto request_item = [&](int it) {
    const float* ph = column(it);
#pragma unroll
    for (int u = 0; u < PSU; ++u) {
      const size_t o = (size_t)min(u, a.S - 1) * a.p_slab;
      x1[u] = ph[o];
      x2[u] = ph[o + PL];
    }
    cs = a.cos_t[(size_t)pos * PL + p];
    sn = a.sin_t[(size_t)pos * PL + p];
  };
  auto finish_item = [&](int it) {
    float s1 = 0.f, s2 = 0.f;
#pragma unroll
    for (int u = 0; u < PSU; ++u)
      if (u < a.S) {
        s1 += x1[u];
        s2 += x2[u];
      }
    for (int u = PSU; u < a.S; ++u) {
      s1 += column(it)[(size_t)u * a.p_slab];
      s2 += column(it)[(size_t)u * a.p_slab + PL];
    }
    s1 = bf2f(f2bf(s1));
    s2 = bf2f(f2bf(s2));
    const bf16_t r1 = f2bf(bf2f(f2bf(s1 * cs)) + bf2f(f2bf(-s2 * sn)));  // rope8's formula and roundings
    const bf16_t r2 = f2bf(bf2f(f2bf(s2 * cs)) + bf2f(f2bf(s1 * sn)));
    asm volatile("" ::"v"((unsigned)r1), "v"((unsigned)r2));  // every load is used on every path
    if (it < G) {
      s_q[it * D + p] = r1;
      s_q[it * D + PL + p] = r2;
    } else if (it < n_items) {
      const int slot = ld_uniform(a.slots + b);
      bf16_t* dst = (it == G ? const_cast<bf16_t*>(a.kc) : const_cast<bf16_t*>(a.vc)) +
                    (((size_t)(slot / KT) * a.Hkv + kvh) * KT + (slot % KT)) * D + p;
      dst[0] = it == G ? r1 : f2bf(s1);
      dst[PL] = it == G ? r2 : f2bf(s2);
    }
  };
  // One trip to memory for the queries and the wave's first tile, the queries first: vector loads return in order, so behind the
  // tile their sums waited for it. Requests are unconditional (a wave without a tile asks for the block's last one, which another
  // wave reads): where paths with and without them meet, the compiler waits for every load in flight. The tile that the new token
  // goes into is asked for again behind the barrier, by its wave.
  // KL asks for a wave's own tile, once: its pieces go to LDS, in front of whose next access the compiler waits for all that is in
  // flight anyway, and whole pages by waves without a tile, and again behind the barrier, were most of a short context's loads
  // (512 pairs of 12 to 20 / 60 to 100 tokens 18.1 / 18.3 us, now 11.5 / 13.4).
  const int kt_first = min(kt0 + wid_u, kt1 - 1);
  if (rope) {
    request_item(it0);
  } else {
    const int g = fr < G ? fr : 0;
    const bf16_t* qp = a.q + (size_t)b * a.q_stride + (kvh * G + g) * D + 8 * fh;
#pragma unroll
    for (int s = 0; s < C::KS; ++s) qf[s] = *reinterpret_cast<const bf16x8*>(qp + 32 * s);
  }
  __builtin_amdgcn_sched_barrier(0);
  auto request_first = [&]() __attribute__((always_inline)) {
    request_k(kt_first);
    __builtin_amdgcn_sched_barrier(0);  // K before V: the scores and the softmax run while V is landing
    request_v(kt_first);
  };
  // now: asked for in front of the queries' sums; again: behind the append
  auto prologue = [&](bool now, bool again) __attribute__((always_inline)) {
    if (now) request_first();
    __builtin_amdgcn_sched_barrier(0);
    if (!rope) return;
    finish_item(it0);
    for (int i0 = NW * IPW; i0 < n_items; i0 += NW * IPW) {  // block-uniform
      request_item(i0 + it0);
      finish_item(i0 + it0);
    }
    if (append) {
      __syncthreads();  // q in LDS; the appended row visible to every wave of this block (same CU)
      if (again) {
        if constexpr (!REGS && !KL) wait_vmcnt0();  // (into the LDS that its first request fills)
        request_first();
      }
    } else {
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // no LDS access moves to either side
    }
  };
  const bool mine = kt0 + wid_u < kt1, late = append && kt_first == n_kt - 1;
  prologue(!KL || (mine && !late), mine && late);
  if (rope) {
#pragma unroll
    for (int s = 0; s < C::KS; ++s) qf[s] = *reinterpret_cast<const bf16x8*>(s_q + min(fr, G - 1) * D + 32 * s + 8 * fh);
  }
#pragma unroll
  for (int s = 0; s < C::KS; ++s)
    if (fr >= G) qf[s] = (bf16x8){0, 0, 0, 0, 0, 0, 0, 0};
  f32x4 o[C::DT];
#pragma unroll
  for (int dt = 0; dt < C::DT; ++dt) o[dt] = (f32x4){0.f, 0.f, 0.f, 0.f};
  float m_i = -INFINITY, l_i = 0.f;
  unsigned dsink = 0;

  // One tile. MORE: the wave's next one is requested meanwhile (a form of its own: behind a branch around the requests the
  // compiler would wait for them where it waits for this tile's values).
  auto tile = [&](int kt, auto more_t) {
    constexpr bool MORE = decltype(more_t)::value;
    const bool have = kt == kt0 + wid_u;  // requested above
    if constexpr (KL) {
      if (!have) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // previous tile's K / V reads retired
        request_k(kt);
        request_v(kt);
      }
      // K first: QK^T and the softmax run while the V tile (the 16 youngest LDS-DMAs) is still landing. The
      // builtin wait (not inline asm) updates the compiler's own counter model, so it adds no vmcnt(0) of its own.
      static_assert(C::PIECES < 64, "vmcnt range");
      __builtin_amdgcn_s_waitcnt((C::PIECES & 15) | (((C::PIECES >> 4) & 3) << 14) | (0x7 << 4) | (0xF << 8));
#pragma unroll
      for (int t = 0; t < KU / 16; ++t)
#pragma unroll
        for (int s = 0; s < C::KS; ++s) kf[t][s] = load_k<D>(sK, t, s, lane);
    } else if constexpr (DG == 2) {
      const bf16_t* kb = a.kc + page(kt);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      request_v(kt);
      stage_kv<D, false, NT, 1>(sV, 0, 1, lane, [&](int r) { return kb + (size_t)r * D; });
#pragma unroll
      for (int t = 0; t < KU / 16; ++t)
#pragma unroll
        for (int s = 0; s < C::KS; ++s) kf[t][s] = (bf16x8){0, 0, 0, 0, 0, 0, 0, 0};
    } else if (DG == 1 && !have) {
      request_k(kt);
      request_v(kt);
    }
    if constexpr (DG != 0) {
#pragma unroll
      for (int t = 0; t < KU / 16; ++t)
#pragma unroll
        for (int s = 0; s < C::KS; ++s) dsink ^= __builtin_bit_cast(u32x4, kf[t][s])[0];
      if constexpr (REGS) {
#pragma unroll
        for (int i = 0; i < VPC; ++i) dsink ^= vr[i][0];
      } else {
        wait_vmcnt0();
        dsink ^= *reinterpret_cast<const unsigned*>(sV + 4 * lane);
      }
      return;
    }
    f32x4 s4[KU / 16];
#pragma unroll
    for (int t = 0; t < KU / 16; ++t) {
      s4[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < C::KS; ++s) s4[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[t][s], qf[s], s4[t], 0, 0, 0);
    }
    if constexpr (MORE) {  // the next tile's K travels behind this one's softmax and P.V
      __builtin_amdgcn_sched_barrier(0);
      request_k(kt + NW);
      __builtin_amdgcn_sched_barrier(0);
    }
    const int k0 = kt * KU;
    float mx = -INFINITY;
#pragma unroll
    for (int t = 0; t < KU / 16; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int kj = k0 + 16 * t + 4 * fh + r;
        const float x = kj < kv_len ? s4[t][r] * a.scale_log2 : -INFINITY;
        s4[t][r] = x;
        mx = fmaxf(mx, x);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float m_new = fmaxf(m_i, mx);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    // raw v_exp_f32 (the libm exp2f adds a denormal-range fixup per call: ~4 VALU; softmax terms below
    // 2^-126 do not change any fp32 sum here)
    const float alpha = __builtin_amdgcn_exp2f(m_i - m_use);
    float ls = 0.f;
#pragma unroll
    for (int t = 0; t < KU / 16; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float p = __builtin_amdgcn_exp2f(s4[t][r] - m_use);
        s4[t][r] = p;
        ls += p;
      }
    l_i = l_i * alpha + ls;
    m_i = m_new;
#pragma unroll
    for (int dt = 0; dt < C::DT; ++dt) o[dt] *= alpha;
    bf16x8 pb[KU / 32];
#pragma unroll
    for (int ks = 0; ks < KU / 32; ++ks) pb[ks] = pack_p(s4[2 * ks], s4[2 * ks + 1]);
    if constexpr (REGS) {
#pragma unroll
      for (int i = 0; i < VPC; ++i) *reinterpret_cast<u32x4*>(sV + i * 1024 + lane * 16) = vr[i];
      if constexpr (MORE) request_v(kt + NW);
      // (the wave's own LDS accesses stay in order: written above, read below, written again in the next iteration)
    } else {
      __builtin_amdgcn_s_waitcnt((0x7 << 4) | (0xF << 8));  // V tile landed (vmcnt(0), seen by the compiler)
    }
#pragma unroll
    for (int dt = 0; dt < C::DT; ++dt)
#pragma unroll
      for (int ks = 0; ks < KU / 32; ++ks)
        o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(load_vt<D>(sV, dt, ks, lane), pb[ks], o[dt], 0, 0, 0);
  };
  int kt = kt0 + wid_u;
  if constexpr (AHEAD) {
    if (kt < kt1) {
      for (; kt + NW < kt1; kt += NW) tile(kt, std::true_type{});
      tile(kt, std::false_type{});
    }
  } else {
    for (; kt < kt1; kt += NW) tile(kt, std::false_type{});
  }

  if constexpr (DG != 0) {
    if (dsink == 0x9e3779b9u) a.out[(size_t)b * a.out_stride + lane] = 0;  // keeps the loads alive
    return;
  }
  // ---- combine the waves in LDS: each puts its G rows and their statistics where its V tile lay, rows 16 bytes apart in the
  // banks (as 16 rows of D floats behind a barrier, one float a lane, this was 1 us of a block) ----
  constexpr int OS = D + 4, PER = VB / 4;  // floats of a row, of a wave
  static_assert((G * OS + 2 * G) * 4 <= VB, "a wave's rows fit its V tile");
  float* so = reinterpret_cast<float*>(smem);
  if constexpr (!REGS) wait_vmcnt0();  // pieces that no tile waited for
  l_i += __shfl_xor(l_i, 16, 64);
  l_i += __shfl_xor(l_i, 32, 64);
  if (fr < G) {
    float* w = so + wid_u * PER;
#pragma unroll
    for (int dt = 0; dt < C::DT; ++dt) *reinterpret_cast<f32x4*>(w + fr * OS + 16 * dt + 4 * fh) = o[dt];
    if (fh == 0) *reinterpret_cast<float2*>(w + G * OS + 2 * fr) = make_float2(m_i, l_i);
  }
  __syncthreads();
  for (int e = threadIdx.x; e < G * D / 4; e += NTH) {
    const int g = e / (D / 4), d = e % (D / 4) * 4;
    float2 ml[NW];
    f32x4 ov[NW];
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      ml[w] = *reinterpret_cast<const float2*>(so + w * PER + G * OS + 2 * g);
      ov[w] = *reinterpret_cast<const f32x4*>(so + w * PER + g * OS + d);
      M = fmaxf(M, ml[w].x);
    }
    const float Mu = M == -INFINITY ? 0.f : M;
    float L = 0.f;
    f32x4 O = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float sc = exp2f(ml[w].x - Mu);
      L += ml[w].y * sc;
      O += ov[w] * sc;
    }
    const int hq = kvh * G + g;
    if (nparts == 1) {
      if (!(L > 0.f)) O = (f32x4){0.f, 0.f, 0.f, 0.f}, L = 1.f;
      *reinterpret_cast<u32x2_a2*>(a.out + (size_t)b * a.out_stride + hq * D + d) =
          (u32x2_a2){pk2bf(O[0] / L, O[1] / L), pk2bf(O[2] / L, O[3] / L)};
    } else {
      const size_t pi = ((size_t)b * a.Hq + hq) * a.max_parts + part;
      *reinterpret_cast<f32x4_a4*>(a.part_o + pi * D + d) = O;
      if (d == 0) *reinterpret_cast<f32x2_a4*>(a.part_ml + pi * 2) = (f32x2_a4){M, L};
    }
  }
}

template <int D, int G, bool NT = false, int NW = 4, int DG = 0, bool KL = false>
__global__ __launch_bounds__(NW * 64, (NW == 4 && !KL) ? 2 : 1) void attn_decode_kernel(DecodeArgs a) {
  __shared__ __attribute__((aligned(16))) char smem[decode_lds_bytes<D, G, NW, KL, DG>()];
  attn_decode_block<D, G, NT, NW, DG, KL>(a, blockIdx.z, blockIdx.x, blockIdx.y, smem);
}

// merge split-K partitions: grid (Hq, B), block D threads (join_parts)
constexpr int RED_MAXP = 256;  // most partitions of a sequence
__global__ void attn_decode_reduce_kernel(DecodeArgs a, int D) {
  const int hq = blockIdx.x, b = blockIdx.y, t = threadIdx.x;
  const size_t p0 = ((size_t)b * a.Hq + hq) * a.max_parts;
  int nparts = 0;
  const float2 r = join_parts(
      a.part_ml + p0 * 2, a.part_o + p0 * D, D, a.max_parts, t, false,
      [&] {
        const int n = (a.kv_lens[b] + DEC_U - 1) / DEC_U, pt = decode_part_units(n, a);
        return nparts = (n + pt - 1) / pt;
      },
      [](float x) { return exp2f(x); });
  if (nparts <= 1) return;  // the partition kernel wrote the output itself
  a.out[(size_t)b * a.out_stride + hq * D + t] = f2bf(r.y > 0.f ? r.x / r.y : 0.f);
}

// Block order (prefill_block): a 1-D grid, head group fastest, so the heaviest causal tiles of every head
// start first and consecutive blocks (round-robin over the XCDs) put one KV head on each XCD.
// Kernel per config:
//   * Llama (D 128, 4 query heads per KV head, causal, paged cache < 4 GiB): the software-pipelined
//     8-wave kernel with the whole-row LDS epilogue (attn_prefill_v3_kernel<8, ..., WIDE>; 64-query
//     tiles), tools/attn_pp_ab.py; few blocks: its 4-wave form, two blocks a tile (V3_HALF);
//   * every other 4-heads-per-block config: attn_prefill_kernel with 8 waves (64-query tiles, two 32-row
//     groups sharing each K/V tile);
//   * 1 or 2 heads per block (encoders, GPT-2, odd GQA ratios): the 4-wave attn_prefill_kernel.
// Up to this many 64-query blocks the pipelined kernel runs as twice as many of 32 queries: with CUs to spare, a wave that has its
// SIMD to itself takes a key tile faster than two that share it. 32 query heads over 8, one prompt, us: 64 tokens 7.8 -> 6.8, 300
// 13.7 -> 11.7, 700 22.2 -> 18.3, 1000 (128 blocks) 29.3 -> 24.8; 16 heads over 4, 2000 tokens 49.3 -> 40.3; 3 of 300 15.0 -> 12.8.
// Past 128 blocks the halves no longer fit one round: 10 prompts of 100 tokens (160 blocks) 10.5 against 13.4, one of 1300 (168)
// 36.5 against 30.9; the entry does not know which it has.
constexpr unsigned V3_HALF = 128;
template <int D, int GB, bool CAUSAL, bool PAGED>
hipError_t launch_prefill(PrefillArgs a, int n_tiles, hipStream_t st) {
  const int G = a.Hq / a.Hkv;
  const int n_hg = a.Hkv * (G / GB);
  a.n_hg = n_hg;
  const dim3 grid(n_tiles * n_hg);
  if constexpr (D == 128 && GB == 4 && CAUSAL && PAGED) {
    if (a.kv_bytes) {
      if (grid.x <= V3_HALF) {
        hipLaunchKernelGGL((attn_prefill_v3_kernel<4, false, 0, 0, true>), dim3(grid.x, 2), dim3(256), 0, st, a);
        return hipGetLastError();
      }
      hipLaunchKernelGGL((attn_prefill_v3_kernel<8, false, 0, 1, true>), grid, dim3(512), 0, st, a);
      return hipGetLastError();
    }
  }
  if constexpr (!CAUSAL && !PAGED && GB == 1 && D <= 64) {
    // rows on 16 bytes, a tile's 64 within 31-bit offsets
    if (G == 1 && ((uintptr_t)a.k | (uintptr_t)a.v) % 16 == 0 && a.kv_stride % 8 == 0 && a.kv_stride < 1 << 24) {
      hipLaunchKernelGGL((attn_encoder_kernel<D>), grid, dim3(256), 0, st, a);
      return hipGetLastError();
    }
  }
  if constexpr (GB == 4)
    hipLaunchKernelGGL((attn_prefill_kernel<D, GB, CAUSAL, PAGED, false, 8>), grid, dim3(512), 0, st, a);
  else
    hipLaunchKernelGGL((attn_prefill_kernel<D, GB, CAUSAL, PAGED>), grid, dim3(256), 0, st, a);
  return hipGetLastError();
}

}  // namespace

// Query rows per block (the host builds `tiles` with this step): 64 for 4 heads per block, else 128 / GB.
RAGK_API int ragk_attn_prefill_qtile(int Hq, int Hkv) {
  const int G = Hq / Hkv;
  const int GB = G % 4 == 0 ? 4 : (G % 2 == 0 ? 2 : 1);
  return 32 * ((GB == 4 ? 8 : 4) / GB);
}

RAGK_API int ragk_attn_prefill(const void* q, int q_stride, const void* k, const void* v, int kv_stride,
                               const int* block_tables, int bt_stride, const int* cu_q, const int* cu_kv,
                               const int* kv_lens, const int* tiles, int n_tiles, void* out, int out_stride,
                               int Hq, int Hkv, int D, int causal, int paged, float scale, hipStream_t st) {
  if (n_tiles <= 0) return 0;
  if (Hq % Hkv) return (int)hipErrorInvalidValue;
  // paged: kv_stride = number of cache blocks (sizes the buffer descriptors of the BUF staging)
  const unsigned long long cache_bytes = paged ? (unsigned long long)kv_stride * Hkv * KT * D * 2 : 0ull;
  PrefillArgs a{(const bf16_t*)q, q_stride, (const bf16_t*)k, (const bf16_t*)v, kv_stride, block_tables, bt_stride,
                cu_q, cu_kv, kv_lens, tiles, (bf16_t*)out, out_stride, Hq, Hkv, scale * 1.4426950408889634f,
                cache_bytes < (1ull << 32) ? (unsigned)cache_bytes : 0u, 0};
  const int G = Hq / Hkv;
  const int GB = G % 4 == 0 ? 4 : (G % 2 == 0 ? 2 : 1);
#define RAGK_PF(DD, GG, CC, PP)                                                          \
  if (D == DD && GB == GG && (bool)causal == CC && (bool)paged == PP)                      \
    return (int)launch_prefill<DD, GG, CC, PP>(a, n_tiles, st);
  RAGK_PF(128, 4, true, true)
  RAGK_PF(128, 1, true, true)
  RAGK_PF(128, 2, true, true)
  RAGK_PF(64, 1, true, true)
  RAGK_PF(64, 4, true, true)
  RAGK_PF(128, 4, true, false)
  RAGK_PF(64, 1, false, false)
  RAGK_PF(32, 1, false, false)
  RAGK_PF(128, 1, false, false)
  RAGK_PF(64, 1, true, false)
#undef RAGK_PF
  return (int)hipErrorInvalidValue;
}


// K/V cache-policy switch for decode (0 = default, 1 = non-temporal loads; the KV stream is read
// once per step). A/B in tools/bench_kernels.py --quick.
static int g_decode_nt = 0;
// 8-wave single-partition decode attention once batch x KV heads reaches this (0 = never)
static int g_decode_nw8_min = 0;
// diagnostic instantiation of the 8-wave kernel (DG above; A/B tooling only, 0 = off)
static int g_decode_diag = 0;
// single-partition grid on 4-wave blocks with K tiles by LDS-DMA (KL above; 0 = the 8-wave kernel)
static int g_decode_kl = 0;
RAGK_API int ragk_attn_decode_set_kl(int on) {
  g_decode_kl = on ? 1 : 0;
  return 0;
}
RAGK_API int ragk_attn_decode_set_diag(int dg) {
  g_decode_diag = (dg == 1 || dg == 2) ? dg : 0;
  return 0;
}
RAGK_API int ragk_attn_decode_set_nw8(int min_pairs) {
  g_decode_nw8_min = min_pairs > 0 ? min_pairs : 0;
  return 0;
}
RAGK_API int ragk_attn_decode_set_nt(int nt) {
  g_decode_nt = nt ? 1 : 0;
  return 0;
}

static int launch_attn_decode(DecodeArgs a, int B, int D, int max_parts, hipStream_t st);

// Deferred merge: the next decode-attention launches leave the split-K partitions unmerged (no
// attn_decode_reduce launch) for a consumer that merges them itself (gemm_part.hip MergeArgs: the
// o_proj GEMM). The host sets it around one launch.
static int g_decode_defer = 0;
RAGK_API int ragk_attn_decode_set_defer(int on) {
  g_decode_defer = on ? 1 : 0;
  return 0;
}

RAGK_API int ragk_attn_decode(const void* q, int q_stride, const void* kc, const void* vc, const int* block_tables,
                              int bt_stride, int bt_cols, const int* kv_lens, float* part_o, float* part_ml, void* out,
                              int out_stride, int B, int Hq, int Hkv, int D, int part_tiles, int max_parts,
                              float scale, hipStream_t st) {
  if (B <= 0) return 0;
  if (Hq % Hkv || part_tiles < 1 || max_parts < 1 || max_parts > RED_MAXP) return (int)hipErrorInvalidValue;
  DecodeArgs a{(const bf16_t*)q, q_stride, (const bf16_t*)kc, (const bf16_t*)vc, block_tables, bt_stride, bt_cols, kv_lens,
               part_o, part_ml, (bf16_t*)out, out_stride, Hq, Hkv, part_tiles, max_parts,
               scale * 1.4426950408889634f};
  return launch_attn_decode(a, B, D, max_parts, st);
}

// Decode attention fed by the qkv projection's split-K partial slabs P[S][B][ldp] (gemm_part.hip):
// RoPE of q and k, the KV append at slots[b] and the attention in one launch (replaces
// rope_kv_partials + attn_decode). Cache blocks hold KT tokens.
RAGK_API int ragk_attn_decode_rope(const float* P, int S, int ldp, const int* positions, const int* slots,
                                   const float* cos_t, const float* sin_t, void* kc, void* vc,
                                   const int* block_tables, int bt_stride, int bt_cols, const int* kv_lens, float* part_o,
                                   float* part_ml, void* out, int out_stride, int B, int Hq, int Hkv, int D,
                                   int part_tiles, int max_parts, float scale, hipStream_t st) {
  if (B <= 0) return 0;
  if (Hq % Hkv || part_tiles < 1 || max_parts < 1 || max_parts > RED_MAXP || S < 1 || D % 64 ||
      ldp < (Hq + 2 * Hkv) * D || !P || !positions || !slots || !cos_t || !sin_t)
    return (int)hipErrorInvalidValue;
  DecodeArgs a{nullptr, 0, (const bf16_t*)kc, (const bf16_t*)vc, block_tables, bt_stride, bt_cols, kv_lens,
               part_o, part_ml, (bf16_t*)out, out_stride, Hq, Hkv, part_tiles, max_parts,
               scale * 1.4426950408889634f, P, (long long)B * ldp, ldp, S, positions, slots, cos_t, sin_t};
  return launch_attn_decode(a, B, D, max_parts, st);
}

static int launch_attn_decode(DecodeArgs a, int B, int D, int max_parts, hipStream_t st) {
  const int Hq = a.Hq, Hkv = a.Hkv;
  const int G = Hq / Hkv;
  // Partitions vary slowest: a context shorter than the longest allowed fills only the first ones, and so the blocks with work
  // come first and spread evenly over XCDs and CUs. With the partitions fastest they fell where the grid's width put them, at 8
  // partitions on two XCDs of eight (2 KV heads, 30 sequences of 300 tokens in 8 partitions 17.0 us, in 9 12.7; now 12.0).
  // Decode steps of four Llama layers, us: 4 / 8 rows of 4096 / 2000 tokens, 4 KV heads, 268 / 260 -> 256 / 246; where 512 blocks
  // are all at work they take 1 % more (8 rows of 4096 tokens, 8 KV heads: 537 -> 543).
  dim3 grid(Hkv, B, max_parts);
  if (D == 128 && G == 4 && max_parts == 1 && g_decode_nw8_min > 0 && B * Hkv >= g_decode_nw8_min) {
    // one partition per sequence over >= 1 block per CU: 8-wave blocks, no merge launch
    if (g_decode_kl && !g_decode_diag)
      hipLaunchKernelGGL((attn_decode_kernel<128, 4, true, 4, 0, true>), grid, dim3(256), 0, st, a);
    else if (g_decode_diag == 1)
      hipLaunchKernelGGL((attn_decode_kernel<128, 4, true, 8, 1>), grid, dim3(512), 0, st, a);
    else if (g_decode_diag == 2)
      hipLaunchKernelGGL((attn_decode_kernel<128, 4, true, 8, 2>), grid, dim3(512), 0, st, a);
    else if (g_decode_nt)
      hipLaunchKernelGGL((attn_decode_kernel<128, 4, true, 8>), grid, dim3(512), 0, st, a);
    else
      hipLaunchKernelGGL((attn_decode_kernel<128, 4, false, 8>), grid, dim3(512), 0, st, a);
    return (int)hipGetLastError();
  }
#define RAGK_DC(DD, GG)                                                            \
  if (D == DD && G == GG) {                                                          \
    if (g_decode_nt)                                                                 \
      hipLaunchKernelGGL((attn_decode_kernel<DD, GG, true>), grid, dim3(256), 0, st, a); \
    else                                                                             \
      hipLaunchKernelGGL((attn_decode_kernel<DD, GG, false>), grid, dim3(256), 0, st, a); \
    if (max_parts > 1 && !g_decode_defer)                                            \
      hipLaunchKernelGGL(attn_decode_reduce_kernel, dim3(Hq, B), dim3(DD), 0, st, a, DD); \
    return (int)hipGetLastError();                                                   \
  }
  RAGK_DC(128, 4)
  RAGK_DC(128, 8)
  RAGK_DC(128, 1)
  RAGK_DC(64, 1)
  RAGK_DC(64, 4)
  RAGK_DC(128, 2)
#undef RAGK_DC
  return (int)hipErrorInvalidValue;
}

