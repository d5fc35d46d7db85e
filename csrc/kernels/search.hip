// Exact squared-L2 k-nearest-neighbour search for gfx950 (faiss IndexFlatL2
// semantics: squared distances, ascending, ties -> lower id, missing results = (-1, FLT_MAX)).
// Reference: faiss index.search at /root/reference/llm/rag.py:116.
//
// The database stays resident in HBM in a COLUMN-major layout xt[d][cap] (cap = row
// capacity): lane l of a wave reads row r0 + l of one dimension per load, 256 contiguous
// bytes per wave instruction, no LDS for the data. Queries come by scalar loads. Distances are sum((x - q)^2) in fp32 (faiss' exact path).
//
// Top-k without sorting the scanned rows: every wave keeps a RUNNING sorted top-64 list per
// query in its lanes (lane j = j-th best). A tile of 64 fresh distances (one per lane) is
// skipped outright when none beats the current k-th best (after the first few tiles almost
// all of them); otherwise it is bitonic-sorted across the lanes (21 shuffle steps) and merged
// into the running list (min against the reversed list + 6 bitonic-merge steps).
//   l2_scan:   grid (row-tile groups, query groups); each block loops over its row tiles and
//              emits one sorted top-k per query -> partial lists [nq][G][k]
//   ivf_scan:  the same per (query, probe): the probed inverted list's row range
//   topk_lists_merge: one block per query merges the G sorted lists with the same wave
//              machinery (64 candidates per step, skip test first).
// Small indexes split each row tile's dimensions over S waves (S = 4 below 64k rows) so that
// a 10k-row index still spreads over ~160 blocks; the partial sums are added in slice order.
#include <chrono>
#include <climits>
#include "common.h"
#include <float.h>
using namespace ragk;

namespace {

constexpr int ST = 256;   // threads per block (4 waves)
constexpr int DCH = 256;  // dims that the slices of a row tile split between them at a time
constexpr int UNR = 16;   // dims (independent loads) in flight per lane

// wave_offer for QB queries at once (the same 64 rows, one candidate per lane and query): the QB
// bitonic networks run interleaved step by step, so the cross-lane permutes of one query's
// dependent chain hide behind the others' (one query at a time left a 16-query block
// latency-bound on ~28 dependent permute round trips per query). Skipped outright when no query's
// candidates beat its current k-th best.
template <int QB>
__device__ __forceinline__ void wave_offer_q(float (&bv)[QB], int (&bi)[QB], float (&v)[QB], int id, int nqb, int k,
                                             int lane) {
  bool any = false;
#pragma unroll
  for (int q = 0; q < QB; ++q) {
    if (q < nqb) {
      const float tv = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(bv[q]), k - 1));
      const int ti = __builtin_amdgcn_readlane(bi[q], k - 1);
      any |= __any(cand_lt(v[q], id, tv, ti));
    }
  }
  if (!any) return;  // wave-uniform
  int ix[QB];
#pragma unroll
  for (int q = 0; q < QB; ++q) ix[q] = id;
#pragma unroll
  for (int kk = 2; kk <= 64; kk <<= 1)
#pragma unroll
    for (int j = kk >> 1; j > 0; j >>= 1)
#pragma unroll
      for (int q = 0; q < QB; ++q) cx(v[q], ix[q], lane, j, (lane & kk) == 0);
#pragma unroll
  for (int q = 0; q < QB; ++q) {
    const float rv = rev_lane(v[q], lane);
    const int ri = rev_lane(ix[q], lane);
    if (cand_lt(rv, ri, bv[q], bi[q])) {
      bv[q] = rv;
      bi[q] = ri;
    }
  }
#pragma unroll
  for (int j = 32; j > 0; j >>= 1)
#pragma unroll
    for (int q = 0; q < QB; ++q) cx(bv[q], bi[q], lane, j, true);
}

// As wave_offer_q with a separate candidate id per query (lists of different queries).
template <int NQ>
__device__ __forceinline__ void wave_offer_multi(float (&bv)[NQ], int (&bi)[NQ], float (&v)[NQ], int (&ix)[NQ], int k,
                                                 int lane) {
  bool any = false;
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    const float tv = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(bv[q]), k - 1));
    const int ti = __builtin_amdgcn_readlane(bi[q], k - 1);
    any |= __any(cand_lt(v[q], ix[q], tv, ti));
  }
  if (!any) return;
#pragma unroll
  for (int kk = 2; kk <= 64; kk <<= 1)
#pragma unroll
    for (int j = kk >> 1; j > 0; j >>= 1)
#pragma unroll
      for (int q = 0; q < NQ; ++q) cx(v[q], ix[q], lane, j, (lane & kk) == 0);
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    const float rv = rev_lane(v[q], lane);
    const int ri = rev_lane(ix[q], lane);
    if (cand_lt(rv, ri, bv[q], bi[q])) {
      bv[q] = rv;
      bi[q] = ri;
    }
  }
#pragma unroll
  for (int j = 32; j > 0; j >>= 1)
#pragma unroll
    for (int q = 0; q < NQ; ++q) cx(bv[q], bi[q], lane, j, true);
}

// Distances of 64 rows (one per lane, at xt + rc) over dims [t0, t1) for QB queries, whose values are wave-uniform: they come
// by scalar loads (qp[j] = query j, or the last one past the batch), so no LDS, staging or barrier stands between the loads
// of the rows. U dims in flight.
template <int QB, int U = (QB <= 2 ? 32 : QB <= 4 ? 16 : 8)>
__device__ __forceinline__ void scan_dims(const float* __restrict__ xt, size_t cap, int rc, int t0, int t1,
                                          const float* const (&qp)[QB], float* acc) {
  const float* col = xt + (size_t)t0 * cap + rc;
  int t = t0;
  for (; t + U <= t1; t += U, col += U * cap) {
    float x[U];
#pragma unroll
    for (int u = 0; u < U; ++u) x[u] = col[(size_t)u * cap];
#pragma unroll
    for (int j = 0; j < QB; ++j) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const float df = x[u] - qp[j][t + u];
        acc[j] = fmaf(df, df, acc[j]);
      }
    }
  }
  for (; t < t1; ++t, col += cap) {
    const float x = *col;
#pragma unroll
    for (int j = 0; j < QB; ++j) {
      const float df = x - qp[j][t];
      acc[j] = fmaf(df, df, acc[j]);
    }
  }
}

// Flat scan. Row tile = 64 * (4 / S) rows: wave w scans rows 64 * (w / S) .. +63 of the tile over
// dim slice w % S of every 256-dim chunk. Block bx of G handles tiles bx, bx + G, ...; its
// queries are q0 = blockIdx.y * QB .. + QB. Output: per query one sorted list of k at [q][bx].
// Grid (8, query groups, ceil(G / 8)): workgroups go to the XCDs in turn, so the groups that read the same rows are
// neighbours on one XCD and all but the first find them in its L2: 13 queries of 500000 x 1024 take 528 us, as grid (G, query
// groups), where each group streams the index from HBM, 724. (Before, with the queries' chunks staged in LDS: 8 queries 710 us
// and now 408, 13 queries 1032, 32 queries of k = 10 1340 and now 901; 8 of 10000 x 1024: 71 and 37, launches included.)
template <int QB, int S>
__global__ __launch_bounds__(ST) void l2_scan_kernel(const float* __restrict__ xt, int cap, int d, int row_begin,
                                                     int row_end, int ntiles, const float* __restrict__ q, int nq,
                                                     int k, float* __restrict__ out_d, int* __restrict__ out_i,
                                                     const int* __restrict__ ids_map, int G) {
  constexpr int RG = 4 / S;
  constexpr int RB = 64 * RG;
  const int bx = blockIdx.z * 8 + blockIdx.x;
  if (bx >= G) return;
  extern __shared__ __attribute__((aligned(16))) float sc_smem[];
  float* red = sc_smem;  // [S - 1][RG][QB][64]
  __shared__ float mv[4][64];
  __shared__ int mi[4][64];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = w / S, s = w % S;
  const int q0 = blockIdx.y * QB;
  const int nqb = min(QB, nq - q0);
  const float* qp[QB];
#pragma unroll
  for (int j = 0; j < QB; ++j) qp[j] = q + (size_t)(q0 + min(j, nqb - 1)) * d;
  float bv[QB];
  int bi[QB];
#pragma unroll
  for (int j = 0; j < QB; ++j) {
    bv[j] = FLT_MAX;
    bi[j] = -1;
  }
  for (int tile = bx; tile < ntiles; tile += G) {
    const int row = row_begin + tile * RB + 64 * g + lane;
    const int rc = min(row, cap - 1);  // rows in [row_end, cap) are valid memory; masked below
    float acc[QB];
#pragma unroll
    for (int j = 0; j < QB; ++j) acc[j] = 0.f;
    for (int dc = 0; dc < d; dc += DCH) {
      const int dn = min(DCH, d - dc);
      const int per = (dn + S - 1) / S;
      const int t0 = min(dn, s * per), t1 = min(dn, t0 + per);
      scan_dims<QB>(xt, (size_t)cap, rc, dc + t0, dc + t1, qp, acc);
    }
    if (S > 1) {
      __syncthreads();  // the previous tile's slices are summed
      if (s > 0) {
#pragma unroll
        for (int j = 0; j < QB; ++j) red[(((s - 1) * RG + g) * QB + j) * 64 + lane] = acc[j];
      }
      __syncthreads();
      if (s == 0) {
#pragma unroll
        for (int ss = 1; ss < S; ++ss)
#pragma unroll
          for (int j = 0; j < QB; ++j) acc[j] += red[(((ss - 1) * RG + g) * QB + j) * 64 + lane];
      }
    }
    if (s == 0) {  // wave-uniform
      const bool ok = row < row_end;
      const int id = ok ? (ids_map ? ids_map[row] : row) : -1;
#pragma unroll
      for (int j = 0; j < QB; ++j) acc[j] = (ok && j < nqb) ? acc[j] : FLT_MAX;
      wave_offer_q<QB>(bv, bi, acc, ok ? id : -1, nqb, k, lane);
    }
  }
  // block merge: the RG list-holding waves (s == 0) -> wave 0 -> k outputs per query
#pragma unroll
  for (int j = 0; j < QB; ++j) {
    if (j >= nqb) continue;  // block-uniform
    if (RG > 1) {
      __syncthreads();
      if (s == 0 && g > 0) {
        mv[g][lane] = bv[j];
        mi[g][lane] = bi[j];
      }
      __syncthreads();
      if (w == 0)
        for (int gg = 1; gg < RG; ++gg) wave_merge64(bv[j], bi[j], mv[gg][lane], mi[gg][lane], lane);
    }
    if (w == 0 && lane < k) {
      const size_t o = ((size_t)(q0 + j) * G + bx) * k + lane;
      out_d[o] = bv[j];
      out_i[o] = bi[j];
    }
  }
}

// Batched queries (nq >= 16: the BLAS path of faiss' IndexFlatL2): ||x||^2 + ||q||^2 - 2 x.q with the
// dot products on the exact fp32-input MFMA (v_mfma_f32_16x16x4_f32: a k-ordered fmaf chain), 16 rows x
// 16 queries per instruction, QT query tiles of 16 (all of a <= 32-query batch in one block: the index is streamed
// from HBM once).
//
// The stream bounds it (32 queries: 209 us of MFMA for the 2 GB that take 360 us to read), so nothing may stand between
// a wave and its next loads: the whole q^T lies in LDS (up to 128 KB, one block of 8 waves a CU), staged once, and each
// wave walks its own tiles of 16 * RT rows without a barrier, three groups of loads deep. Row RT m + rt of a tile is row m
// of MFMA rt, so the A operands of the RT MFMAs are one load of RT consecutive rows of a dimension: 16 B a lane at RT = 4.
// (Before: 4-wave blocks that staged q^T in chunks of 256 dims for every 256 rows, 4-B loads.)
// 32 queries, 500000 x 1024: 606 -> 387 us; 100000 x 1024: 250 -> 124; 10000 x 384: 40 -> 29 (launches included).
//
// Lane l of a wave holds x[rows][k0 + (l >> 4)] (A fragment), reads q^T[k0 + (l >> 4)][16 qt + (l & 15)] (B fragment), and
// its accumulators hold MFMA rows 4 (l >> 4) + r of query 16 qt + (l & 15).
// Selection: every lane keeps a sorted list of the MK best (distance, id) of its query among the rows it sees
// (MK >= k); the four lanes of a query merge theirs, then the block its waves' -> one sorted list of k per query.
// Distances clamp at 0 like faiss.
constexpr int MQ_MK = 8;   // k <= 8 on this path
constexpr int MQ_KU = 4;   // k-steps (of 4 dims) per group of loads
constexpr int MQ_DMAX = 1024;
constexpr int MQ_NW = 8;   // waves of a block
constexpr int MQ_CAND = MQ_NW * MQ_MK;  // candidates of a query at the block's merge: one a lane
static_assert(MQ_CAND == 64, "one wave merges a query");

// LDS floats: q^T during the scan, the candidates (values, ids) at the merge; then ||q||^2 and the waves' ||x||^2
__host__ __device__ inline int mq_region0(int d, int QT) { return max(d * 16 * QT, 2 * 16 * QT * MQ_CAND); }
__host__ __device__ inline int mq_floats(int d, int QT) { return mq_region0(d, QT) + 16 * QT + MQ_NW * 64; }

template <int QT, int RT>
__global__ __launch_bounds__(MQ_NW * 64, 2) void l2_mfma_kernel(const float* __restrict__ xt, int cap, int d, int row_begin,
                                                             int row_end, int ntiles, const float* __restrict__ q, int nq,
                                                             int k, float* __restrict__ out_d, int* __restrict__ out_i,
                                                             const int* __restrict__ ids_map) {
  constexpr int NQ = 16 * QT, TH = MQ_NW * 64;
  // RT consecutive rows of a dimension; only 4-byte aligned (cap and row_begin are arbitrary)
  struct __attribute__((packed, aligned(4))) Rows { float v[RT]; };
  extern __shared__ __attribute__((aligned(16))) float mq_smem[];
  float* qsT = mq_smem;                              // [d][16][QT]
  float* cd = mq_smem;                               // [NQ][MQ_CAND] candidates (merge, aliases qsT)
  int* ci = reinterpret_cast<int*>(mq_smem + NQ * MQ_CAND);
  float* qn = mq_smem + mq_region0(d, QT);           // [NQ] ||q||^2
  float* xnl = qn + NQ;                              // [waves][64] ||x||^2 of the wave's rows
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int q0 = blockIdx.y * NQ;
  const int nqb = min(NQ, nq - q0);
  // consecutive threads take consecutive queries, so the transposed LDS words they write are consecutive; eight loads a
  // thread in flight
  struct __attribute__((packed, aligned(4))) Quad { float v[4]; };
  const int quads = NQ * (d >> 2);
  for (int e0 = threadIdx.x; e0 < quads; e0 += 8 * TH) {
    Quad v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int e = min(e0 + u * TH, quads - 1);
      v[u] = *reinterpret_cast<const Quad*>(q + (size_t)(q0 + min(e % NQ, nqb - 1)) * d + (e / NQ) * 4);
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int e = e0 + u * TH;
      if (e < quads) {
        const int j = e % NQ, t = (e / NQ) * 4;
#pragma unroll
        for (int i = 0; i < 4; ++i) qsT[(t + i) * NQ + (j & 15) * QT + (j >> 4)] = j < nqb ? v[u].v[i] : 0.f;
      }
    }
  }
  __syncthreads();
  {
    // ||q||^2: thread (part p, word j) sums dims p, p + P, ...; the parts are added in order
    constexpr int P = TH / NQ;
    const int j = threadIdx.x % NQ, p = threadIdx.x / NQ;
    float sq = 0.f;
#pragma unroll 8
    for (int t = p; t < d; t += P) sq = fmaf(qsT[t * NQ + j], qsT[t * NQ + j], sq);
    xnl[p * NQ + j] = sq;  // TH floats
    __syncthreads();
    if (p == 0) {
      for (int o = 1; o < P; ++o) sq += xnl[o * NQ + j];
      qn[(j % QT) * 16 + j / QT] = sq;
    }
  }
  __syncthreads();
  const int fr = lane & 15, fg = lane >> 4;
  // per-lane sorted lists, one per query tile
  float lv[QT][MQ_MK];
  int lix[QT][MQ_MK];
#pragma unroll
  for (int qt = 0; qt < QT; ++qt)
#pragma unroll
    for (int m = 0; m < MQ_MK; ++m) {
      lv[qt][m] = FLT_MAX;
      lix[qt][m] = -1;
    }
  float qnv[QT];
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) qnv[qt] = qn[16 * qt + fr];
  const float* qb = qsT + fg * NQ + fr * QT;
  float* xw = xnl + 64 * w;
  for (int tile = w * gridDim.x + blockIdx.x; tile < ntiles; tile += MQ_NW * gridDim.x) {
    const int first = row_begin + tile * 16 * RT;
    // a tile over the store's end moves back (the rows of the tile before it are masked below), so that it loads like any
    const int rbase = max(0, min(first, cap - 16 * RT));
    f32x4 acc[RT][QT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int qt = 0; qt < QT; ++qt) acc[rt][qt] = f32x4{0.f, 0.f, 0.f, 0.f};
    float xs[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) xs[rt] = 0.f;
    const int nk = d / 4;  // multiple of MQ_KU
    auto mma = [&](int t, const Rows& a) __attribute__((always_inline)) {  // k-step t
      float b[QT];
#pragma unroll
      for (int qt = 0; qt < QT; ++qt) b[qt] = qb[4 * t * NQ + qt];
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        xs[rt] = fmaf(a.v[rt], a.v[rt], xs[rt]);
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) acc[rt][qt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.v[rt], b[qt], acc[rt][qt], 0, 0, 0);
      }
    };
    if (rbase + 16 * RT <= cap) {
      const float* col = xt + (size_t)fg * cap + rbase + RT * fr;
      auto load_grp = [&](Rows (&a)[MQ_KU]) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < MQ_KU; ++u) {
          a[u] = *reinterpret_cast<const Rows*>(col);
          col += (size_t)4 * cap;
        }
      };
      auto mma_grp = [&](int k0, const Rows (&a)[MQ_KU]) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < MQ_KU; ++u) mma(k0 + u, a[u]);
      };
      // four register buffers, refilled as soon as their MFMAs are issued (a group's take 0.4 us, the other wave of the SIMD
      // as long): three groups in flight
      constexpr int NB = 4;
      Rows a[NB][MQ_KU];
#pragma unroll
      for (int i = 0; i < NB; ++i)
        if (i * MQ_KU < nk) load_grp(a[i]);
#pragma unroll 1
      for (int k0 = 0; k0 < nk; k0 += NB * MQ_KU) {
#pragma unroll
        for (int i = 0; i < NB; ++i) {
          if (k0 + i * MQ_KU >= nk) break;
          mma_grp(k0 + i * MQ_KU, a[i]);
          if (k0 + (i + NB) * MQ_KU < nk) load_grp(a[i]);
        }
      }
    } else {  // a store smaller than a tile: one row at a time, clamped
#pragma unroll 1
      for (int t = 0; t < nk; ++t) {
        Rows a;
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) a.v[rt] = xt[(size_t)(4 * t + fg) * cap + min(rbase + RT * fr + rt, cap - 1)];
        mma(t, a);
      }
    }
    // ||x||^2 of row RT fr + rt: the 4 dim phases (lanes fr, fr+16, fr+32, fr+48) summed in order
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      float t = xs[rt];
      t += __int_as_float(xor_lane(__float_as_int(t), 16, lane));
      t += __int_as_float(xor_lane(__float_as_int(t), 32, lane));
      if (fg == 0) xw[RT * fr + rt] = t;
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave's xnl writes landed (wave-local rows)
    __builtin_amdgcn_wave_barrier();
    // a lane's rows in ascending order: without a map of ids an equal distance stays behind the ones already listed, and
    // an insertion is one median a slot (l'[m] = med3(l[m - 1], l[m], c)) instead of a chain of compare-exchanges
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        const int rl = RT * (4 * fg + r) + rt;
        const int row = rbase + rl;
        const bool ok = row >= first && row < row_end;
        const int id = ok ? (ids_map ? ids_map[row] : row) : -1;
        const float xn = xw[rl];
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) {
          const float dv = ok ? fmaxf(xn + qnv[qt] - 2.f * acc[rt][qt][r], 0.f) : FLT_MAX;
          if (!ids_map) {
            if (dv < lv[qt][MQ_MK - 1]) {
#pragma unroll
              for (int m = MQ_MK - 1; m >= 0; --m) {
                const bool here = dv < lv[qt][m], before = m > 0 && dv < lv[qt][m > 0 ? m - 1 : 0];
                lix[qt][m] = before ? lix[qt][m > 0 ? m - 1 : 0] : (here ? id : lix[qt][m]);
                lv[qt][m] = m > 0 ? __builtin_amdgcn_fmed3f(lv[qt][m > 0 ? m - 1 : 0], lv[qt][m], dv) : fminf(lv[qt][0], dv);
              }
            }
          } else if (cand_lt(dv, id, lv[qt][MQ_MK - 1], lix[qt][MQ_MK - 1])) {
            float cv = dv;
            int cidx = id;
#pragma unroll
            for (int m = 0; m < MQ_MK; ++m) {
              if (cand_lt(cv, cidx, lv[qt][m], lix[qt][m])) {
                const float tv = lv[qt][m];
                const int ti = lix[qt][m];
                lv[qt][m] = cv;
                lix[qt][m] = cidx;
                cv = tv;
                cidx = ti;
              }
            }
          }
        }
      }
    __builtin_amdgcn_wave_barrier();
  }
  // a query's four lanes (fr, fr + 16, + 32, + 48) emit the best MK of their lists in order: the smallest head goes out,
  // its lane moves on
  __syncthreads();  // every wave is done reading q^T: the candidates reuse its LDS
#pragma unroll
  for (int m = 0; m < MQ_MK; ++m)
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      float mv = lv[qt][0];
      int mi = lix[qt][0];
#pragma unroll
      for (int jx = 16; jx < 64; jx <<= 1) {
        const float ov = __int_as_float(xor_lane(__float_as_int(mv), jx, lane));
        const int oi = xor_lane(mi, jx, lane);
        const bool take = cand_lt(ov, oi, mv, mi);
        mv = take ? ov : mv;
        mi = take ? oi : mi;
      }
      const bool won = (lv[qt][0] == mv) & (lix[qt][0] == mi);
#pragma unroll
      for (int n = 0; n < MQ_MK; ++n) {
        lv[qt][n] = won ? (n + 1 < MQ_MK ? lv[qt][n + 1] : FLT_MAX) : lv[qt][n];
        lix[qt][n] = won ? (n + 1 < MQ_MK ? lix[qt][n + 1] : -1) : lix[qt][n];
      }
      if (fg == 0) {
        cd[(16 * qt + fr) * MQ_CAND + w * MQ_MK + m] = mv;
        ci[(16 * qt + fr) * MQ_CAND + w * MQ_MK + m] = mi;
      }
    }
  __syncthreads();
  // a wave merges queries w, w + MQ_NW, ...: k rounds of a wave-wide argmin over the lanes' candidates, the winner drops out
  {
    constexpr int NQW = NQ / MQ_NW;
    float v0[NQW];
    int i0[NQW];
#pragma unroll
    for (int t = 0; t < NQW; ++t) {
      v0[t] = cd[(size_t)(w + MQ_NW * t) * MQ_CAND + lane];
      i0[t] = ci[(size_t)(w + MQ_NW * t) * MQ_CAND + lane];
    }
    for (int r = 0; r < k; ++r) {
      float mv[NQW];
      int mi[NQW];
#pragma unroll
      for (int t = 0; t < NQW; ++t) {
        mv[t] = v0[t];
        mi[t] = i0[t];
      }
#pragma unroll
      for (int jx = 1; jx < 64; jx <<= 1)
#pragma unroll
        for (int t = 0; t < NQW; ++t) {
          const float ov = __int_as_float(xor_lane(__float_as_int(mv[t]), jx, lane));
          const int oi = xor_lane(mi[t], jx, lane);
          const bool take = cand_lt(ov, oi, mv[t], mi[t]);
          mv[t] = take ? ov : mv[t];
          mi[t] = take ? oi : mi[t];
        }
#pragma unroll
      for (int t = 0; t < NQW; ++t) {
        const bool won = (v0[t] == mv[t]) & (i0[t] == mi[t]);
        v0[t] = won ? FLT_MAX : v0[t];
        i0[t] = won ? -1 : i0[t];
        const int j = w + MQ_NW * t;
        if (j < nqb && lane == 0) {
          const size_t o = ((size_t)(q0 + j) * gridDim.x + blockIdx.x) * k + r;
          out_d[o] = mv[t];
          out_i[o] = mi[t];
        }
      }
    }
  }
}

// IVF-Flat scan: block (probe p, query qi) scans the whole inverted list probes[qi][p] (store rows
// [offsets[list], ends[list]); packed lists when ends == nullptr: end = offsets[list + 1]) in
// 256-row tiles (one wave per 64 rows) -> one sorted list of k at [qi][p].
constexpr int IVF_DMAX = 2048;
__global__ __launch_bounds__(ST) void ivf_scan_kernel(const float* __restrict__ xt, int cap, int d,
                                                      const float* __restrict__ q, const int* __restrict__ probes,
                                                      int nprobe, const int* __restrict__ offsets,
                                                      const int* __restrict__ ends, const int* __restrict__ ids_map,
                                                      int k, float* __restrict__ out_d, int* __restrict__ out_i) {
  __shared__ float qs[IVF_DMAX];
  __shared__ float mv[4][64];
  __shared__ int mi[4][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int qi = blockIdx.y, p = blockIdx.x;
  const int list = probes[(size_t)qi * nprobe + p];
  const int lbeg = list >= 0 ? offsets[list] : 0;
  const int lend = list < 0 ? 0 : (ends ? ends[list] : offsets[list + 1]);
  for (int t = threadIdx.x; t < d; t += ST) qs[t] = q[(size_t)qi * d + t];
  __syncthreads();
  float bv = FLT_MAX;
  int bi = -1;
  for (int r0 = lbeg; r0 < lend; r0 += 4 * 64) {
    const int row = r0 + 64 * w + lane;
    const int rc = min(row, cap - 1);
    float acc = 0.f;
    const float* col = xt + rc;
    int t = 0;
    for (; t + UNR <= d; t += UNR, col += (size_t)UNR * cap) {
      float x[UNR];
#pragma unroll
      for (int u = 0; u < UNR; ++u) x[u] = col[(size_t)u * cap];
#pragma unroll
      for (int u = 0; u < UNR; ++u) {
        const float df = x[u] - qs[t + u];
        acc = fmaf(df, df, acc);
      }
    }
    for (; t < d; ++t, col += cap) {
      const float df = *col - qs[t];
      acc = fmaf(df, df, acc);
    }
    const bool ok = row < lend;
    wave_offer(bv, bi, ok ? acc : FLT_MAX, ok ? ids_map[row] : -1, k, lane);
  }
  if (w > 0) {
    mv[w][lane] = bv;
    mi[w][lane] = bi;
  }
  __syncthreads();
  if (w == 0) {
    for (int gg = 1; gg < 4; ++gg) wave_merge64(bv, bi, mv[gg][lane], mi[gg][lane], lane);
    if (lane < k) {
      const size_t o = ((size_t)qi * gridDim.x + p) * k + lane;
      out_d[o] = bv;
      out_i[o] = bi;
    }
  }
}

// in: [nq][G][k] sorted lists -> out: [nq][k] (distances fp32, ids int64). One block of MW waves per query; each wave takes 64
// candidates at a time (64 / k whole lists per step) and offers them to its running top list; the
// waves' lists are merged last, pairwise.
constexpr int MW = 16;
__global__ __launch_bounds__(MW * 64) void topk_lists_merge_kernel(const float* __restrict__ in_d,
                                                                   const int* __restrict__ in_i, int G, int k,
                                                                   float* __restrict__ out_d,
                                                                   long long* __restrict__ out_i) {
  __shared__ float mv[MW][64];
  __shared__ int mi[MW][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int qi = blockIdx.x;
  const int lpw = 64 / k;  // whole lists per 64-lane step
  const int li = lane / k, e = lane % k;
  const size_t base = (size_t)qi * G * k;
  float bv = FLT_MAX;
  int bi = -1;
  // software-pipelined: the next step's candidates are loaded before this step's network runs (its
  // data-dependent branch otherwise keeps hipcc from hoisting them: one memory latency per step)
  int l0 = w * lpw;
  bool ok = li < lpw && l0 + li < G;
  float v = ok ? in_d[base + (size_t)(l0 + li) * k + e] : FLT_MAX;
  int id = ok ? in_i[base + (size_t)(l0 + li) * k + e] : -1;
  for (; l0 < G; l0 += MW * lpw) {
    const int ln = l0 + MW * lpw + li;
    const bool okn = li < lpw && ln < G;
    const float vn = okn ? in_d[base + (size_t)ln * k + e] : FLT_MAX;
    const int idn = okn ? in_i[base + (size_t)ln * k + e] : -1;
    wave_offer(bv, bi, v, id, k, lane);
    v = vn;
    id = idn;
  }
  // the waves' lists as a tree: four dependent merges instead of fifteen
#pragma unroll
  for (int h = MW / 2; h > 0; h >>= 1) {
    mv[w][lane] = bv;
    mi[w][lane] = bi;
    __syncthreads();
    if (w < h) wave_merge64(bv, bi, mv[w + h][lane], mi[w + h][lane], lane);
    __syncthreads();
  }
  if (w == 0 && lane < k) {  // (through to memory: a host may be watching the results arrive)
    __hip_atomic_store(out_d + (size_t)qi * k + lane, bv, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    // int64 ids: the caller's final type, no widening launch
    __hip_atomic_store(out_i + (size_t)qi * k + lane, (long long)bi, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// fill columns [n0, n0+n) of the column-major store from row-major rows x[n][d]
__global__ void l2_append_kernel(float* xt, int cap, int d, int n0, const float* __restrict__ x, int n) {
  const int row = blockIdx.x * blockDim.x + threadIdx.x;
  const int dim = blockIdx.y;
  if (row < n) xt[(size_t)dim * cap + n0 + row] = x[(size_t)row * d + dim];
}

// scatter row-major rows x[j] into column-major store slots pos[j] (IVF list appends)
__global__ void l2_scatter_kernel(float* xt, int cap, int d, const int* __restrict__ pos, const float* __restrict__ x,
                                  int n) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  const int dim = blockIdx.y;
  if (j < n) xt[(size_t)dim * cap + pos[j]] = x[(size_t)j * d + dim];
}

// gather rows (by index) out of the column-major store -> row-major [n][d]
__global__ void l2_gather_kernel(const float* __restrict__ xt, int cap, int d, const int* __restrict__ idx, int n,
                                 float* out) {
  const int i = blockIdx.x;
  const int row = idx[i];
  for (int t = threadIdx.x; t < d; t += blockDim.x) out[(size_t)i * d + t] = row >= 0 ? xt[(size_t)t * cap + row] : 0.f;
}

// ---------------------------------------------------------------------------------------------
// k-means assignment as an MFMA distance GEMM with a fused argmin (index/ivf.py training, IVF
// list assignment). ||x - c||^2 = ||x||^2 + (||c||^2 - 2 x.c): the x.c products run on the exact
// fp32-input MFMA (v_mfma_f32_16x16x4_f32: a k-ordered fmaf chain, 1/16 of the bf16 rate but
// exact like faiss' sgemm path), the argmin over centroids is kept per lane in registers.
// Block = 32 rows of X resident in LDS (pitch d + 4 floats: 16 distinct 16-B slots for the 16 rows
// a ds_read_b128 lane group touches) x every centroid, streamed in [64 centroids][64 dims] chunks.
// Wave w: rows 16*(w >> 1) .. +15 against centroids 32*(w & 1) .. +31 of each 64-centroid tile (two
// 16x16 accumulator tiles). MFMA k-slot mapping: lane l feeds dims 4*(l >> 4) + s of a 16-dim step
// in MFMA s = 0..3, so A and B fragments are single ds_read_b128s.
constexpr int KA_ROWS = 32, KA_CT = 64, KA_DC = 64, KA_DMAX = 1024;

__device__ __forceinline__ void ka_better(float v, int i, float& bv, int& bi) {
  if (v < bv || (v == bv && i < bi)) {
    bv = v;
    bi = i;
  }
}

// DUMP: also write every (row, centroid) score -(||c||^2 - 2 x.c) to scores[row][k] -- the IVF
// coarse search takes its top-nprobe from these (topk_lds, ties -> lower id), so probing and list
// assignment rank centroids by the SAME numbers (a vector is always found by a query at its own
// position with nprobe = 1).
template <bool DUMP>
__global__ __launch_bounds__(256) void kmeans_assign_kernel(const float* __restrict__ X, int n, int d,
                                                            const float* __restrict__ C,
                                                            const float* __restrict__ cnorm, int k,
                                                            int* __restrict__ assign, float* __restrict__ dist,
                                                            float* __restrict__ scores) {
  extern __shared__ __attribute__((aligned(16))) float ka_smem[];
  const int xp = d + 4;
  float* xs = ka_smem;                          // [KA_ROWS][xp]
  float* cs = ka_smem + KA_ROWS * xp;           // [KA_CT][KA_DC + 4]
  __shared__ float s_bv[2][KA_ROWS];
  __shared__ int s_bi[2][KA_ROWS];
  __shared__ float s_xn[KA_ROWS];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int row0 = blockIdx.x * KA_ROWS;
  // X tile -> LDS (rows past n are zero)
  const int d4 = d / 4;
  for (int e = tid; e < KA_ROWS * d4; e += 256) {
    const int r = e / d4, c4 = e % d4;
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (row0 + r < n) v = *reinterpret_cast<const f32x4*>(X + (size_t)(row0 + r) * d + 4 * c4);
    *reinterpret_cast<f32x4*>(xs + r * xp + 4 * c4) = v;
  }
  __syncthreads();
  if (tid < KA_ROWS) {
    float sq = 0.f;
    for (int t = 0; t < d; ++t) sq = fmaf(xs[tid * xp + t], xs[tid * xp + t], sq);
    s_xn[tid] = sq;
  }
  const int rg = wid >> 1, ch = wid & 1;  // row group, centroid half
  const int fr = lane & 15, fg = lane >> 4;
  const float* xrow = xs + (16 * rg + fr) * xp + 4 * fg;
  float bv[4] = {FLT_MAX, FLT_MAX, FLT_MAX, FLT_MAX};
  int bi[4] = {0x7fffffff, 0x7fffffff, 0x7fffffff, 0x7fffffff};
  for (int c0 = 0; c0 < k; c0 += KA_CT) {
    f32x4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
    for (int d0 = 0; d0 < d; d0 += KA_DC) {
      __syncthreads();  // previous chunk fully consumed
      for (int e = tid; e < KA_CT * (KA_DC / 4); e += 256) {
        const int r = e / (KA_DC / 4), c4 = e % (KA_DC / 4);
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
        if (c0 + r < k) v = *reinterpret_cast<const f32x4*>(C + (size_t)(c0 + r) * d + d0 + 4 * c4);
        *reinterpret_cast<f32x4*>(cs + r * (KA_DC + 4) + 4 * c4) = v;
      }
      __syncthreads();
      const float* c0row = cs + (32 * ch + fr) * (KA_DC + 4) + 4 * fg;
      const float* c1row = c0row + 16 * (KA_DC + 4);
#pragma unroll
      for (int kk = 0; kk < KA_DC; kk += 16) {
        const f32x4 a = *reinterpret_cast<const f32x4*>(xrow + d0 + kk);
        const f32x4 b0 = *reinterpret_cast<const f32x4*>(c0row + kk);
        const f32x4 b1 = *reinterpret_cast<const f32x4*>(c1row + kk);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          acc0 = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s], b0[s], acc0, 0, 0, 0);
          acc1 = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s], b1[s], acc1, 0, 0, 0);
        }
      }
    }
    // lane holds rows 4*fg + r (of this wave's 16), centroids c0 + 32*ch + fr (acc0) / + 16 (acc1)
    const int ca = c0 + 32 * ch + fr, cb = ca + 16;
    const float na = ca < k ? cnorm[ca] : 0.f, nb = cb < k ? cnorm[cb] : 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float va = na - 2.f * acc0[r], vb = nb - 2.f * acc1[r];
      if (ca < k) ka_better(va, ca, bv[r], bi[r]);
      if (cb < k) ka_better(vb, cb, bv[r], bi[r]);
      if (DUMP) {
        const int row = row0 + 16 * rg + 4 * fg + r;
        if (row < n) {
          if (ca < k) scores[(size_t)row * k + ca] = -va;
          if (cb < k) scores[(size_t)row * k + cb] = -vb;
        }
      }
    }
  }
  // argmin across the 16 lanes of a row group (same fg), then across the two centroid halves
#pragma unroll
  for (int r = 0; r < 4; ++r) {
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) {
      const float ov = __shfl_xor(bv[r], o, 64);
      const int oi = __shfl_xor(bi[r], o, 64);
      ka_better(ov, oi, bv[r], bi[r]);
    }
  }
  if (fr == 0) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      s_bv[ch][16 * rg + 4 * fg + r] = bv[r];
      s_bi[ch][16 * rg + 4 * fg + r] = bi[r];
    }
  }
  __syncthreads();
  if (tid < KA_ROWS && row0 + tid < n) {
    float v = s_bv[0][tid];
    int i = s_bi[0][tid];
    ka_better(s_bv[1][tid], s_bi[1][tid], v, i);
    if (assign) assign[row0 + tid] = i;
    if (dist) dist[row0 + tid] = fmaxf(s_xn[tid] + v, 0.f);
  }
}

}  // namespace

// dims split over S waves per row tile: more blocks for small indexes (the summation order,
// and so the last bits of a distance, depend on S -- i.e. on the index size only)
static int scan_slices(int n) { return n < 65536 ? 4 : (n < 262144 ? 2 : 1); }

template <int QB, int S>
static void launch_scan(int G, size_t lds, hipStream_t st, const float* xt, int cap, int d, int rb, int re,
                        int ntiles, const float* q, int nq, int k, float* od, int* oi, const int* ids) {
  const dim3 grid(8, (nq + QB - 1) / QB, (G + 7) / 8);
  hipLaunchKernelGGL((l2_scan_kernel<QB, S>), grid, dim3(ST), lds, st, xt, cap, d, rb, re, ntiles, q, nq, k, od, oi,
                     ids, G);
}

template <int QB>
static void launch_scan_s(int S, int G, hipStream_t st, const float* xt, int cap, int d, int rb, int re,
                          int ntiles, const float* q, int nq, int k, float* od, int* oi, const int* ids) {
  const size_t lds = (size_t)(S - 1) * (4 / S) * QB * 64 * 4;
  if (S == 4) launch_scan<QB, 4>(G, lds, st, xt, cap, d, rb, re, ntiles, q, nq, k, od, oi, ids);
  else if (S == 2) launch_scan<QB, 2>(G, lds, st, xt, cap, d, rb, re, ntiles, q, nq, k, od, oi, ids);
  else launch_scan<QB, 1>(G, lds, st, xt, cap, d, rb, re, ntiles, q, nq, k, od, oi, ids);
}

// the MFMA path (batched queries, k <= 8, d % 32 == 0) for nq >= this
static int g_mfma_min_nq = 16;
RAGK_API int ragk_l2_search_set_mfma_min_nq(int n) {
  g_mfma_min_nq = n > 0 ? n : 16;
  return 0;
}
static bool use_mfma(int nq, int k, int d) {
  return nq >= g_mfma_min_nq && k <= MQ_MK && d % 32 == 0 && d <= MQ_DMAX;
}
static size_t mfma_lds(int d, int QT) { return (size_t)mq_floats(d, QT) * 4; }
// A block a CU over all query groups, but eight (one an XCD, which then serves its rows to every group from its L2): 1000
// queries of 10000 x 1024, 256 blocks a group, each staging its q^T for one tile a wave, 1068 us, so 265.
static int mfma_blocks(int nq) { return max(8, 256 / (nq > 16 ? (nq + 31) / 32 : 1)); }
// Rows of a wave's tile / 16. Wider tiles load more a lane and share their queries' reads; narrow ones spread few rows over the
// waves. 16 / 256 queries of 1024 dims on tiles of 16, 32 and 64 rows, us: 10000 rows 34.9 / 90.6, 39.2 / 95.9, 48.9 / 97.4;
// 20000 44.5 / 145, 39.7 / 136, 50.4 / 142; 60000 88.1 / 380, 57.2 / 335, 61.9 / 311; 140000 x 16 queries - / 128 / 139, where
// 64-row tiles leave a second round nearly empty. A row costs a quarter more in the 32-row tile, so the rounds of both decide.
// Over 1000 to 500000 rows, 384 and 1024 dims and 16 to 256 queries that takes 0.5 % more than the best tile in the mean, 10 %
// at most.
static int mfma_rt(int n, int nq) {
  if (n < 16384) return 1;
  const int waves = MQ_NW * mfma_blocks(nq);
  const int r2 = ((n + 31) / 32 + waves - 1) / waves, r4 = ((n + 63) / 64 + waves - 1) / waves;
  return r2 * 2 * 5 <= r4 * 4 * 4 ? 2 : 4;
}

// Partial lists per query that l2_scan emits over rows [row_begin, row_end).
static int scan_groups(int row_begin, int row_end, int nq) {
  const int n = max(0, row_end - row_begin);
  const int S = scan_slices(n);
  const int ntiles = (n + 64 * (4 / S) - 1) / (64 * (4 / S));
  const int qgroups = (max(nq, 1) + 15) / 16;
  const int target = max(1, 2048 / qgroups);  // bounded list count: the merge stays short
  return max(1, min(ntiles, target));
}

// Partial lists per query that ragk_l2_search emits, by the kernel that it launches for (nq, k, d): size its partial buffers
// [nq][G][k] with it.
RAGK_API int ragk_l2_search_groups(int row_begin, int row_end, int nq, int k, int d) {
  if (!use_mfma(nq, k, d)) return scan_groups(row_begin, row_end, nq);
  const int n = max(0, row_end - row_begin);
  const int rows = 16 * mfma_rt(n, nq);
  return max(1, min((n + rows - 1) / rows, mfma_blocks(nq)));
}

// Exact top-k (k <= 64) over rows [row_begin, row_end) of xt[d][cap]; part_d / part_i hold
// nq * ragk_l2_search_groups(row_begin, row_end, nq, k, d) * k entries; results -> out_d / out_i [nq][k].
RAGK_API int ragk_l2_search(const float* xt, int cap, int d, int row_begin, int row_end, const float* q, int nq,
                            int k, const int* ids_map, float* part_d, int* part_i, float* out_d,
                            long long* out_i, hipStream_t st) {
  if (nq <= 0) return 0;
  if (k < 1 || k > 64 || d < 1 || cap < 1 || row_end > cap) return (int)hipErrorInvalidValue;
  if (use_mfma(nq, k, d)) {
    static const hipError_t attr = [] {
      const void* fns[6] = {(const void*)l2_mfma_kernel<1, 1>, (const void*)l2_mfma_kernel<1, 2>,
                            (const void*)l2_mfma_kernel<1, 4>, (const void*)l2_mfma_kernel<2, 1>,
                            (const void*)l2_mfma_kernel<2, 2>, (const void*)l2_mfma_kernel<2, 4>};
      for (int i = 0; i < 6; ++i) {
        const hipError_t e = hipFuncSetAttribute(fns[i], hipFuncAttributeMaxDynamicSharedMemorySize,
                                                 (int)mfma_lds(MQ_DMAX, 1 + i / 3));
        if (e != hipSuccess) return e;
      }
      return hipSuccess;
    }();
    if (attr != hipSuccess) return (int)attr;
    const int n = max(0, row_end - row_begin);
    const int RT = mfma_rt(n, nq);
    const int ntiles = (n + 16 * RT - 1) / (16 * RT);
    const int G = ragk_l2_search_groups(row_begin, row_end, nq, k, d);
    const int QT = nq > 16 ? 2 : 1;
    const dim3 grid(G, (nq + 16 * QT - 1) / (16 * QT));
    const size_t lds = mfma_lds(d, QT);
#define RAGK_MQ(Q, R) hipLaunchKernelGGL((l2_mfma_kernel<Q, R>), grid, dim3(MQ_NW * 64), lds, st, xt, cap, d, row_begin, \
                                         row_end, ntiles, q, nq, k, part_d, part_i, ids_map)
    if (QT == 2) {
      if (RT == 4) RAGK_MQ(2, 4); else if (RT == 2) RAGK_MQ(2, 2); else RAGK_MQ(2, 1);
    } else {
      if (RT == 4) RAGK_MQ(1, 4); else if (RT == 2) RAGK_MQ(1, 2); else RAGK_MQ(1, 1);
    }
#undef RAGK_MQ
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return (int)e;
    hipLaunchKernelGGL(topk_lists_merge_kernel, dim3(nq), dim3(MW * 64), 0, st, part_d, part_i, G, k, out_d, out_i);
    return (int)hipGetLastError();
  }
  const int n = max(0, row_end - row_begin);
  const int S = scan_slices(n);
  const int ntiles = (n + 64 * (4 / S) - 1) / (64 * (4 / S));
  const int G = ragk_l2_search_groups(row_begin, row_end, nq, k, d);
  // queries per block, padded to the next count below. Twelve or sixteen spill the scalar registers, and one pass of them loses
  // to two groups of eight that share the L2: 12 queries of 500000 x 1024 594 us, 15 837; in groups of eight 528
  const int QB = nq > 4 ? 8 : (nq > 2 ? 4 : nq);
  // (a grid's second dimension ends at 65535 query groups)
  for (int q0 = 0, qn; q0 < nq; q0 += qn) {
    qn = min(nq - q0, 65535 * QB);
    const float* qs = q + (size_t)q0 * d;
    float* pd = part_d + (size_t)q0 * G * k;
    int* pi = part_i + (size_t)q0 * G * k;
    if (QB == 8) launch_scan_s<8>(S, G, st, xt, cap, d, row_begin, row_end, ntiles, qs, qn, k, pd, pi, ids_map);
    else if (QB == 4) launch_scan_s<4>(S, G, st, xt, cap, d, row_begin, row_end, ntiles, qs, qn, k, pd, pi, ids_map);
    else if (QB == 2) launch_scan_s<2>(S, G, st, xt, cap, d, row_begin, row_end, ntiles, qs, qn, k, pd, pi, ids_map);
    else launch_scan_s<1>(S, G, st, xt, cap, d, row_begin, row_end, ntiles, qs, qn, k, pd, pi, ids_map);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return (int)e;
  hipLaunchKernelGGL(topk_lists_merge_kernel, dim3(nq), dim3(MW * 64), 0, st, part_d, part_i, G, k, out_d, out_i);
  return (int)hipGetLastError();
}

// IVF: part buffers hold nq * nprobe * k entries; results -> out [nq][k]
RAGK_API int ragk_ivf_search(const float* xt, int cap, int d, const float* q, int nq, const int* probes, int nprobe,
                             const int* offsets, const int* ends, const int* ids_map, int k, float* part_d,
                             int* part_i, float* out_d, long long* out_i, hipStream_t st) {
  if (nq <= 0) return 0;
  if (d > IVF_DMAX || k < 1 || k > 64 || nprobe < 1 || cap < 1) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(ivf_scan_kernel, dim3(nprobe, nq), dim3(ST), 0, st, xt, cap, d, q, probes, nprobe, offsets, ends,
                     ids_map, k, part_d, part_i);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return (int)e;
  hipLaunchKernelGGL(topk_lists_merge_kernel, dim3(nq), dim3(MW * 64), 0, st, part_d, part_i, nprobe, k, out_d,
                     out_i);
  return (int)hipGetLastError();
}

// k-means / IVF assignment: a[i] = argmin_c ||x_i - c||^2 over the k centroids (ties -> lower c),
// dist[i] = that squared distance. X [n][d], C [k][d] fp32 row-major, cnorm[c] = ||c||^2.
// scores (optional, nullptr = none): [n][k] floats, see kmeans_assign_kernel<true>
RAGK_API int ragk_kmeans_assign(const float* X, int n, int d, const float* C, const float* cnorm, int k, int* assign,
                                float* dist, float* scores, hipStream_t st) {
  if (n <= 0) return 0;
  if (d % KA_DC || d > KA_DMAX || k <= 0 || ((uintptr_t)X & 15) || ((uintptr_t)C & 15)) return (int)hipErrorInvalidValue;
  const size_t lds = (size_t)KA_ROWS * (d + 4) * 4 + (size_t)KA_CT * (KA_DC + 4) * 4;
  static bool attr_set = false;  // > 64 KiB of dynamic LDS needs the opt-in (d up to 1024: ~149 KiB)
  if (!attr_set) {
    const int mx = KA_ROWS * (KA_DMAX + 4) * 4 + KA_CT * (KA_DC + 4) * 4;
    hipError_t e = hipFuncSetAttribute((const void*)kmeans_assign_kernel<false>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, mx);
    if (e == hipSuccess)
      e = hipFuncSetAttribute((const void*)kmeans_assign_kernel<true>, hipFuncAttributeMaxDynamicSharedMemorySize, mx);
    if (e != hipSuccess) return (int)e;
    attr_set = true;
  }
  if (scores)
    hipLaunchKernelGGL(kmeans_assign_kernel<true>, dim3((n + KA_ROWS - 1) / KA_ROWS), dim3(256), lds, st, X, n, d, C,
                       cnorm, k, assign, dist, scores);
  else
    hipLaunchKernelGGL(kmeans_assign_kernel<false>, dim3((n + KA_ROWS - 1) / KA_ROWS), dim3(256), lds, st, X, n, d, C,
                       cnorm, k, assign, dist, scores);
  return (int)hipGetLastError();
}

// Results watched in host memory. A search's merge stores them into pinned memory itself, and the host needs no more than those
// stores: waiting for the stream instead adds the kernel's end, its signal and the runtime's way back, 5.5 us behind a result that
// has arrived (a kernel of one store: seen after 5.4 us, hipStreamSynchronize back after 11.0). Every entry is marked beforehand
// with an id and a distance that no search gives, and taken once neither is left, so the order of the stores does not matter.
namespace {
constexpr long long PENDING_ID = LLONG_MIN;
constexpr unsigned PENDING_D = 0xffc0deadu;  // a NaN that no arithmetic gives (should one be handed through: the stream is waited for)
constexpr auto WATCH_LIMIT = std::chrono::milliseconds(5);  // then the stream is waited for, which also reports what went wrong
}  // namespace

// block: pinned, n int64 ids and behind them n distances. Ahead of the search's launches; refused while the stream is captured (a
// graph's results would not be there to be watched).
RAGK_API int ragk_search_arm(void* block, int n, hipStream_t st) {
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  const hipError_t e = hipStreamIsCapturing(st, &cs);
  if (e != hipSuccess) return (int)e;
  if (cs != hipStreamCaptureStatusNone) return (int)hipErrorStreamCaptureUnsupported;
  long long* ids = (long long*)block;
  unsigned* d = (unsigned*)(ids + n);
  for (int i = 0; i < n; ++i) {
    __atomic_store_n(ids + i, PENDING_ID, __ATOMIC_RELAXED);
    __atomic_store_n(d + i, PENDING_D, __ATOMIC_RELAXED);
  }
  __atomic_thread_fence(__ATOMIC_SEQ_CST);
  return 0;
}

// Behind the launches: the n results into host memory as they arrive.
RAGK_API int ragk_search_collect(const void* block, int n, long long* out_i, float* out_d, hipStream_t st) {
  const long long* ids = (const long long*)block;
  const unsigned* d = (const unsigned*)(ids + n);
  const auto until = std::chrono::steady_clock::now() + WATCH_LIMIT;
  bool watch = true;
  for (int i = 0; i < n; ++i) {
    long long id;
    unsigned v;
    for (int spin = 0;; ++spin) {
      id = __atomic_load_n(ids + i, __ATOMIC_RELAXED);
      v = __atomic_load_n(d + i, __ATOMIC_RELAXED);
      if (!watch || (id != PENDING_ID && v != PENDING_D)) break;
      if ((spin & 63) == 63 && std::chrono::steady_clock::now() > until) {
        const hipError_t e = hipStreamSynchronize(st);
        if (e != hipSuccess) return (int)e;
        watch = false;
      }
    }
    out_i[i] = id;
    __builtin_memcpy(out_d + i, &v, 4);
  }
  return 0;
}

// Returns when everything enqueued on the stream is done.
RAGK_API int ragk_stream_wait(hipStream_t st) { return (int)hipStreamSynchronize(st); }

RAGK_API int ragk_l2_append(float* xt, int cap, int d, int n0, const float* x, int n, hipStream_t st) {
  if (n <= 0) return 0;
  if (n0 + n > cap) return (int)hipErrorInvalidValue;
  dim3 grid((n + 255) / 256, d);
  hipLaunchKernelGGL(l2_append_kernel, grid, dim3(256), 0, st, xt, cap, d, n0, x, n);
  return (int)hipGetLastError();
}

// x [n][d] row-major -> store slots pos[j] (every pos < cap; the launcher's caller checks)
RAGK_API int ragk_l2_scatter(float* xt, int cap, int d, const int* pos, const float* x, int n, hipStream_t st) {
  if (n <= 0) return 0;
  dim3 grid((n + 255) / 256, d);
  hipLaunchKernelGGL(l2_scatter_kernel, grid, dim3(256), 0, st, xt, cap, d, pos, x, n);
  return (int)hipGetLastError();
}

RAGK_API int ragk_l2_gather(const float* xt, int cap, int d, const int* idx, int n, float* out, hipStream_t st) {
  if (n <= 0) return 0;
  hipLaunchKernelGGL(l2_gather_kernel, dim3(n), dim3(256), 0, st, xt, cap, d, idx, n, out);
  return (int)hipGetLastError();
}
