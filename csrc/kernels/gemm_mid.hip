// bf16 GEMM for row counts between decode and full prefill steps: C[M,N] = A[M,K] . B[N,K]^T (+ fused epilogue).
//
// A few hundred to a few thousand rows give the 256x256 tiles of gemm_w4.hip too few tiles for 256 CUs (112 at
// 1777 x 4096), and a 128x128 tile with one K-tile in flight waits for memory on every K-tile. Here:
//  * tiles of 32*MI x 128 (MI = 3 .. 8: 96 to 256 rows) and of 160 x 256, chosen with the K-split by a cost model of the
//    whole launch (ops/native.py gemm_plan), so rows are padded little and the last round of tiles is full;
//  * a ring of D K-tiles (64 deep, 3 to 5 of them in LDS), a slot refilled as soon as it is read out; one persistent
//    block per CU streams the K-tiles of its work items through it as one sequence, so only the first item waits;
//  * split-K: work item = (slab, tile); fp32 slabs P[S][M][N] go to a consumer that sums them (row norms) or to
//    splitk_finish (bias / residual / activation / gated pairs).
// 4 waves as 2 x 2, wave tile 16*MI x 16*NJ (NJ = 4: 128 columns, 8: 256): per K-tile a wave reads (16 MI + 16 NJ) x 128 B
// for 2 MI NJ MFMAs. LDS traffic with the DMA writes bounds small MI (768 of 512 MFMA clocks at MI = 4, 1152 of 1024 at
// MI = 8); 160 x 256 is the largest tile that leaves a ring of three K-tiles and the one that LDS bounds least (1248 clocks
// of 1280): two of the 160 x 128 tiles it stands for take 1728. 192 x 192 and 224 x 192 tiles came to the same rates and won
// where neither size divides well only (1500 x 6144 x 4096 64 us against 66), 96 and 128 rows of 256 columns nowhere.
//
// Measured (us, cold weights; before: the 128x128 double-buffered tile / gemm_w4 from 1024 rows): 300 x 4096 x 4096
// 48 -> 24, 300 x 4096 x 14336 193 -> 51, 300 x 28672 x 4096 126 -> 86, 800 x 4096 x 4096 51 -> 31, 1777 x 4096 x 4096
// 79 -> 55, 1777 x 4096 x 14336 263 -> 181, 3000 x 1024 x 4096 69 -> 28 (on the slowest card seen a tenth more: 24.4, 53,
// 94, 34, 61, 197, 31). With 160 x 256 and 224 x 128 beside the other tiles (both on that card): 300 x 28672 x 4096 89 -> 75,
// 600 x 28672 x 4096 154 -> 135, 600 x 4096 x 14336 in slabs 81 -> 67, 1500 x 6144 x 4096 81 -> 67, 1777 x 4096 x 4096 56 ->
// 54, 1777 x 4096 x 14336 183 -> 175, 200 x 28672 x 4096 65 -> 61.
// A K-tile takes 0.28 us at MI = 3 and 0.62 at MI = 8 on few blocks (LDS bound: 0.28 and 0.48), with
// every CU busy 0.40 and 0.83; of 160 x 256 0.76 and 0.96.
//
// The weight fragment is the first MFMA operand: a lane holds four consecutive output columns of one row, eight with
// the staged weight rows permuted (mid_row), so epilogues load and store 16 B straight from registers. K order and
// MFMA shape equal gemm_w4's: without a K-split the results are bit-identical to it.
#include <type_traits>

#include "attn_tiles.h"
using namespace ragk;

namespace {

constexpr int MID_BK = 64, MID_THREADS = 256;
constexpr int MID_GROUP_M = 8;
constexpr int MID_LDS = 160 * 1024;
constexpr int MID_WIDE = 16;  // added to a tile's rows / 32 in the C entries' `mi`: 256 columns instead of 128

constexpr int mid_stage(int mi, int nj) { return 32 * (mi + nj) * MID_BK * 2; }
constexpr int mid_depth(int mi, int nj) { return MID_LDS / mid_stage(mi, nj) < 5 ? MID_LDS / mid_stage(mi, nj) : 5; }

__device__ __forceinline__ int mswz(int row, int chunk) { return chunk ^ ((row >> 1) & 7); }

// Weight row (within the tile) staged at LDS row q, so that lane (fr, fh) of MFMA tiles 2p, 2p + 1 of a wave holds eight
// consecutive output columns. PAIR: groups of 128 rows are [64 first | 64 second] (gate / up; the halves of a rotated head)
// and tile j of a wave pairs with tile j + NJ / 2, so both members of a pair are in one lane: 128 columns are one group
// that two waves share, a wave of the 256-column tile has a group of its own and needs no other order than without pairs.
template <int NJ, bool PAIR>
__device__ __forceinline__ int mid_row(int q) {
  const int h = q / (16 * NJ), j = (q >> 4) % NJ, c = (q >> 2) & 3, k = q & 3;
  if constexpr (PAIR && NJ == 4) return 64 * (j >> 1) + 32 * h + 8 * c + 4 * (j & 1) + k;
  return 16 * NJ * h + 32 * (j >> 1) + 8 * c + 4 * (j & 1) + k;
}

// Inline asm ties source and destination of an accumulator (with the builtin hipcc rotates them through other registers
// and copies them back, 60 moves a K-tile). The compiler pads no hazards of these: mid_pin before the first of a tile
// and before the epilogue's reads.
__device__ __forceinline__ void mid_mfma(f32x4& c, const bf16x8& w, const bf16x8& x) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(w), "v"(x));
}
template <int MI, int NJ>
__device__ __forceinline__ void mid_pin(f32x4 (&acc)[MI][NJ]) {
  asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 1" ::: "memory");
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) asm volatile("" : "+a"(acc[i][j])::"memory");
}

struct MidItem {
  int m0, n0, k0, k1, z;  // tile origin, K-tile range, slab
};

// Work item -> tile. Items are numbered so that each XCD owns a contiguous range (a block keeps its XCD: the grid is
// a multiple of 8 or one round), M-tiles of one weight panel next to each other.
__device__ __forceinline__ MidItem mid_item(int it, int total, int tiles_m, int tiles_n, int nk, int S, int bm,
                                           int bn) {
  const int nt = tiles_m * tiles_n;
  int l = xcd_remap(it, total);
  MidItem w;
  w.z = __builtin_amdgcn_readfirstlane(l / nt);
  l -= w.z * nt;
  const int group = l / (MID_GROUP_M * tiles_n);
  const int first = group * MID_GROUP_M;
  const int gm = min(tiles_m - first, MID_GROUP_M);
  const int in = l - group * MID_GROUP_M * tiles_n;
  // (uniform; the divisions run on the vector unit)
  w.m0 = __builtin_amdgcn_readfirstlane((first + in % gm) * bm);
  w.n0 = __builtin_amdgcn_readfirstlane((in / gm) * bn);
  w.k0 = __builtin_amdgcn_readfirstlane((int)((unsigned)(nk * w.z) / (unsigned)S));
  w.k1 = __builtin_amdgcn_readfirstlane((int)((unsigned)(nk * (w.z + 1)) / (unsigned)S));
  return w;
}

constexpr bool mid_has_bias(int e) { return e == EPI_BIAS || e == EPI_BIAS_RESID || e == EPI_BIAS_GELU || e == EPI_BIAS_GELU_TANH; }
constexpr bool mid_has_resid(int e) { return e == EPI_RESID || e == EPI_BIAS_RESID; }

// values of eight consecutive outputs + bias, residual (as loaded), activation (the order and rounding of gemm_w4's epilogue)
template <int EPI>
__device__ __forceinline__ void mid_finish8(float (&o)[8], u32x4 bias, u32x4 resid) {
  if constexpr (mid_has_bias(EPI)) {
    float b[8];
    unpack8(bias, b);
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] += b[e];
  }
  if constexpr (mid_has_resid(EPI)) {
    float r[8];
    unpack8(resid, r);
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] += r[e];
  }
  if constexpr (EPI == EPI_BIAS_GELU || EPI == EPI_GELU) {
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = gelu_erf(o[e]);
  }
  if constexpr (EPI == EPI_BIAS_GELU_TANH) {
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = gelu_tanh(o[e]);
  }
}

__device__ __forceinline__ void mid_store8(void* C, size_t at, const float (&o)[8], int out_f32) {
  if (out_f32) {
    f32x4* d = reinterpret_cast<f32x4*>(reinterpret_cast<float*>(C) + at);
    d[0] = (f32x4){o[0], o[1], o[2], o[3]};
    d[1] = (f32x4){o[4], o[5], o[6], o[7]};
  } else {
    *reinterpret_cast<u32x4*>(reinterpret_cast<bf16_t*>(C) + at) = pack8(o);
  }
}

// What rope_kv's work on eight column pairs of a row takes from memory, beside the row's position.
struct MidTurn {
  f32x4 cs[2], sn[2];
  int slot;
};
__device__ __forceinline__ MidTurn mid_turn(const RopeKV& rk, int pos, int row, int hd, int d) {
  MidTurn t;
  if (hd < rk.Hq + rk.Hkv) {
    const f32x4* c = reinterpret_cast<const f32x4*>(rk.cos_t + (size_t)pos * 64 + d);
    const f32x4* s = reinterpret_cast<const f32x4*>(rk.sin_t + (size_t)pos * 64 + d);
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      t.cs[e] = c[e];
      t.sn[e] = s[e];
    }
  }
  t.slot = hd < rk.Hq ? -1 : rk.slot[row];
  return t;
}

// Eight columns d .. d+7 and their partners d + 64 .. of head hd in row `row`: rope_kv's work on the bf16 projection (norm.hip,
// the same rounding of every op), C and the caches written.
__device__ __forceinline__ void mid_rope8(float (&x1)[8], float (&x2)[8], const RopeKV& rk, const MidTurn& t, bf16_t* C, int ldc,
                                          int row, int hd, int d) {
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    x1[e] = bf2f(f2bf(x1[e]));
    x2[e] = bf2f(f2bf(x2[e]));
  }
  if (hd < rk.Hq + rk.Hkv) {
    float o1[8], o2[8], cs[8], sn[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      cs[e] = t.cs[e >> 2][e & 3];
      sn[e] = t.sn[e >> 2][e & 3];
    }
    rope8(x1, x2, cs, sn, o1, o2);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      x1[e] = o1[e];
      x2[e] = o2[e];
    }
  }
  const u32x4 p1 = pack8(x1), p2 = pack8(x2);
  bf16_t* c = C + (size_t)row * ldc + hd * 128 + d;
  *reinterpret_cast<u32x4*>(c) = p1;
  *reinterpret_cast<u32x4*>(c + 64) = p2;
  if (t.slot >= 0) {
    const bool isk = hd < rk.Hq + rk.Hkv;
    const int kvh = hd - rk.Hq - (isk ? 0 : rk.Hkv);
    bf16_t* dst = (isk ? rk.kc : rk.vc) + (((size_t)(t.slot / rk.BS) * rk.Hkv + kvh) * rk.BS + t.slot % rk.BS) * 128 + d;
    *reinterpret_cast<u32x4*>(dst) = p1;
    *reinterpret_cast<u32x4*>(dst + 64) = p2;
  }
}

// Weights that one row of tiles reads once, by the streaming policy: 28672 x 4096 at 66 / 140 / 256 rows 50.8 / 56.2 / 66.2 -> 46.9 /
// 53.4 / 61.9 us, 22528 x 2048 25.4 / 29.1 / 33.8 -> 23.4 / 27.6 / 31.3; also behind whole rounds of larger tiles that have just read
// them (700 / 3000 rows, the last 188 / 184 here, 146 / 503 -> 141 / 502; 5192 of 22528 x 2048, the last 72, 344 -> 340). Where tiles
// share them (several rows of tiles, a K-split) it costs 2 to 11 % instead, and weights that the caches hold from call to call keep
// the other policy.
__device__ __forceinline__ void blds16_nt_asm(i32x4 srd, int voff, int soff, unsigned lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen nt lds" ::"s"(lds_addr), "v"(voff), "s"(srd),
               "s"(soff));
}
constexpr bool mid_has_nt(int e) { return e == EPI_NONE || epi_pair(e); }
constexpr long long MID_NT_BYTES = 64LL << 20;  // twice the L2s

template <int MI, int NJ, int EPI, bool NT = false>
__global__ __launch_bounds__(MID_THREADS, 1) void gemm_mid_kernel(
    const bf16_t* __restrict__ A, int lda, const bf16_t* __restrict__ B, int ldb, void* C, int ldc,
    const bf16_t* __restrict__ bias, const bf16_t* resid, int ldr, int M, int N, int K, int S, int out_f32, RopeKV rk) {
  constexpr bool PAIR = epi_pair(EPI) || EPI == EPI_ROPE_KV;
  constexpr int BM = 32 * MI, BN = 32 * NJ, STAGE = mid_stage(MI, NJ), D = mid_depth(MI, NJ);
  constexpr int PW = MI + NJ;          // DMA pieces (and fragment reads a half) a wave
  constexpr int DSTEP = NJ * MI / PW;  // MFMAs between two pieces
  constexpr int OFF_B = BM * 128;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = wid >> 1, wc = wid & 1, fr = lane & 15, fh = lane >> 4;
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  const int total = tiles_m * tiles_n * S, nk = K / MID_BK, grid = gridDim.x;

  // ---- DMA side: the K-tile that is issued next. Descriptors start at the tile's own rows, so offsets stay small.
  int d_it = blockIdx.x;
  MidItem dw = mid_item(d_it, total, tiles_m, tiles_n, nk, S, BM, BN);
  int dk = dw.k0, off_a[MI], off_b[NJ];
  i32x4 srd_a, srd_b;
  auto origin = [&](const MidItem& w) {
    // rows past the edge read the last valid row: their outputs are never stored
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const int r = (wid * MI + i) * 8 + (lane >> 3);
      off_a[i] = min(r, M - 1 - w.m0) * lda * 2 + 16 * mswz(r, lane & 7);
    }
#pragma unroll
    for (int i = 0; i < NJ; ++i) {
      const int r = (wid * NJ + i) * 8 + (lane >> 3);
      off_b[i] = min(mid_row<NJ, PAIR>(r), N - 1 - w.n0) * ldb * 2 + 16 * mswz(r, lane & 7);
    }
    srd_a = make_srd(A + (size_t)w.m0 * lda, 0x7fffffffu);
    srd_b = make_srd(B + (size_t)w.n0 * ldb, 0x7fffffffu);
  };
  origin(dw);
  const unsigned lds0 = __builtin_amdgcn_readfirstlane(lds_addr(smem));
  unsigned d_slot = lds0;
  // piece q of the K-tile at (dk, d_slot): the activation's first, then the weight's
  auto piece = [&](int q) {
    const int so = dk * (MID_BK * 2);
    if (q < MI) blds16_asm(srd_a, off_a[q], so, d_slot + (wid * MI + q) * 1024);
    else if constexpr (NT) blds16_nt_asm(srd_b, off_b[q - MI], so, d_slot + OFF_B + (wid * NJ + q - MI) * 1024);
    else blds16_asm(srd_b, off_b[q - MI], so, d_slot + OFF_B + (wid * NJ + q - MI) * 1024);
  };
  auto advance = [&]() {
    d_slot = d_slot + STAGE == lds0 + D * STAGE ? lds0 : d_slot + STAGE;
    if (++dk == dw.k1) {
      const int nx = d_it + grid;
      if (nx < total) {
        d_it = nx;
        dw = mid_item(nx, total, tiles_m, tiles_n, nk, S, BM, BN);
        dk = dw.k0;
        origin(dw);
      } else {
        --dk;  // nothing left: the last K-tile again (valid addresses, never read), so the waits' counts hold
      }
    }
  };

  // ---- fragment reads: the swizzle of row 16 i + fr does not depend on i
  const char* ra[2];
  const char* rb[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int cs = 16 * ((4 * s + fh) ^ ((fr >> 1) & 7));
    ra[s] = smem + (wr * 16 * MI + fr) * 128 + cs;
    rb[s] = smem + OFF_B + (wc * 16 * NJ + fr) * 128 + cs;
  }
  bf16x8 a0[MI], b0[NJ], a1[MI], b1[NJ];
  auto read = [&](bf16x8 (&a)[MI], bf16x8 (&b)[NJ], int s, unsigned slot, int q) {
    if (q < NJ) b[q] = *reinterpret_cast<const bf16x8*>(rb[s] + slot + q * 2048);
    else a[q - NJ] = *reinterpret_cast<const bf16x8*>(ra[s] + slot + (q - NJ) * 2048);
  };
  f32x4 acc[MI][NJ];
  // MFMA m of a 32-deep half, then what else goes out there: the order is the written one (one wave a SIMD: nothing
  // else fills the gap that a burst of reads or DMAs leaves)
  auto half = [&](const bf16x8 (&a)[MI], const bf16x8 (&b)[NJ], bf16x8 (&na)[MI], bf16x8 (&nb)[NJ], int ns, unsigned nslot,
                  auto dma) {
#pragma unroll
    for (int m = 0; m < NJ * MI; ++m) {
      const int i = m / NJ, j = m % NJ;
      mid_mfma(acc[i][j], b[j], a[i]);
      if (m < PW) read(na, nb, ns, nslot, m);
      if constexpr (decltype(dma)::value) {
        if (m % DSTEP == DSTEP - 1 && m / DSTEP < PW) piece(m / DSTEP);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

#pragma unroll
  for (int d = 0; d < D; ++d) {
#pragma unroll
    for (int q = 0; q < PW; ++q) piece(q);
    advance();
  }
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((D - 1) * PW) : "memory");
  unsigned slot = 0;
#pragma unroll
  for (int q = 0; q < PW; ++q) read(a0, b0, 0, slot, q);

  for (int it = blockIdx.x; it < total; it += grid) {
    const MidItem w = mid_item(it, total, tiles_m, tiles_n, nk, S, BM, BN);
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
        asm volatile("" : "+a"(acc[i][j]));
      }
    asm volatile("s_nop 7" ::: "memory");
    for (int k = w.k0; k < w.k1; ++k) {
      half(a0, b0, a1, b1, 1, slot, std::false_type{});
      // this slot is read out, and the next K-tile has landed, in every wave
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((D - 2) * PW) : "memory");
      __builtin_amdgcn_sched_barrier(0);
      slot = slot + STAGE == D * STAGE ? 0 : slot + STAGE;
      half(a1, b1, a0, b0, 0, slot, std::true_type{});  // its DMAs refill the slot just read out
      advance();
    }
    mid_pin(acc);
    // ---- epilogue
    if constexpr (EPI == EPI_ROPE_KV) {
      // Positions of all rows together, then tables and slots a row ahead of their use, instead of two loads in turn a row:
      // 1300 x 6144 x 4096 on 160-row tiles 78.1 -> 75.4 us, 8192 x 3072 x 2048 on 256-row ones 108.5 -> 99.4 (without the
      // rotation 67.3 and 85.1).
      // A wave of the 128-column tile turns 32 of a head's column pairs, one of the 256-column tile a whole head (the last such
      // tile may hold one head only).
      const int hd = (w.n0 >> 7) + (NJ == 8 ? wc : 0), r0 = w.m0 + wr * 16 * MI + fr;
      int pos[MI];
#pragma unroll
      for (int i = 0; i < MI; ++i) pos[i] = rk.pos[min(r0 + 16 * i, M - 1)];
      if (hd * 128 < N) {
#pragma unroll
        for (int p = 0; p < NJ / 4; ++p) {
          const int d = (NJ == 8 ? 32 * p : 32 * wc) + 8 * fh;
          MidTurn t = mid_turn(rk, pos[0], min(r0, M - 1), hd, d), next = t;
#pragma unroll
          for (int i = 0; i < MI; ++i) {
            const int row = r0 + 16 * i;
            if (i + 1 < MI) next = mid_turn(rk, pos[i + 1 < MI ? i + 1 : i], min(row + 16, M - 1), hd, d);
            if (row < M) {
              float x1[8], x2[8];
#pragma unroll
              for (int e = 0; e < 8; ++e) {
                x1[e] = acc[i][2 * p + (e >> 2)][e & 3];
                x2[e] = acc[i][2 * p + NJ / 2 + (e >> 2)][e & 3];
              }
              mid_rope8(x1, x2, rk, t, reinterpret_cast<bf16_t*>(C), ldc, row, hd, d);
            }
            t = next;
          }
        }
      }
    } else if constexpr (PAIR) {
      const GluPar gp = glu_par<EPI>(bias);
#pragma unroll
      for (int p = 0; p < NJ / 4; ++p) {
        const int col = (w.n0 >> 1) + (NJ == 8 ? 64 * wc + 32 * p : 32 * wc) + 8 * fh;
        if (2 * col < N) {
#pragma unroll
          for (int i = 0; i < MI; ++i) {
            const int row = w.m0 + wr * 16 * MI + 16 * i + fr;
            float o[8];
#pragma unroll
            for (int e = 0; e < 8; ++e)
              o[e] = glu_act<EPI>(acc[i][2 * p + (e >> 2)][e & 3], acc[i][2 * p + NJ / 2 + (e >> 2)][e & 3], gp);
            if (row < M) *reinterpret_cast<u32x4*>(reinterpret_cast<bf16_t*>(C) + (size_t)row * ldc + col) = pack8(o);
          }
        }
      }
    } else {
      void* Cz = out_f32 ? (void*)(reinterpret_cast<float*>(C) + (size_t)w.z * M * ldc) : C;
      // The tile's bias and residual are requested together, ahead of any use: loaded where they are added, each of the 2 MI
      // row pieces waited for memory once more (8192 x 3072 x 1024 on 256-row tiles, us: bias 65.4 -> 56.5, without an epilogue
      // 55.1; GELU 78.2 -> 68.3; 13762 x 1024 x 4096, bias and residual, 160-row tiles 118.7 -> 116.8).
      u32x4 bv[NJ / 2] = {}, rv[MI][NJ / 2] = {};
#pragma unroll
      for (int p = 0; p < NJ / 2; ++p) {
        const int col = min(w.n0 + 16 * NJ * wc + 32 * p + 8 * fh, N - 8);
        if constexpr (mid_has_bias(EPI)) bv[p] = *reinterpret_cast<const u32x4*>(bias + col);
        if constexpr (mid_has_resid(EPI)) {
#pragma unroll
          for (int i = 0; i < MI; ++i)
            rv[i][p] = *reinterpret_cast<const u32x4*>(resid + (size_t)min(w.m0 + wr * 16 * MI + 16 * i + fr, M - 1) * ldr + col);
        }
      }
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        const int row = w.m0 + wr * 16 * MI + 16 * i + fr;
#pragma unroll
        for (int p = 0; p < NJ / 2; ++p) {
          const int col = w.n0 + 16 * NJ * wc + 32 * p + 8 * fh;
          if (row < M && col < N) {
            float o[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = acc[i][2 * p + (e >> 2)][e & 3];
            mid_finish8<EPI>(o, bv[p], rv[i][p]);
            mid_store8(Cz, (size_t)row * ldc + col, o, out_f32);
          }
        }
      }
    }
  }
  // the surplus DMAs land before the block's LDS is released
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// Sum of the fp32 slabs P[S][M][Np] + epilogue (Np = N, or 2 N packed [64 gate | 64 up] columns). One thread per eight
// output columns.
template <int EPI>
__global__ __launch_bounds__(256) void splitk_finish_kernel(const float* __restrict__ P, int S, void* C, int ldc,
                                                            const bf16_t* __restrict__ bias, const bf16_t* resid, int ldr,
                                                            int M, int N, int out_f32) {
  const int vec = N >> 3;
  const long long v = (long long)blockIdx.x * 256 + threadIdx.x;
  if (v >= (long long)M * vec) return;
  const int row = (int)(v / vec), col = (int)(v % vec) * 8;
  float o[8];
  if constexpr (epi_pair(EPI)) {
    const size_t slab = (size_t)M * 2 * N;
    const float* p = P + (size_t)row * 2 * N + (col >> 6) * 128 + (col & 63);
    float g[8], u[8];
    sum_slabs8(p, S, slab, g);
    sum_slabs8(p + 64, S, slab, u);
    const GluPar gp = glu_par<EPI>(bias);
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = glu_act<EPI>(g[e], u[e], gp);
  } else {
    u32x4 bv = {}, rv = {};
    if constexpr (mid_has_bias(EPI)) bv = *reinterpret_cast<const u32x4*>(bias + col);
    if constexpr (mid_has_resid(EPI)) rv = *reinterpret_cast<const u32x4*>(resid + (size_t)row * ldr + col);
    sum_slabs8(P + (size_t)row * N + col, S, (size_t)M * N, o);
    mid_finish8<EPI>(o, bv, rv);
  }
  mid_store8(C, (size_t)row * ldc + col, o, out_f32);
}

// The same for the rotated projection: one thread per (row, head, eight column pairs).
__global__ __launch_bounds__(256) void splitk_rope_kernel(const float* __restrict__ P, int S, bf16_t* C, int ldc, int M, int N,
                                                          RopeKV rk) {
  const int vec = N >> 4;
  const long long v = (long long)blockIdx.x * 256 + threadIdx.x;
  if (v >= (long long)M * vec) return;
  const int row = (int)(v / vec), r = (int)(v % vec), hd = r >> 3, d = (r & 7) * 8;
  const float* p = P + (size_t)row * N + hd * 128 + d;
  const MidTurn t = mid_turn(rk, rk.pos[row], row, hd, d);
  float x1[8], x2[8];
  sum_slabs8(p, S, (size_t)M * N, x1);
  sum_slabs8(p + 64, S, (size_t)M * N, x2);
  mid_rope8(x1, x2, rk, t, C, ldc, row, hd, d);
}

// An operand's rows as the DMA takes them: 16-byte pieces, a tile's (at most 256) rows within 32-bit offsets.
bool mid_rows_ok(const void* p, int ld, int K) {
  return (uintptr_t)p % 16 == 0 && ld % 8 == 0 && 256LL * ld * 2 + 2LL * K < (1LL << 31);
}

int mid_grid(int total) {
  static int cus = 0;
  if (!cus) {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
      n = 256;
    cus = n / 8 * 8;
  }
  return total < cus ? total : cus;
}

template <int MI, int NJ, int EPI, bool NT = false>
int launch_mid(const void* A, int lda, const void* B, int ldb, void* C, int ldc, const void* bias, const void* resid, int ldr,
               int M, int N, int K, int S, int out_f32, hipStream_t st,
               const RopeKV& rk = RopeKV{}) {
  if constexpr (!NT && mid_has_nt(EPI))
    if (M <= 32 * MI && S == 1 && 2LL * N * K >= MID_NT_BYTES)
      return launch_mid<MI, NJ, EPI, true>(A, lda, B, ldb, C, ldc, bias, resid, ldr, M, N, K, S, out_f32, st, rk);
  constexpr int lds = mid_stage(MI, NJ) * mid_depth(MI, NJ);
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_mid_kernel<MI, NJ, EPI, NT>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (attr != hipSuccess) return (int)attr;
  const long long total = (long long)((M + 32 * MI - 1) / (32 * MI)) * ((N + 32 * NJ - 1) / (32 * NJ)) * S;
  if (total > 0x7fffffff) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL((gemm_mid_kernel<MI, NJ, EPI, NT>), dim3(mid_grid((int)total)), dim3(MID_THREADS), lds, st, (const bf16_t*)A,
                     lda, (const bf16_t*)B, ldb, C, ldc, (const bf16_t*)bias, (const bf16_t*)resid, ldr, M, N, K, S, out_f32, rk);
  return (int)hipGetLastError();
}

template <int EPI>
int dispatch_mid(int mi, const void* A, int lda, const void* B, int ldb, void* C, int ldc, const void* bias, const void* resid,
                 int ldr, int M, int N, int K, int S, int out_f32, hipStream_t st, const RopeKV& rk = RopeKV{}) {
  switch (mi) {
#define RAGK_TILE(CODE, MI, NJ) \
  case CODE: return launch_mid<MI, NJ, EPI>(A, lda, B, ldb, C, ldc, bias, resid, ldr, M, N, K, S, out_f32, st, rk);
    RAGK_TILE(3, 3, 4)
    RAGK_TILE(4, 4, 4)
    RAGK_TILE(5, 5, 4)
    RAGK_TILE(6, 6, 4)
    RAGK_TILE(7, 7, 4)
    RAGK_TILE(8, 8, 4)
    RAGK_TILE(MID_WIDE + 5, 5, 8)
#undef RAGK_TILE
    default: return (int)hipErrorInvalidValue;
  }
}

template <int EPI>
int launch_finish(const float* P, int S, void* C, int ldc, const void* bias, const void* resid, int ldr, int M, int N,
                  int out_f32, hipStream_t st) {
  const long long blocks = ((long long)M * (N >> 3) + 255) / 256;
  hipLaunchKernelGGL((splitk_finish_kernel<EPI>), dim3((unsigned)blocks), dim3(256), 0, st, P, S, C, ldc, (const bf16_t*)bias,
                     (const bf16_t*)resid, ldr, M, N, out_f32);
  return (int)hipGetLastError();
}

}  // namespace

#define RAGK_MID_EPIS(X) \
  X(EPI_NONE) X(EPI_BIAS) X(EPI_RESID) X(EPI_BIAS_RESID) X(EPI_BIAS_GELU) X(EPI_GELU) X(EPI_BIAS_GELU_TANH) \
  X(EPI_SILU_MUL) X(EPI_GLU_CLIP)

// C = epilogue of the sum of P's S fp32 slabs [M][weight rows]. C, bias and resid rows start on 16 bytes, N % 8 == 0.
RAGK_API int ragk_slabs_finish(const float* P, int S, void* C, int ldc, const void* bias, const void* resid, int ldr, int M,
                               int N, int epi, int out_f32, hipStream_t st) {
  if (M <= 0 || N <= 0) return 0;
  if (S < 1 || !P || N % (epi_pair(epi) ? 64 : 8) || (epi_pair(epi) && out_f32)) return (int)hipErrorInvalidValue;
  if (((mid_has_bias(epi) || epi == EPI_GLU_CLIP) && !bias) || (mid_has_resid(epi) && !resid)) return (int)hipErrorInvalidValue;
#define RAGK_FIN(E) \
  case E: return launch_finish<E>(P, S, C, ldc, bias, resid, ldr, M, N, out_f32, st);
  switch (epi) {
    RAGK_MID_EPIS(RAGK_FIN)
    default: return (int)hipErrorInvalidValue;
  }
#undef RAGK_FIN
}

// N = output columns (for the pair epilogues the weight has 2 N rows in the packed [64 gate | 64 up] layout, N % 64 == 0).
// Rows of A and B start on 16 bytes. mi = rows of a tile / 32. S > 1: K-split through the fp32 slabs ws [S][M][weight rows],
// summed with the epilogue by a second launch. S slabs without a consumer here: epi NONE, out_f32 = 2 (C holds the slabs).
RAGK_API int ragk_gemm_mid(const void* A, int lda, const void* B, int ldb, void* C, int ldc, const void* bias,
                           const void* resid, int ldr, int M, int N, int K, int epi, int out_f32, int mi, int S, float* ws,
                           hipStream_t st) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const int nk = K / MID_BK;
  if (K % MID_BK || S < 1 || S > nk || N % 8) return (int)hipErrorInvalidValue;
  if (epi_pair(epi) && (N % 64 || out_f32)) return (int)hipErrorInvalidValue;
  if (epi == EPI_GLU_CLIP && !bias) return (int)hipErrorInvalidValue;
  if (!mid_rows_ok(A, lda, K) || !mid_rows_ok(B, ldb, K)) return (int)hipErrorInvalidValue;
  const int rows = epi_pair(epi) ? 2 * N : N;
  if (out_f32 == 2) {
    if (epi != EPI_NONE || ldc != N) return (int)hipErrorInvalidValue;
    return dispatch_mid<EPI_NONE>(mi, A, lda, B, ldb, C, ldc, nullptr, nullptr, 0, M, N, K, S, 1, st);
  }
  if (S > 1) {
    if (!ws) return (int)hipErrorInvalidValue;
    const int rc = dispatch_mid<EPI_NONE>(mi, A, lda, B, ldb, ws, rows, nullptr, nullptr, 0, M, rows, K, S, 1, st);
    return rc ? rc : ragk_slabs_finish(ws, S, C, ldc, bias, resid, ldr, M, N, epi, out_f32, st);
  }
#define RAGK_MID(E) \
  case E: return dispatch_mid<E>(mi, A, lda, B, ldb, C, ldc, bias, resid, ldr, M, rows, K, 1, out_f32, st);
  switch (epi) {
    RAGK_MID_EPIS(RAGK_MID)
    default: return (int)hipErrorInvalidValue;
  }
#undef RAGK_MID
}

RAGK_API int ragk_gemm_stream_part(const void* X, int ldx, const void* W, int ldw, float* P, int M, int N, int K, int S,
                                   int rows, int short_sums, hipStream_t st);

// At most 64 rows: the LDS-DMA weight stream's fp32 slabs ws [S][M][N] (gemm_stream.hip; `rows` of a tile, S | K / 64) and
// their sum with the epilogue, as above; no pair epilogues.
RAGK_API int ragk_gemm_slabs(const void* X, int ldx, const void* W, int ldw, void* C, int ldc, const void* bias,
                             const void* resid, int ldr, int M, int N, int K, int epi, int S, int rows, float* ws, hipStream_t st) {
  if (M <= 0 || N <= 0) return 0;
  if (N % 8 || epi_pair(epi) || !ws) return (int)hipErrorInvalidValue;
  const int rc = ragk_gemm_stream_part(X, ldx, W, ldw, ws, M, N, K, S, rows, 1, st);
  return rc ? rc : ragk_slabs_finish(ws, S, C, ldc, bias, resid, ldr, M, N, epi, 0, st);
}

// qkv = A . B^T, B = [(Hq + 2 Hkv) * 128][K], with rope_kv's work in the epilogue: q and k rotated (positions pos[M], tables
// cos_t / sin_t [positions][64]), k and v rows also into the paged caches at slot[M]. S > 1: slabs ws [S][M][N] as above.
RAGK_API int ragk_gemm_mid_rope_kv(const void* A, int lda, const void* B, int ldb, void* C, int ldc, int M, int K,
                                   const int* pos, const int* slot, const float* cos_t, const float* sin_t, void* kc, void* vc,
                                   int Hq, int Hkv, int BS, int mi, int S, float* ws, hipStream_t st) {
  if (M <= 0) return 0;
  const int N = (Hq + 2 * Hkv) * 128;
  if (K % MID_BK || K <= 0 || S < 1 || S > K / MID_BK || Hq < 1 || Hkv < 1 || BS < 1 || ldc % 8 || (S > 1 && !ws))
    return (int)hipErrorInvalidValue;
  if (!pos || !slot || !cos_t || !sin_t || !kc || !vc) return (int)hipErrorInvalidValue;
  if (!mid_rows_ok(A, lda, K) || !mid_rows_ok(B, ldb, K)) return (int)hipErrorInvalidValue;
  const RopeKV rk{pos, slot, cos_t, sin_t, (bf16_t*)kc, (bf16_t*)vc, Hq, Hkv, BS};
  if (S == 1)
    return dispatch_mid<EPI_ROPE_KV>(mi, A, lda, B, ldb, C, ldc, nullptr, nullptr, 0, M, N, K, 1, 0, st, rk);
  const int rc = dispatch_mid<EPI_NONE>(mi, A, lda, B, ldb, ws, N, nullptr, nullptr, 0, M, N, K, S, 1, st);
  if (rc) return rc;
  const long long blocks = ((long long)M * (N >> 4) + 255) / 256;
  hipLaunchKernelGGL(splitk_rope_kernel, dim3((unsigned)blocks), dim3(256), 0, st, ws, S, (bf16_t*)C, ldc, M, N, rk);
  return (int)hipGetLastError();
}
