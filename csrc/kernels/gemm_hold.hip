// Decode gate/up projection with the activations held in registers (gfx950): out[M, N] = act(x . Wg^T, x . Wu^T) over the
// packed [64 gate | 64 up] weight rows, bf16 or fp8 (e4m3fn with a scale a row), a few tens of rows of x.
//
// The weights' stream bounds it; what kept the other kernels from it is the activation block. A block of a few weight rows
// reads all of x again for them: as fragments from L2 (gemm_fp8_dec, gemm_skinny: as many bytes of x as of fp8 weights at 16
// rows) or through the LDS ring (gemm_stream: half of the ring, so half of the weights in flight). Here one block a CU walks
// its whole share of the rows, and each of its eight waves owns an eighth of K for all of them: its fragments of x (16 MT
// rows x K / 8, 16 MT K / 1024 registers a lane) are loaded once and stay, and every load after that is a weight. NB tiles
// of 16 weight rows (8 gate, the 8 up rows they pair with) are in flight in registers, 64 KB of fp8 each at K = 4096; their
// eight partial products meet in LDS, double-buffered, with one barrier a tile that waits for no load.
// Plain loads: non-temporal ones take 27.7 us for 27.5 at 28672 x 4096 fp8, 11 rows. Loading x behind the first weight tile and
// ahead of the others is worth 1 us: in order, the first product would wait for everything in flight.
//
// Nothing in a round of tiles may wait for more than its own loads. Loads behind a branch (the share's end) and the scales, asked
// for at their tile, did: the first makes the compiler wait for all that may be in flight wherever two paths meet, the second in
// order for all weights asked for before it. So the rounds load without a branch (fp8; the last tile again past the end), the
// last round loads nothing and has its own copy, and the scales of a block's tiles come in front of everything into LDS. us,
// before and after: fp8 28672 x 4096 (117 MB) at 11 / 32 rows 26.8 / 32.5 -> 25.8 / 31.2 (4.6 TB/s), 14336 x 4096 17.1 / 21.6 ->
// 15.4 / 20.5, 11264 x 2048 8.1 / 10.6 -> 7.5 / 10.0; bf16 11264 x 2048 (46 MB) at 12 / 32 / 64 rows 11.6 / 14.3 / 17.7 -> 11.1 /
// 13.1 / 17.7 (a block has three tiles there, and a spare load of a fourth would cost 0.5 us: it keeps the branch). Two tiles of
// 64 KB in flight, not three: 27.4 -> 25.9. No more tiles are in flight than a block has, since each spare one is loaded all the
// same: bf16 1024 x 4096 at 1 / 16 rows 10.2 / 12.9 -> 6.9 / 9.6, 4096 x 4096 12.1 / 14.9 -> 9.4 / 11.1, fp8 2048 x 2048 5.4 / 6.7
// -> 4.2 / 5.5, 16384 x 3072 (four tiles, two in flight for three) 12.5 / 13.5 -> 10.3 / 11.4.
//
// More rows than the registers hold (64 of K = 4096 would be a CU's whole register file): SLAB deals the blocks to slabs of 2048
// of K, each with its part of x, and writes fp32 partials of plain weight rows. fp8 28672 x 4096 at 33 / 64 rows: two launches
// 54 / 61 us, slabs 29 / 34 and the pass that sums and pairs them 4.
#include <type_traits>

#include "common.h"
using namespace ragk;

namespace {

constexpr int HW = 8;      // waves of a block, each an eighth of K
constexpr int HCH = 128;   // k of a chunk: wave w owns chunks w, w + 8, ...
constexpr int HTILES = 64; // tiles of a block at most
constexpr int HOLD_LDW = 1 << 24;  // a weight row's stride: a lane's row of a tile is a 32-bit offset

__device__ __forceinline__ unsigned f32pair_to_bf16x2(f32x2 f) {
  return __builtin_amdgcn_perm(__float_as_uint(f[1]), __float_as_uint(f[0]), 0x07060302u);
}
// 8 fp8 -> 8 bf16, exact
__device__ __forceinline__ bf16x8 fp8x8_to_bf16(unsigned lo, unsigned hi) {
  u32x4 r;
  r[0] = f32pair_to_bf16x2(__builtin_amdgcn_cvt_pk_f32_fp8((int)lo, false));
  r[1] = f32pair_to_bf16x2(__builtin_amdgcn_cvt_pk_f32_fp8((int)lo, true));
  r[2] = f32pair_to_bf16x2(__builtin_amdgcn_cvt_pk_f32_fp8((int)hi, false));
  r[3] = f32pair_to_bf16x2(__builtin_amdgcn_cvt_pk_f32_fp8((int)hi, true));
  return __builtin_bit_cast(bf16x8, r);
}

constexpr int hold_regs(int MT, int KI, bool FP8, int NB) { return KI * (16 * MT + (FP8 ? 8 : 16) * NB); }
constexpr int HREGS = 192;  // of a wave's 256: the held x and the weights in flight

// Tiles in flight: three of up to 48 KB if a wave's 256 registers hold them beside x, else two.
constexpr int hold_depth(int MT, int KI, bool FP8) {
  return hold_regs(MT, KI, FP8, 3) <= HREGS && KI * (FP8 ? 1 : 2) < 4 ? 3 : 2;
}

// KI = K / 1024 of a launch (SLAB: of a slab), NB tiles in flight. par: fp32 {limit, alpha, shift} of EPI_GLU_CLIP. SLAB: fp32 slabs
// P[S][M][ldc] of plain weight rows instead, slab blockIdx.y.
template <int MT, int KI, bool FP8, int EPI, bool SLAB, int NB>
__global__ __launch_bounds__(HW * 64, 2) void gemm_hold_kernel(const bf16_t* __restrict__ X, int ldx,
                                                              const unsigned char* __restrict__ W, size_t ldw_bytes,
                                                              const float* __restrict__ sw, void* C, int ldc,
                                                              const bf16_t* __restrict__ par, int M, int tiles, int share) {
  constexpr int L = FP8 ? 2 : 4;     // 16-byte loads of a chunk: 64 contiguous bytes of each row
  constexpr int EB = FP8 ? 1 : 2;
  __shared__ __attribute__((aligned(16))) f32x4 red[2][HW][MT][64];
  __shared__ float scale[FP8 ? HTILES : 1][16];  // asked for at a tile, they would wait for all the weights in flight
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int fr = lane & 15, fh = lane >> 4;
  const int t0 = (int)((long long)tiles * blockIdx.x / share), t1 = (int)((long long)tiles * (blockIdx.x + 1) / share);
  const int k0 = (SLAB ? blockIdx.y * KI * HW : 0) * HCH + w * HCH;
  u32x4 wv[NB][KI][L];
  // lane's row of a tile: output column fr & 7, gate rows in lanes 0-7, up rows in 8-15
  const int lrow = SLAB ? fr : (fr & 7) + (fr >> 3) * 64;
  const unsigned loff = lrow * (unsigned)ldw_bytes + 16 * fh;
  auto first = [&](int t) __attribute__((always_inline)) { return SLAB ? 16 * t : (t >> 3) * 128 + (t & 7) * 8; };
  float sc[HTILES / 32];
  if constexpr (FP8)
#pragma unroll
    for (int j = 0; j < HTILES / 32; ++j) sc[j] = sw[first(min(t0 + 32 * j + (int)(threadIdx.x >> 4), t1 - 1)) + lrow];
  __builtin_amdgcn_sched_barrier(0);
  auto load = [&](u32x4 (&d)[KI][L], int t) __attribute__((always_inline)) {
    const unsigned char* p = W + (size_t)first(t) * ldw_bytes + k0 * EB;
#pragma unroll
    for (int i = 0; i < KI; ++i)
#pragma unroll
      for (int l = 0; l < L; ++l)
        d[i][l] = *reinterpret_cast<const u32x4*>(p + loff + i * HW * HCH * EB + 64 * l);
  };
  load(wv[0], t0);
  // x in the order of the weights: a 16-byte load of fp8 holds the 8 k of two products
  bf16x8 xf[MT][KI][4];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const bf16_t* p = X + (size_t)min(16 * m + fr, M - 1) * ldx + k0;
#pragma unroll
    for (int i = 0; i < KI; ++i)
#pragma unroll
      for (int s = 0; s < 4; ++s)
        xf[m][i][s] = *reinterpret_cast<const bf16x8*>(p + i * HW * HCH + (FP8 ? 64 * (s >> 1) + 16 * fh + 8 * (s & 1)
                                                                              : 32 * s + 8 * fh));
  }
#pragma unroll
  for (int b = 1; b < NB; ++b) load(wv[b], min(t0 + b, t1 - 1));  // behind x: the first tile waits for neither
  if constexpr (NB > 1) __builtin_amdgcn_sched_barrier(0);
  if constexpr (FP8)
#pragma unroll
    for (int j = 0; j < HTILES / 32; ++j) scale[32 * j + (threadIdx.x >> 4)][fr] = sc[j];
  const GluPar gp = glu_par<EPI>(par);
  if (!FP8 && NB > 1 && t0 + NB < t1) {  // x is here before the loop, whose waits would else be for the prologue's order of loads
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int i = 0; i < KI; ++i)
#pragma unroll
        for (int s = 0; s < 4; ++s) asm volatile("" ::"v"(xf[m][i][s]));
  }
  auto tile = [&](u32x4 (&d)[KI][L], int t, auto more) __attribute__((always_inline)) {
    f32x4 acc[MT];
    if (t < t1) {
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[m] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < KI; ++i)
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          bf16x8 wf;
          if constexpr (FP8) wf = fp8x8_to_bf16(d[i][s >> 1][2 * (s & 1)], d[i][s >> 1][2 * (s & 1) + 1]);
          else wf = __builtin_bit_cast(bf16x8, d[i][s]);
#pragma unroll
          for (int m = 0; m < MT; ++m) acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf[m][i][s], wf, acc[m], 0, 0, 0);
        }
    }
    if constexpr (FP8) __builtin_amdgcn_sched_barrier(0);  // the loads stay behind the products that free their registers
    if (decltype(more)::value && (FP8 || t + NB < t1)) load(d, min(t + NB, t1 - 1));
    if (t >= t1) return;
    f32x4 (*rd)[MT][64] = red[(t - t0) & 1];
#pragma unroll
    for (int m = 0; m < MT; ++m) rd[w][m][lane] = acc[m];
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // the buffer's readers passed the barrier before this one
    constexpr int CW = SLAB ? 16 : 8;
#pragma unroll
    for (int e0 = 0; e0 < 16 * MT * CW; e0 += HW * 64) {
      const int e = e0 + (int)threadIdx.x, row = e / CW, c = e % CW;
      if (row >= M || e >= 16 * MT * CW) break;
      const int m = row >> 4, ln = ((row & 15) >> 2) * 16 + c, r = row & 3;
      auto sum = [&](int l) __attribute__((always_inline)) {
        auto two = [&](int g) __attribute__((always_inline)) { return rd[g][m][l][r] + rd[g + 1][m][l][r]; };
        const float v = (two(0) + two(2)) + (two(4) + two(6));
        if constexpr (FP8) return v * scale[t - t0][l & 15];
        return v;
      };
      if constexpr (SLAB) {
        reinterpret_cast<float*>(C)[((size_t)blockIdx.y * M + row) * ldc + 16 * t + c] = sum(ln);
      } else {
        reinterpret_cast<bf16_t*>(C)[(size_t)row * ldc + 8 * t + c] = f2bf(glu_act<EPI>(sum(ln), sum(ln + 8), gp));
      }
    }
  };
  int t = t0;
  for (; t + NB < t1; t += NB)
#pragma unroll
    for (int b = 0; b < NB; ++b) tile(wv[b], t + b, std::true_type{});
#pragma unroll
  for (int b = 0; b < NB; ++b) tile(wv[b], t + b, std::false_type{});
}

// Blocks that share the tiles: one a CU, more where theirs would be more than HTILES.
int hold_share(int tiles, int blocks) { return max(min(tiles, blocks), (tiles + HTILES - 1) / HTILES); }

// Tiles in flight, at most hold_depth: no more than the largest share has, and two of four where three would ask for two spare ones.
template <int DEPTH, typename F>
int hold_with_depth(int tiles, int share, F f) {
  const int per = (tiles + share - 1) / share;
  if (per == 1) f(std::integral_constant<int, 1>{});
  else if (DEPTH == 2 || per == 2 || per == 4) f(std::integral_constant<int, 2>{});
  else f(std::integral_constant<int, DEPTH>{});
  return (int)hipGetLastError();
}

template <int MT, int KI, bool FP8, int EPI>
int launch_hold(const void* X, int ldx, const void* W, int ldw, const float* sw, void* C, int ldc, const void* par, int M,
                int N, int blocks, hipStream_t st) {
  if constexpr (hold_regs(MT, KI, FP8, 2) <= HREGS) {
    const int tiles = N / 8, share = hold_share(tiles, blocks);
    return hold_with_depth<hold_depth(MT, KI, FP8)>(tiles, share, [&](auto nb) {
      hipLaunchKernelGGL((gemm_hold_kernel<MT, KI, FP8, EPI, false, decltype(nb)::value>), dim3(share), dim3(HW * 64), 0, st,
                         (const bf16_t*)X, ldx, (const unsigned char*)W, (size_t)ldw * (FP8 ? 1 : 2), sw, C, ldc, (const bf16_t*)par,
                         M, tiles, share);
    });
  } else {
    return (int)hipErrorInvalidValue;
  }
}

template <int KI, bool FP8, int EPI>
int hold_mt(const void* X, int ldx, const void* W, int ldw, const float* sw, void* C, int ldc, const void* par, int M, int N,
            int blocks, hipStream_t st) {
  switch ((M + 15) / 16) {
    case 1: return launch_hold<1, KI, FP8, EPI>(X, ldx, W, ldw, sw, C, ldc, par, M, N, blocks, st);
    case 2: return launch_hold<2, KI, FP8, EPI>(X, ldx, W, ldw, sw, C, ldc, par, M, N, blocks, st);
    case 3: return launch_hold<3, KI, FP8, EPI>(X, ldx, W, ldw, sw, C, ldc, par, M, N, blocks, st);
    case 4: return launch_hold<4, KI, FP8, EPI>(X, ldx, W, ldw, sw, C, ldc, par, M, N, blocks, st);
    default: return (int)hipErrorInvalidValue;
  }
}

template <bool FP8, int EPI>
int hold_ki(const void* X, int ldx, const void* W, int ldw, const float* sw, void* C, int ldc, const void* par, int M, int N,
            int K, int blocks, hipStream_t st) {
  switch (K / 1024) {
    case 1: return hold_mt<1, FP8, EPI>(X, ldx, W, ldw, sw, C, ldc, par, M, N, blocks, st);
    case 2: return hold_mt<2, FP8, EPI>(X, ldx, W, ldw, sw, C, ldc, par, M, N, blocks, st);
    case 3: return hold_mt<3, FP8, EPI>(X, ldx, W, ldw, sw, C, ldc, par, M, N, blocks, st);
    case 4: return hold_mt<4, FP8, EPI>(X, ldx, W, ldw, sw, C, ldc, par, M, N, blocks, st);
    case 5: return hold_mt<5, FP8, EPI>(X, ldx, W, ldw, sw, C, ldc, par, M, N, blocks, st);
    default: return (int)hipErrorInvalidValue;
  }
}

}  // namespace

// Rows of x that one launch takes (a multiple of 16, at most 64), 0: none.
RAGK_API int ragk_gemm_hold_rows(int K, int fp8) {
  if (K % 1024 || K > 5 * 1024 || K <= 0) return 0;
  int rows = 0;
  for (int mt = 1; mt <= 4; ++mt)
    if (hold_regs(mt, K / 1024, fp8 != 0, 2) <= HREGS) rows = 16 * mt;
  return rows;
}

// epi: EPI_SILU_MUL or EPI_GLU_CLIP (bf16 weights; par fp32 {limit, alpha, shift}). W: 2 N packed rows, sw: their fp32 scales
// (fp8) or null (bf16). N % 64 == 0, 16-byte aligned rows of x and W, M <= ragk_gemm_hold_rows(K, fp8). blocks: one a CU.
RAGK_API int ragk_gemm_hold(const void* X, int ldx, const void* W, int ldw, const float* sw, void* C, int ldc,
                            const void* par, int M, int N, int K, int epi, int blocks, hipStream_t st) {
  if (M <= 0 || N <= 0) return 0;
  if (N % 64 || blocks < 1 || M > ragk_gemm_hold_rows(K, sw != nullptr) || ldx % 8 || ldw % (sw ? 16 : 8) ||
      ldw >= HOLD_LDW)
    return (int)hipErrorInvalidValue;
  if (sw) return epi == EPI_SILU_MUL ? hold_ki<true, EPI_SILU_MUL>(X, ldx, W, ldw, sw, C, ldc, par, M, N, K, blocks, st)
                                     : (int)hipErrorInvalidValue;
  if (epi == EPI_SILU_MUL) return hold_ki<false, EPI_SILU_MUL>(X, ldx, W, ldw, sw, C, ldc, par, M, N, K, blocks, st);
  if (epi == EPI_GLU_CLIP && par) return hold_ki<false, EPI_GLU_CLIP>(X, ldx, W, ldw, sw, C, ldc, par, M, N, K, blocks, st);
  return (int)hipErrorInvalidValue;
}

RAGK_API int ragk_slabs_finish(const float* P, int S, void* C, int ldc, const void* bias, const void* resid, int ldr, int M,
                               int N, int epi, int out_f32, hipStream_t st);

// fp32 slabs P[K / 2048][M][N] of x . W^T, W fp8 with a scale a row: M <= 64, K % 2048 == 0, N % 16 == 0, 16-byte aligned rows.
// blocks: one a CU.
RAGK_API int ragk_gemm_hold_slabs(const void* X, int ldx, const void* W, int ldw, const float* sw, float* P, int M, int N,
                                  int K, int blocks, hipStream_t st) {
  if (M <= 0 || N <= 0) return 0;
  const int S = K / 2048;
  if (M > 64 || K <= 0 || K % 2048 || N % 16 || S > blocks || ldx % 8 || ldw % 16 || ldw >= HOLD_LDW || !sw) return (int)hipErrorInvalidValue;
  const int share = hold_share(N / 16, blocks / S);
  auto launch = [&](auto mt) {
    constexpr int MT = decltype(mt)::value;
    return hold_with_depth<hold_depth(MT, 2, true)>(N / 16, share, [&](auto nb) {
      hipLaunchKernelGGL((gemm_hold_kernel<MT, 2, true, EPI_NONE, true, decltype(nb)::value>), dim3(share, S), dim3(HW * 64), 0, st,
                         (const bf16_t*)X, ldx, (const unsigned char*)W, (size_t)ldw, sw, P, N, nullptr, M, N / 16, share);
    });
  };
  switch ((M + 15) / 16) {
    case 1: return launch(std::integral_constant<int, 1>{});
    case 2: return launch(std::integral_constant<int, 2>{});
    case 3: return launch(std::integral_constant<int, 3>{});
    default: return launch(std::integral_constant<int, 4>{});
  }
}

// The packed gate/up projection (2 N rows of W) through those slabs and a pass that sums and pairs them.
RAGK_API int ragk_gemm_hold_slabs_silu(const void* X, int ldx, const void* W, int ldw, const float* sw, void* C, int ldc, int M,
                                       int N, int K, int blocks, float* ws, hipStream_t st) {
  if (N % 64 || !ws) return (int)hipErrorInvalidValue;
  const int rc = ragk_gemm_hold_slabs(X, ldx, W, ldw, sw, ws, M, 2 * N, K, blocks, st);
  return rc ? rc : ragk_slabs_finish(ws, K / 2048, C, ldc, nullptr, nullptr, 0, M, N, EPI_SILU_MUL, 0, st);
}
