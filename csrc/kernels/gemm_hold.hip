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
// 28672 x 4096 fp8 (117 MB), 11 rows: 38 -> 27.5 us (4.3 TB/s), 32 rows 37 -> 33; 11264 x 2048 bf16 (46 MB), 12 rows 14.7 ->
// 11.8, 50 rows 24 -> 17. Plain loads: non-temporal ones take 27.7, 33.2, 12.7 and 17.3. Loading x behind the first weight
// tile and ahead of the others is worth 1 us: in order, the first product would wait for everything in flight.
#include "common.h"
using namespace ragk;

namespace {

constexpr int HW = 8;      // waves of a block, each an eighth of K
constexpr int HCH = 128;   // k of a chunk: wave w owns chunks w, w + 8, ...

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

// KI = K / 1024. par: fp32 {limit, alpha, shift} of EPI_GLU_CLIP.
template <int MT, int KI, bool FP8, int EPI>
__global__ __launch_bounds__(HW * 64, 2) void gemm_hold_kernel(const bf16_t* __restrict__ X, int ldx,
                                                              const unsigned char* __restrict__ W, size_t ldw_bytes,
                                                              const float* __restrict__ sw, bf16_t* __restrict__ C, int ldc,
                                                              const bf16_t* __restrict__ par, int M, int tiles) {
  const GluPar gp = glu_par<EPI>(par);
  constexpr int NB = hold_regs(MT, KI, FP8, 3) <= HREGS ? 3 : 2;
  constexpr int L = FP8 ? 2 : 4;     // 16-byte loads of a chunk: 64 contiguous bytes of each row
  constexpr int EB = FP8 ? 1 : 2;
  __shared__ __attribute__((aligned(16))) f32x4 red[2][HW][MT][64];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int fr = lane & 15, fh = lane >> 4;
  const int t0 = (int)((long long)tiles * blockIdx.x / gridDim.x), t1 = (int)((long long)tiles * (blockIdx.x + 1) / gridDim.x);
  u32x4 wv[NB][KI][L];
  auto load = [&](u32x4 (&d)[KI][L], int t) __attribute__((always_inline)) {
    const int c = 8 * t + (fr & 7);  // output column of this lane's weight row: gate rows in lanes 0-7, up rows in 8-15
    const unsigned char* p = W + (size_t)((c >> 6) * 128 + (c & 63) + (fr >> 3) * 64) * ldw_bytes + w * HCH * EB + 16 * fh;
#pragma unroll
    for (int i = 0; i < KI; ++i)
#pragma unroll
      for (int l = 0; l < L; ++l)
        d[i][l] = *reinterpret_cast<const u32x4*>(p + i * HW * HCH * EB + 64 * l);
  };
  load(wv[0], t0);
  // x in the order of the weights: a 16-byte load of fp8 holds the 8 k of two products
  bf16x8 xf[MT][KI][4];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const bf16_t* p = X + (size_t)min(16 * m + fr, M - 1) * ldx + w * HCH;
#pragma unroll
    for (int i = 0; i < KI; ++i)
#pragma unroll
      for (int s = 0; s < 4; ++s)
        xf[m][i][s] = *reinterpret_cast<const bf16x8*>(p + i * HW * HCH + (FP8 ? 64 * (s >> 1) + 16 * fh + 8 * (s & 1)
                                                                              : 32 * s + 8 * fh));
  }
#pragma unroll
  for (int b = 1; b < NB; ++b)
    if (t0 + b < t1) load(wv[b], t0 + b);  // behind x: the first tile waits for neither
  auto tile = [&](u32x4 (&d)[KI][L], int t) __attribute__((always_inline)) {
    f32x4 acc[MT];
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
    if (t + NB < t1) load(d, t + NB);
    f32x4 (*rd)[MT][64] = red[(t - t0) & 1];
#pragma unroll
    for (int m = 0; m < MT; ++m) rd[w][m][lane] = acc[m];
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // the buffer's readers passed the barrier before this one
    for (int e = threadIdx.x; e < 128 * MT; e += HW * 64) {
      const int row = e >> 3, c = e & 7;
      if (row >= M) break;
      const int ln = ((row & 15) >> 2) * 16 + c, r = row & 3, m = row >> 4;
      float v = 0.f, u = 0.f;
#pragma unroll
      for (int g = 0; g < HW; ++g) {
        v += rd[g][m][ln][r];
        u += rd[g][m][ln + 8][r];
      }
      const int col = 8 * t + c;
      if constexpr (FP8) {
        const int pr = (col >> 6) * 128 + (col & 63);
        v *= sw[pr];
        u *= sw[pr + 64];
      }
      C[(size_t)row * ldc + col] = f2bf(glu_act<EPI>(v, u, gp));
    }
  };
  for (int t = t0; t < t1; t += NB) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      if (t + b >= t1) break;
      tile(wv[b], t + b);
    }
  }
}

template <int MT, int KI, bool FP8, int EPI>
int launch_hold(const void* X, int ldx, const void* W, int ldw, const float* sw, void* C, int ldc, const void* par, int M,
                int N, int blocks, hipStream_t st) {
  if constexpr (hold_regs(MT, KI, FP8, 2) <= HREGS) {
    const int tiles = N / 8;
    hipLaunchKernelGGL((gemm_hold_kernel<MT, KI, FP8, EPI>), dim3(min(tiles, blocks)), dim3(HW * 64), 0, st, (const bf16_t*)X,
                       ldx, (const unsigned char*)W, (size_t)ldw * (FP8 ? 1 : 2), sw, (bf16_t*)C, ldc, (const bf16_t*)par, M, tiles);
    return (int)hipGetLastError();
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
  if (N % 64 || blocks < 1 || M > ragk_gemm_hold_rows(K, sw != nullptr) || ldx % 8 || ldw % (sw ? 16 : 8))
    return (int)hipErrorInvalidValue;
  if (sw) return epi == EPI_SILU_MUL ? hold_ki<true, EPI_SILU_MUL>(X, ldx, W, ldw, sw, C, ldc, par, M, N, K, blocks, st)
                                     : (int)hipErrorInvalidValue;
  if (epi == EPI_SILU_MUL) return hold_ki<false, EPI_SILU_MUL>(X, ldx, W, ldw, sw, C, ldc, par, M, N, K, blocks, st);
  if (epi == EPI_GLU_CLIP && par) return hold_ki<false, EPI_GLU_CLIP>(X, ldx, W, ldw, sw, C, ldc, par, M, N, K, blocks, st);
  return (int)hipErrorInvalidValue;
}
