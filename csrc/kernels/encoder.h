// The arguments of one sentence encoder forward.
#pragma once
#include "common.h"

namespace ragk {

constexpr int FEW_T = 32, FEW_H = 1024;  // rows and columns that encoder_few.hip takes

// Launches of one product: rows r0 .. r1 on gemm_mid (tile mi, S slabs), gemm_w4 (mi 0: 256 rows a tile, or 32 + rows / 32) or the
// decode kernels (mi -1).
struct Piece { int r0, r1, mi, S; };
struct Plan { int n, slabs; Piece p[2]; };  // slabs: p[0].S fp32 slabs of all rows for the norm behind it

// (mirrored by ops/_lib.py EncoderCall)
struct EncoderCall {
  const void *word, *pos_table, *type_row, *ln_g, *ln_b;
  const void* const* layers;  // 12 a layer: wqkv bqkv wo bo ln1_g ln1_b wi bi wo2 bo2 ln2_g ln2_b
  const int *ids, *pos, *cu, *lens, *tiles, *rows;  // rows: output row of every sequence
  const int* ids_host;                              // few: the ids if they are not on the device (ids null)
  void *h, *a, *qkv, *attn, *f;
  float *ws, *out;
  float* y;  // few: [T][H]
  int n_layers, T, B, H, I, heads, n_tiles, pooling, normalize, ldo;
  int few, first_pos;  // few: encoder_few.hip's launches, into the row that out points at
  int l0, l1;          // few: this call's layers of n_layers (l1 0: the last), calls in order sharing their buffers
  float eps;
  Plan plans[4];  // qkv, attention output, up, down
};

int encoder_few_forward(const EncoderCall& c, hipStream_t st);

}  // namespace ragk
