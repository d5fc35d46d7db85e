"""Distance between the rows of large weights in device memory.

Blocks that stream a weight walk along its rows side by side: at any moment the whole chip reads the same few columns of
thousands of rows. Rows 4, 8 or 12 KB apart put these on a fraction of the memory channels. With 128 bytes between the rows
(us, 256 rotating MB and more): slabs of the weight stream, 28672 x 4096, 8 / 32 / 64 rows 48.8 / 53.9 / 51.8 -> 38.0 / 39.5 / 43.3,
18688 x 4096 34.6 / 37.9 / 38.9 -> 30.8 / 35.5 / 37.2, 28672 x 2048 28.4 / 29.4 / 31.1 -> 21.1 / 22.5 / 25.0, 28672 x 6144 75 / 75 / 75 ->
56 / 59 / 65; gate/up 28672 x 4096 at 1 / 8 / 32 / 64 rows 43.9 / 42.9 / 44.5 / 51.1 -> 38.9 / 39.2 / 42.3 / 49.7, 36864 x 6144 at 8 / 64
99.9 / 115.2 -> 89.9 / 102.2. Smaller weights end before it shows (9216 x 2048 11.9 -> 12.6 at 32 rows, 6144 x 4096 and 4096 x
4096 the same within 2 %), and rows 10, 14, 16 or 28 KB apart lose instead (18688 x 7168 at 8 rows 52.8 -> 54.7, 28672 x 8192
gate/up 91.6 -> 86.8 but 9216 x 8192 35.5 -> 36.9).

Prompts read the same weights. Gate/up 28672 x 4096 at 65 / 100 / 140 / 200 / 300 rows -3 / +2 / +1 / 0 / +2 %, at 400 to 1400 within 1,
at 1777 / 2200 / 3000 / 5193 / 15576 -1.2 / -0.2 / -0.4 / -0.7 / -0.9; 36864 x 6144 at 300 / 1000 / 5193 -10 / -2 / -1.5, 32768 x 2048 at
300 / 1000 / 3000 / 5193 -4 / -1 / +0.6 / -0.8. The batch-1 decode tail, whose loader keeps to a few rows a block, takes 66.0 -> 65.7 us
a layer on one card and 64.1 -> 64.6 on another.

One byte a value: 4 KB rows that gemm_part streams, 4096 and 6144 x 4096 at 1 / 11 / 50 rows 5.7 / 6.3 / 9.5 and 7.7 / 8.3 / 14.4 -> 5.5 /
6.1 / 9.1 and 7.2 / 7.9 / 13.8; longer rows the same or worse. Gate/up 28672 x 4096 does not mind (held activations, 1 to 64 rows, -0.5
to +0.9 %; tiles, 65 / 140 rows -5 / -6 %, 300 to 5193 -1.3 to +0.4), nor do the tiles of the other two (65 to 5193 rows -1.3 to +0.9).
"""
from __future__ import annotations

import torch

GAP = 128  # bytes between the end of a row and the next one
MIN_BYTES = 1 << 26
ROW_BYTES = (4096, 8192, 12288)
MIN_BYTES_FP8 = 1 << 24
ROW_BYTES_FP8 = (4096,)


def wants_gap(rows, row_bytes, itemsize):
    if itemsize == 1:
        return row_bytes in ROW_BYTES_FP8 and rows * row_bytes >= MIN_BYTES_FP8
    return itemsize == 2 and row_bytes in ROW_BYTES and rows * row_bytes >= MIN_BYTES


def empty_rows(rows, columns, dtype, device):
    """A weight to be filled, laid out as pitched() does it."""
    size = dtype.itemsize
    gap = torch.device(device).type == "cuda" and dtype.is_floating_point and wants_gap(rows, columns * size, size)
    return torch.empty((rows, columns + gap * GAP // size), dtype=dtype, device=device)[:, :columns]


def pitched(w):
    """The weight [rows, columns], or a copy of it whose rows lie GAP bytes further apart, where its products read that faster."""
    size = w.element_size()
    if not (w.is_cuda and w.dim() == 2 and w.is_contiguous() and w.is_floating_point()
            and wants_gap(w.shape[0], w.shape[1] * size, size)):
        return w
    return empty_rows(*w.shape, w.dtype, w.device).copy_(w)
