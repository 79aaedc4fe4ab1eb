// Outputs of single activation rows on the vector units, for the matrix-core
// products whose operand planes do not hold a row.
#pragma once

#include "formats.h"

// Outputs y[m0 + r][c0 .. c1) over the columns [k0, k1) of x and w for each
// row r whose bit is set, by one wave: its lanes share the columns, eight rows
// at a time, products and sums in float64. Such rows are rare, so what counts
// is that the calling kernel's loops stay as they are (no case is slower by
// it); loads in flight bound the rows themselves: 77 rows of 6912 values with
// 2560 rows of F16 take 0.42 ms with one row of them here and 1.65 ms with all
// (31 us with none; 1.3 ms on the vector-unit GEMM).
template <int F>
__device__ __forceinline__ void plain_rows(MatDesc w, const float *x, int64_t ldx, uint64_t rows, int m0, int c0,
                                           int c1, int k0, int k1, float *y, int64_t ldy) {
  w.fmt = F;
  const int lane = threadIdx.x & 63;
  constexpr int R = 8;
  while (rows) {
    int m[R], n = 0;
#pragma unroll
    for (int i = 0; i < R; i++) {  // past the last row: it again, not stored
      m[i] = rows ? m0 + __builtin_ctzll(rows) : m[i > 0 ? i - 1 : 0];
      n += rows != 0;
      rows &= rows - 1;
    }
    for (int c = c0; c < c1; c++) {
      double s[R] = {};
#pragma unroll 4
      for (int k = k0 + lane; k < k1; k += 64) {
        const double v = mat_value(w, c, k);
#pragma unroll
        for (int i = 0; i < R; i++) s[i] += v * x[m[i] * ldx + k];
      }
#pragma unroll
      for (int i = 0; i < R; i++) {
        const double t = wave_total_d(s[i]);
        if (lane == 0 && i < n) y[m[i] * ldy + c] = (float)t;
      }
    }
  }
}
