// pauli_f32.h -- output layouts and the store of the fp32 Pauli products (pauli_f32.hip on the
// fp32 MFMA units, pauli_split.hip on the bf16 ones).
#pragma once

#include "pauli_common.h"

namespace ygg {

enum PauliF32Out : int { kF32OutPauliRows = 0, kF32OutBlade = 1, kF32OutPartial = 2, kF32OutBladeT = 3 };

// One output multivector (token row, column j) from its Pauli sums Y[a][b] = (re, im):
// blade map, bias (split 0 only for partial planes), the pre-activation rows when
// Ypre is set, activation, and the store in the OUT layout.
template <int ACT, int OUT>
__device__ inline void f32_store_mv(float y00r, float y00i, float y01r, float y01i, float y10r, float y10i, float y11r,
                                    float y11i, const float* __restrict__ bias, int e, int row, int j, int d_out,
                                    int split, int P_max, float* __restrict__ Y, float* __restrict__ Ypre,
                                    const int32_t* __restrict__ row_map) {
  float y[8];
  pauli_to_blade(y00r, y00i, y01r, y01i, y10r, y10i, y11r, y11i, y);
  if (bias != nullptr && (OUT != kF32OutPartial || split == 0)) {
#pragma unroll
    for (int c = 0; c < 8; ++c) y[c] += bias[((size_t)e * d_out + j) * 8 + blade_to_mask(c)];
  }
  if constexpr (OUT == kF32OutPauliRows) {
    if (Ypre != nullptr) {  // the pre-activation rows, blade order (kept for the backward)
      float4* q = reinterpret_cast<float4*>(Ypre + ((size_t)row * d_out + j) * 8);
      q[0] = make_float4(y[0], y[1], y[2], y[3]);
      q[1] = make_float4(y[4], y[5], y[6], y[7]);
    }
    activate_blade<ACT>(y);
    float c0[4], c1[4];
    blade_to_pauli(y, c0, c1);  // c0 = (M00, M10), c1 = (M01, M11)
    float4* q = reinterpret_cast<float4*>(Y + ((size_t)row * d_out + j) * 8);  // [b][k][c]
    q[0] = make_float4(c0[0], c0[2], c0[1], c0[3]);
    q[1] = make_float4(c1[0], c1[2], c1[1], c1[3]);
  } else {
    size_t mv = OUT == kF32OutBladeT ? (size_t)j * P_max + row : (size_t)row * d_out + j;
    if constexpr (OUT == kF32OutPartial)  // partial planes: at row_map[row] when given (slot rows)
      mv = (size_t)split * P_max * d_out + (size_t)(row_map != nullptr ? row_map[row] : row) * d_out + j;
    else activate_blade<ACT>(y);
    float4* p = reinterpret_cast<float4*>(Y + mv * 8);
    p[0] = make_float4(y[0], y[1], y[2], y[3]);
    p[1] = make_float4(y[4], y[5], y[6], y[7]);
  }
}

}  // namespace ygg
