// pauli_tile.h -- a tile of the bf16 Pauli products: its description, the start of its
// accumulators and its epilogue, shared by the 64 x 64 tiles (pauli_gemm.hip) and the
// products of few rows (pauli_small.hip), which give the same outputs bit for bit.
#pragma once

#include "pauli_common.h"

namespace ygg {

enum PauliIn : int { kInBladeGather = 0, kInPauliRows = 1 };
enum PauliOut : int { kOutPauliRows = 0, kOutBlade = 1 };

struct PauliTileInfo {
  int e, row0, row_end, col0;
  int half;  // -1: the whole tile; 0 / 1: only row block `half` of every wave
  // a compact tile (the last row tile of an expert, at most 32 rows): computed as a
  // half tile (block 0 of every wave), its rows staged at the token slots that block
  // covers, 0-15 and 32-47, so wave row group wt holds rows 16 wt .. 16 wt + 15
  bool compact = false;
};

// One output multivector from its eight sums (a0b0, a0b1, a1b0, a1b1 as re, im pairs): the inverse
// Pauli map, the bias unless the sums started from it, the activation and the output layout,
// stored at v_off + s_off of y_rsrc.
template <int ACT, int OUT, int OUT_DT, bool BIAS_IN_ACC>
__device__ __forceinline__ void pauli_store_mv(float a0b0r, float a0b0i, float a0b1r, float a0b1i, float a1b0r, float a1b0i,
                                               float a1b1r, float a1b1i, const float* bv, __amdgpu_buffer_rsrc_t y_rsrc,
                                               uint32_t v_off, uint32_t s_off, int d_out) {
  typedef unsigned int pu32x2_t __attribute__((ext_vector_type(2)));
  typedef unsigned int pu32x4_t __attribute__((ext_vector_type(4)));
  float y[8];
  pauli_to_blade(a0b0r, a0b0i, a0b1r, a0b1i, a1b0r, a1b0i, a1b1r, a1b1i, y);
  if constexpr (!BIAS_IN_ACC) {
#pragma unroll
    for (int c = 0; c < 8; ++c) y[c] += bv[c];
  }
  activate_blade<ACT>(y);
  if constexpr (OUT == kOutPauliRows) {
    float c0[4], c1[4];
    blade_to_pauli(y, c0, c1);
    const pu32x2_t h0 = {pack2_bf16(c0[0], c0[1]), pack2_bf16(c0[2], c0[3])};
    const pu32x2_t h1 = {pack2_bf16(c1[0], c1[1]), pack2_bf16(c1[2], c1[3])};
    __builtin_amdgcn_raw_buffer_store_b64(h0, y_rsrc, v_off, s_off, 0);
    __builtin_amdgcn_raw_buffer_store_b64(h1, y_rsrc, v_off + (uint32_t)d_out * 8, s_off, 0);
  } else if constexpr (OUT_DT == kBF16) {
    const pu32x4_t o = {pack2_bf16(y[0], y[1]), pack2_bf16(y[2], y[3]), pack2_bf16(y[4], y[5]), pack2_bf16(y[6], y[7])};
    __builtin_amdgcn_raw_buffer_store_b128(o, y_rsrc, v_off, s_off, 0);
  } else {
    const pu32x4_t lo = {__builtin_bit_cast(unsigned, y[0]), __builtin_bit_cast(unsigned, y[1]),
                         __builtin_bit_cast(unsigned, y[2]), __builtin_bit_cast(unsigned, y[3])};
    const pu32x4_t hi = {__builtin_bit_cast(unsigned, y[4]), __builtin_bit_cast(unsigned, y[5]),
                         __builtin_bit_cast(unsigned, y[6]), __builtin_bit_cast(unsigned, y[7])};
    __builtin_amdgcn_raw_buffer_store_b128(lo, y_rsrc, v_off, s_off, 0);
    __builtin_amdgcn_raw_buffer_store_b128(hi, y_rsrc, v_off + 16, s_off, 0);
  }
}

// Epilogue of one tile for one wave: the inverse Pauli map, bias, grade-wise
// activation and the output layout, all in the lane that holds the 8 reals of
// an output multivector.  acc[rb][cb][a][re/im] is wave row block rb (of WR,
// each 16 tokens x b = 0, 1), column block cb (of WC, 32 output multivectors);
// bv[cb] is the bias of this lane's column in blade order, added here unless
// BIAS_IN_ACC (the accumulators started from it).  The output is written by
// buffer stores: y_rsrc starts at output row `row_base` and ends at the output's
// true end, the row-dependent part of each offset is a scalar, the lane's part a
// fixed per-lane offset.
template <int ACT, int OUT, int OUT_DT, int WR, int WC, int BWT, bool BIAS_IN_ACC>
__device__ __forceinline__ void pauli_tile_epilogue(const pf32x16_t (&acc)[WR][WC][2][2], const float (&bvs)[WC][8],
                                                    const PauliTileInfo& ti, int wave, int g, int l32, int d_out,
                                                    __amdgpu_buffer_rsrc_t y_rsrc, int row_base) {
  const int wt = wave % BWT, wj = wave / BWT;
  // bytes per output row (Pauli half-row pair, bf16 blade or fp32 blade row)
  constexpr int MV_BYTES = (OUT == kOutPauliRows || OUT_DT == kBF16) ? 16 : 32;
#pragma unroll
  for (int cb = 0; cb < WC; ++cb) {
    const int j = ti.col0 + (wj * WC + cb) * 32 + l32;
    if (j >= d_out) continue;
    const float* bv = bvs[cb];
    // lane part of the offset: token 2 g of the group of four, column j
    const uint32_t v_off = OUT == kOutPauliRows ? (uint32_t)((4 * g) * d_out + j) * 8
                                                : (uint32_t)((2 * g) * d_out + j) * MV_BYTES;
#pragma unroll
    for (int rb = 0; rb < WR; ++rb) {
      if (ti.half >= 0 && rb > 0) break;  // a half tile: the first accumulators hold block `half`
      const int rbr = ti.half >= 0 ? ti.half : rb;
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int rs = ti.row0 + (ti.compact ? wt * 16 : (wt * WR + rbr) * 16) + 4 * q + h;  // row of lanes with g = 0
          if (rs + 2 * g >= ti.row_end) continue;
          const uint32_t s_off = (uint32_t)(rs - row_base) * d_out * MV_BYTES;
          const int v0 = 4 * q + 2 * h;  // b = 0 at v0, b = 1 at v0 + 1
          pauli_store_mv<ACT, OUT, OUT_DT, BIAS_IN_ACC>(
              acc[rb][cb][0][0][v0], acc[rb][cb][0][1][v0], acc[rb][cb][0][0][v0 + 1], acc[rb][cb][0][1][v0 + 1],
              acc[rb][cb][1][0][v0], acc[rb][cb][1][1][v0], acc[rb][cb][1][0][v0 + 1], acc[rb][cb][1][1][v0 + 1], bv, y_rsrc,
              v_off, s_off, d_out);
        }
    }
  }
}

// What the accumulators of a tile start from: entry (a, b) of the halved Pauli matrix of the
// lane's column bias, re and im (the weights hold W / 2, so the products are half the Pauli
// matrices and pauli_to_blade needs no scale).
__device__ __forceinline__ void pauli_bias_entries(const float (&bv)[8], float (&e)[2][2][2]) {  // [a][re/im][b]
  float c0[4], c1[4];
  blade_to_pauli(bv, c0, c1);  // c0 = (M00, M10), c1 = (M01, M11)
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int ri = 0; ri < 2; ++ri) {
      e[a][ri][0] = 0.5f * c0[2 * a + ri];
      e[a][ri][1] = 0.5f * c1[2 * a + ri];
    }
}
template <int WR, int WC>
__device__ __forceinline__ void pauli_acc_from_bias(pf32x16_t (&acc)[WR][WC][2][2], const float (&bvs)[WC][8]) {
#pragma unroll
  for (int cb = 0; cb < WC; ++cb) {
    float e[2][2][2];
    pauli_bias_entries(bvs[cb], e);
#pragma unroll
    for (int rb = 0; rb < WR; ++rb)
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int ri = 0; ri < 2; ++ri)
#pragma unroll
          for (int v = 0; v < 16; ++v) acc[rb][cb][a][ri][v] = e[a][ri][v & 1];
  }
}

}  // namespace ygg
