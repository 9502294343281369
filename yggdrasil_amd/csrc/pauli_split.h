// pauli_split.h -- fp32 sums of products on the bf16 MFMA units, shared by the fp32 Pauli products
// (pauli_split.hip) and their weight gradients (backward.hip).
//
// Every value is cut into three bf16 parts, hi + mid + lo = v exactly, and six of the nine
// products of parts are added: what is left out is below 2^-23 of a product, typically
// 2^-26.  Nothing is scaled, so a value keeps its 24 bits whatever its neighbours are.
// The six products of 32 terms are summed from zero, the small ones first, and then added to
// the accumulator by the vector units: one rounding of a full sum per 32 terms, where the fp32
// MFMA (K = 2) rounds 16 times.  The bf16 MFMAs cut the low bits of a sum off towards minus
// infinity, some 2^-27 of it: every other step computes the negative of its sum, which cancels
// that (the bias gradient of the up product, which adds a thousand rows of such errors, at 8192
// tokens, d = 128, F = 512, E = 32, k = 4: 1.0e-6 off float64 without, 3.8e-7 with; 4.2e-7 on the fp32 units).
#pragma once

#include "pauli_common.h"

namespace ygg {

typedef __attribute__((address_space(3))) void sp_lds_t;
// 16 bytes per lane from buffer `r` at byte `off` + `soff` to LDS address `lds` + 16 lane
__device__ __forceinline__ void split_dma(__amdgpu_buffer_rsrc_t r, uint32_t lds, uint32_t off, uint32_t soff) {
  const uint32_t m0 = __builtin_amdgcn_readfirstlane(lds), so = __builtin_amdgcn_readfirstlane(soff);
  asm volatile("s_mov_b32 m0, %1\n\tbuffer_load_dwordx4 %0, %2, %3 offen lds" ::"v"(off), "s"(m0), "s"(r), "s"(so)
               : "m0", "memory");
}
// this wave's loads have landed and its LDS reads returned; behind the barrier, every wave's
__device__ __forceinline__ void split_wait() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// a value of the step's sign
__device__ __forceinline__ float split_flip(float v, uint32_t neg) {
  return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, v) ^ neg);
}

// The operand of 32 terms (this lane's eight) as its parts: two rows (or inputs) h of two pairs each
__device__ __forceinline__ void split_operand(uint4 (&A)[3], int h, float x0, float y0, float x1, float y1) {
  uint32_t p[3], q[3];
  split_pair(x0, y0, p[0], p[1], p[2]);
  split_pair(x1, y1, q[0], q[1], q[2]);
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    if (h == 0) { A[i].x = p[i]; A[i].y = q[i]; }
    else { A[i].z = p[i]; A[i].w = q[i]; }
  }
}
// The operands of the real and the imaginary sum, (p, s0 q) and (s1 q, p) for pairs p and q
template <uint32_t NEG0, uint32_t NEG1>
__device__ __forceinline__ void split_operands(uint4 (&B)[2][3], int h, float p0, float p1, float q0, float q1) {
  uint32_t p[3], q[3];
  split_pair(p0, p1, p[0], p[1], p[2]);
  split_pair(q0, q1, q[0], q[1], q[2]);
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    if (h == 0) {
      B[0][i].x = p[i]; B[0][i].y = q[i] ^ NEG0;
      B[1][i].x = q[i] ^ NEG1; B[1][i].y = p[i];
    } else {
      B[0][i].z = p[i]; B[0][i].w = q[i] ^ NEG0;
      B[1][i].z = q[i] ^ NEG1; B[1][i].w = p[i];
    }
  }
}

// acc[r][s][q] += sign (A[r] . B[q]) for the NA operands A, two at a time
template <int NA, int NR, int NS>
__device__ __forceinline__ void split_accumulate(pf32x4_t (&acc)[NR][NS][2], int s, const uint4 (&A)[NA][3],
                                                 const uint4 (&B)[2][3], float sign) {
#pragma unroll
  for (int rp = 0; rp < NA / 2; ++rp) {
    pf32x4_t t[2][2];
#pragma unroll
    for (int o = 0; o < 6; ++o) {
      constexpr int kPa[6] = {2, 0, 1, 1, 0, 0}, kPb[6] = {0, 2, 1, 0, 1, 0};  // the small products first
#pragma unroll
      for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const pf32x4_t from = o == 0 ? pf32x4_t{0.f, 0.f, 0.f, 0.f} : t[r][q];
          t[r][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(pbf16x8_t, A[2 * rp + r][kPa[o]]),
                                                            __builtin_bit_cast(pbf16x8_t, B[q][kPb[o]]), from, 0, 0, 0);
        }
    }
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int q = 0; q < 2; ++q) acc[2 * rp + r][s][q] += sign * t[r][q];
  }
}

}  // namespace ygg
