// pauli_split.hip -- fp32 operands of the Pauli products as two fp16 parts, for the
// split products of pauli_gemm.hip.
//
// A Pauli entry v of a row whose largest entry lies in [2^m, 2^(m+1)) is scaled by 2^s,
// s = 14 - m, and stored as hi = fp16(2^s v) and lo = fp16(2^s v - hi), each rounded to
// nearest even: together 22 bits, v (1 + 2^-23) or closer while |v| is within 2^-16 of
// the row's largest, and within 2^-39 of that largest below.  (The entries of a row with
// a non-finite value are stored unscaled: the row's outputs are then not finite either.)
//
// These kernels are bound by memory (they read fp32 operands once and write as many
// bytes); the second pass over a row, after its maximum is known, hits the caches.

#include <algorithm>

#include "pauli_common.h"

namespace ygg {
namespace {

// entries of a weight multivector as the product's B operand: per a, (c0 u, c0 -v,
// c1 u, c1 -v) of W / 2 (the 1/2 makes the inverse map a plain sum)
__device__ __forceinline__ void w_entries(const float* w8, float (&e0)[4], float (&e1)[4]) {
  float x[8], c0[4], c1[4];
#pragma unroll
  for (int c = 0; c < 8; ++c) x[c] = 0.5f * w8[c];
  blade_to_pauli(x, c0, c1);  // c0 = (M00, M10), c1 = (M01, M11)
  e0[0] = c0[0]; e0[1] = -c0[1]; e0[2] = c1[0]; e0[3] = -c1[1];
  e1[0] = c0[2]; e1[1] = -c0[3]; e1[2] = c1[2]; e1[3] = -c1[3];
}

__device__ __forceinline__ void load8(const float* p, float (&v)[8]) {
  const float4 a = reinterpret_cast<const float4*>(p)[0], b = reinterpret_cast<const float4*>(p)[1];
  v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}

// One output channel's weights, d_in blade multivectors at w, by one wave.
__device__ void split_w_channel(const float* __restrict__ w, int d_in, int lane, unsigned char* __restrict__ out,
                                int32_t* __restrict__ col_exp) {
  uint32_t m = 0;
  for (int i = lane; i < d_in; i += 64) {
    float v[8], e0[4], e1[4];
    load8(w + (size_t)i * 8, v);
    w_entries(v, e0, e1);
#pragma unroll
    for (int q = 0; q < 4; ++q) m = max(m, max(mag_bits(e0[q]), mag_bits(e1[q])));
  }
  const int s = split_exp(__builtin_bit_cast(float, wave_max_u32(m)));
  if (lane == 0) *col_exp = s;
  const int d_pad = (d_in + 7) / 8 * 8;
  for (int i = lane; i < d_pad; i += 64) {
    float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, e0[4], e1[4];
    if (i < d_in) load8(w + (size_t)i * 8, v);
    w_entries(v, e0, e1);
    uint2 h0, l0, h1, l1;
    split4_f16(e0, s, h0, l0);
    split4_f16(e1, s, h1, l1);
    unsigned char* p = out + (size_t)(i >> 3) * 256 + ((i >> 1) & 3) * 32 + (i & 1) * 8;
    *reinterpret_cast<uint2*>(p) = h0;
    *reinterpret_cast<uint2*>(p + 16) = h1;
    *reinterpret_cast<uint2*>(p + 128) = l0;
    *reinterpret_cast<uint2*>(p + 144) = l1;
  }
}

// ---- prepared weights (format 4) -> split weights ------------------------------------
// Workgroup: 8 channels of one expert, thread (input t / 8 of 32, channel t % 8); the
// first pass takes each channel's largest entry, the second writes 32 inputs at a time
// through LDS (the source is contiguous over channels, the result over inputs).
__global__ __launch_bounds__(256) void split_weights_kernel(const float* __restrict__ w, int d_out, int d_in,
                                                            const float* __restrict__ bias,
                                                            unsigned char* __restrict__ out,
                                                            int32_t* __restrict__ col_exp, float* __restrict__ norms) {
  __shared__ uint32_t mx[32][8];
  __shared__ float sq[32][8];
  __shared__ int se[8];
  __shared__ uint2 tile[8][4][32];  // [channel][block of 8 inputs][256 bytes]
  const int nb = (d_out + 7) / 8, e = blockIdx.x / nb, jb = blockIdx.x - e * nb;
  const int t = threadIdx.x, ii = t >> 3, jj = t & 7, j = jb * 8 + jj, jc = min(j, d_out - 1);
  // (u, v) of every entry: the k = 0 record of (e, i, j)
  const float* src = w + (((size_t)e * d_in * 2) * d_out + jc) * 8;
  const size_t step = (size_t)2 * d_out * 8;
  uint32_t m = 0;
#pragma unroll 4
  for (int i = ii; i < d_in; i += 32) {
    float v[8];
    load8(src + i * step, v);
#pragma unroll
    for (int c = 0; c < 8; ++c) m = max(m, mag_bits(v[c]));
  }
  mx[ii][jj] = m;
  __syncthreads();
  if (t < 8) {
    for (int r = 1; r < 32; ++r) m = max(m, mx[r][t]);
    se[t] = split_exp(__builtin_bit_cast(float, m));
    if (jb * 8 + t < d_out) col_exp[(size_t)e * d_out + jb * 8 + t] = se[t];
  }
  __syncthreads();
  const int s = se[jj];
  float n2 = 0.f;
  const size_t rec = pauli_split_row_bytes(d_in);  // bytes per channel
  const int d_pad = (d_in + 7) & ~7;
  float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (ii < d_in) load8(src + ii * step, v);
  for (int i0 = 0; i0 < d_pad; i0 += 32) {
    // v: [c][a][(u, v)]; the operand is (u, -v) per (a, c)
    const float e0[4] = {v[0], -v[1], v[4], -v[5]}, e1[4] = {v[2], -v[3], v[6], -v[7]};
    if (norms != nullptr) {
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        const float x = __builtin_ldexpf(v[c], s);
        n2 += x * x;
      }
    }
    uint2 h0, l0, h1, l1;
    split4_f16(e0, s, h0, l0);
    split4_f16(e1, s, h1, l1);
    const int b8 = ii >> 3, p = ((ii >> 1) & 3) * 4 + (ii & 1);  // 8-byte pieces: pair record, input of the pair
    tile[jj][b8][p] = h0;
    tile[jj][b8][p + 2] = h1;
    tile[jj][b8][p + 16] = l0;
    tile[jj][b8][p + 18] = l1;
    const int in = i0 + 32 + ii;  // the next inputs load while these are written
#pragma unroll
    for (int c = 0; c < 8; ++c) v[c] = 0.f;
    if (in < d_in) load8(src + in * step, v);
    __syncthreads();
    const int oj = t >> 5, ob = (t >> 3) & 3, oq = (t & 7) * 4;  // 32 bytes per thread
    if (jb * 8 + oj < d_out && i0 + ob * 8 < d_pad) {
      const uint2* q = &tile[oj][ob][oq];
      uint4* dst = reinterpret_cast<uint4*>(out + ((size_t)e * d_out + jb * 8 + oj) * rec + (size_t)(i0 / 8 + ob) * 256 + oq * 8);
      dst[0] = make_uint4(q[0].x, q[0].y, q[1].x, q[1].y);
      dst[1] = make_uint4(q[2].x, q[2].y, q[3].x, q[3].y);
    }
    __syncthreads();
  }
  if (norms == nullptr) return;
  sq[ii][jj] = n2;
  __syncthreads();
  if (t < 8) {
    float a = 0.f, b = 0.f;
    for (int r = 0; r < 32; ++r) a += sq[r][t];
    // Frobenius norm of the matrices of W (its halves are stored: 2 |W / 2|)
    a = __builtin_ldexpf(2.f * __builtin_sqrtf(a), -se[t]);
    if (bias != nullptr) {
      const float* bp = bias + ((size_t)e * d_out + min(jb * 8 + t, d_out - 1)) * 8;
      for (int c = 0; c < 8; ++c) b = fmaxf(b, fabsf(bp[c]));
      b *= 2.8284272f;  // at least the norm of the eight
    }
#pragma unroll
    for (int o = 4; o > 0; o >>= 1) {
      a = fmaxf(a, __shfl_xor(a, o));
      b = fmaxf(b, __shfl_xor(b, o));
    }
    if (t == 0) {
      norms[(size_t)e * 2 * nb + jb] = a;
      norms[(size_t)e * 2 * nb + nb + jb] = b;
    }
  }
}

// ---- fp32 blade rows -> split rows ------------------------------------------------------
// One wave per row, a multivector per lane and pass.
//
// The exponent of a slot's hidden row comes from a bound, so that the up product's
// epilogue can write it before the row's maximum is known.  In Frobenius norms of the
// complex matrices |M(y_j)| <= |M(W_j)| |M(x)| + |M(b_j)|; the activations do not enlarge a
// component (sigmoid's stay within 1), and an entry of M(h) is at most its norm.  The
// bound is some 2^4 above the largest entry in practice, which leaves the parts their 22
// bits down to 2^-12 of it.
__global__ __launch_bounds__(256) void split_rows_kernel(const float* __restrict__ x, int N, int d,
                                                         unsigned char* __restrict__ out,
                                                         int32_t* __restrict__ row_exp, SplitHidden hid) {
  const int lane = threadIdx.x & 63, t = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= N) return;
  const float* row = x + (size_t)t * d * 8;
  uint32_t m = 0;
  for (int i = lane; i < d; i += 64) {
    float v[8];
    load8(row + (size_t)i * 8, v);
    m = max(m, pauli_mag(v));
  }
  const int s = split_exp(__builtin_bit_cast(float, wave_max_u32(m)));
  const int d_pad = (d + 7) & ~7;
  unsigned char* o = out + (size_t)t * pauli_split_row_bytes(d);
  float n2 = 0.f;
  for (int i = lane; i < d_pad; i += 64) {
    float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, c0[4], c1[4];
    if (i < d) load8(row + (size_t)i * 8, v);
    blade_to_pauli(v, c0, c1);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const float a = __builtin_ldexpf(c0[c], s), b = __builtin_ldexpf(c1[c], s);
      n2 += a * a + b * b;
    }
    store_split_mv(o, d_pad, i, v, s);
  }
  if (hid.k == 0) {
    if (lane == 0) row_exp[t] = s;
    if (hid.one_offsets != nullptr && t == 0 && lane < 2) hid.one_offsets[lane] = lane * N;
    return;
  }
#pragma unroll
  for (int q = 32; q > 0; q >>= 1) n2 += __shfl_xor(n2, q);
  const float xn = __builtin_ldexpf(__builtin_sqrtf(n2), -s);
  const int nb = (hid.d_ff + 7) / 8;
  for (int q = 0; q < hid.k; ++q) {
    const int e = hid.topk_idx[(size_t)t * hid.k + q];
    float a = 0.f, b = 0.f;
    for (int u = lane; u < nb; u += 64) {
      a = fmaxf(a, hid.norms[(size_t)e * 2 * nb + u]);
      b = fmaxf(b, hid.norms[(size_t)e * 2 * nb + nb + u]);
    }
#pragma unroll
    for (int u = 32; u > 0; u >>= 1) {
      a = fmaxf(a, __shfl_xor(a, u));
      b = fmaxf(b, __shfl_xor(b, u));
    }
    if (lane == 0) {
      // 1.5: |M(b)| = sqrt(2) |b|, and the rounding of the sums behind it
      float bound = 1.01f * (a * xn) + 1.5f * b;
      if (hid.act == kActSigmoid) bound = fmaxf(bound, 3.f);
      const int r = hid.slot_pos[(size_t)t * hid.k + q];
      row_exp[r] = s;
      hid.h_exp[r] = bound == INFINITY ? 15 - 128 : split_exp(bound);
    }
  }
}

constexpr int kGmKBlock = 64;  // inputs whose maxima one workgroup of the first launch takes

// geom_matmul, first launch: workgroups [0, wblocks) split the weight rows of a (four
// channels each); the others take the largest Pauli entry of each column of b over a
// block of 64 inputs.
__global__ __launch_bounds__(256) void split_gm_first_kernel(const float* __restrict__ a, const float* __restrict__ b,
                                                             int M, int K, int N, int wblocks,
                                                             unsigned char* __restrict__ w, int w_stride,
                                                             int32_t* __restrict__ col_exp,
                                                             float* __restrict__ partial,
                                                             int32_t* __restrict__ offsets) {
  const int t = threadIdx.x;
  if ((int)blockIdx.x < wblocks) {
    const int j = blockIdx.x * 4 + (t >> 6);
    if (j < M) split_w_channel(a + (size_t)j * K * 8, K, t & 63, w + (size_t)j * w_stride, col_exp + j);
    return;
  }
  __shared__ uint32_t mx[8][32];
  const int nb = (N + 31) / 32, q = blockIdx.x - wblocks, kb = q / nb, n = (q - kb * nb) * 32 + (t & 31);
  if (q == 0 && t == 0) {
    offsets[0] = 0;
    offsets[1] = N;
  }
  uint32_t m = 0;
  if (n < N) {
#pragma unroll
    for (int u = 0; u < kGmKBlock / 8; ++u) {
      const int k = kb * kGmKBlock + u * 8 + (t >> 5);
      if (k < K) {
        float v[8];
        load8(b + ((size_t)k * N + n) * 8, v);
        m = max(m, pauli_mag(v));
      }
    }
  }
  mx[t >> 5][t & 31] = m;
  __syncthreads();
  if (t < 32 && n < N) {
#pragma unroll
    for (int r = 1; r < 8; ++r) m = max(m, mx[r][t]);
    partial[(size_t)kb * N + n] = __builtin_bit_cast(float, m);
  }
}

// geom_matmul, second launch: b (K, N) blade -> split rows of its transpose.  Tiles of 32
// columns x 8 inputs through LDS, so the reads (32 consecutive columns of one input) and
// the writes (one block of a half-row, 128 bytes) are contiguous.
__global__ __launch_bounds__(256) void split_gm_rows_kernel(const float* __restrict__ b, int K, int N,
                                                            const float* __restrict__ partial,
                                                            unsigned char* __restrict__ x,
                                                            int32_t* __restrict__ row_exp) {
  __shared__ uint2 tile[32][2][2][8];  // [column][b][hi, lo][input]
  __shared__ int se[32];
  const int n0 = blockIdx.x * 32, k0 = blockIdx.y * 8, t = threadIdx.x;
  if (t < 32) {
    const int n = n0 + t;
    uint32_t m = 0;
    if (n < N)
      for (int kb = 0; kb * kGmKBlock < K; ++kb)
        m = max(m, __builtin_bit_cast(uint32_t, partial[(size_t)kb * N + n]));
    se[t] = split_exp(__builtin_bit_cast(float, m));
    if (k0 == 0 && n < N) row_exp[n] = se[t];
  }
  const int kk = t >> 5, nn = t & 31;
  float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, c0[4], c1[4];
  if (k0 + kk < K && n0 + nn < N) load8(b + ((size_t)(k0 + kk) * N + n0 + nn) * 8, v);
  blade_to_pauli(v, c0, c1);
  __syncthreads();
  split4_f16(c0, se[nn], tile[nn][0][0][kk], tile[nn][0][1][kk]);
  split4_f16(c1, se[nn], tile[nn][1][0][kk], tile[nn][1][1][kk]);
  __syncthreads();
  // thread: column t / 8, half-row b, hi or lo part, its half: 32 bytes
  const int wn = t >> 3, wb = (t >> 2) & 1, part = (t >> 1) & 1, hf = t & 1;
  if (n0 + wn < N) {  // (the block's padding inputs were read as zero)
    const int dv = 2 * ((K + 7) / 8 * 8);
    const uint2* s = &tile[wn][wb][part][hf * 4];
    uint4* dst = reinterpret_cast<uint4*>(x + ((size_t)(n0 + wn) * 2 + wb) * dv * 8 + (size_t)(k0 / 8) * 128 +
                                          part * 64 + hf * 32);
    dst[0] = make_uint4(s[0].x, s[0].y, s[1].x, s[1].y);
    dst[1] = make_uint4(s[2].x, s[2].y, s[3].x, s[3].y);
  }
}

}  // namespace
}  // namespace ygg

using namespace ygg;

int ygg::pauli_split_weights(const float* w, int E, int d_out, int d_in, const float* bias, void* out, int32_t* col_exp,
                             float* norms, hipStream_t stream) {
  split_weights_kernel<<<(unsigned)(E * ((d_out + 7) / 8)), 256, 0, stream>>>(
      w, d_out, d_in, bias, static_cast<unsigned char*>(out), col_exp, norms);
  return check_launch("pauli_split_weights");
}

int ygg::pauli_split_rows(const float* x, int N, int d, void* out, int32_t* row_exp, const SplitHidden& hid,
                          hipStream_t stream) {
  if (N == 0) return 0;
  split_rows_kernel<<<(unsigned)((N + 3) / 4), 256, 0, stream>>>(x, N, d, static_cast<unsigned char*>(out), row_exp,
                                                                 hid);
  return check_launch("pauli_split_rows");
}

size_t ygg::pauli_split_gm_partials(int K, int N) { return (size_t)((K + kGmKBlock - 1) / kGmKBlock) * N; }

int ygg::pauli_split_gm_operands(const float* a, const float* b, int M, int K, int N, void* w, int32_t* col_exp,
                                 void* x, int32_t* row_exp, float* partial, int32_t* offsets, hipStream_t stream) {
  const int wblocks = (M + 3) / 4;
  const unsigned bblocks = (unsigned)(((N + 31) / 32) * ((K + kGmKBlock - 1) / kGmKBlock));
  split_gm_first_kernel<<<wblocks + bblocks, 256, 0, stream>>>(a, b, M, K, N, wblocks, static_cast<unsigned char*>(w),
                                                               (int)pauli_split_row_bytes(K), col_exp, partial,
                                                               offsets);
  if (check_launch("pauli_split_gm_first")) return -1;
  split_gm_rows_kernel<<<dim3((unsigned)((N + 31) / 32), (unsigned)((K + 7) / 8)), 256, 0, stream>>>(
      b, K, N, partial, static_cast<unsigned char*>(x), row_exp);
  return check_launch("pauli_split_gm_rows");
}
