// pauli_small.hip -- bf16 Pauli expert products of few rows (decode and short prompts).
//
// The same products as pauli_gemm.hip (layouts there), cut for the case where the weights
// are read once or a few times and set the time: its 64 x 64 tiles walk the whole
// contraction in one workgroup, so a few tiles leave most of the chip idle behind a chain
// of K / 8 steps (16 tokens, 64 experts, d = 256, F = 1024, k = 2: up 26, down 64 us for 105 MB
// of weights each, 21 us at the rate of a large copy).
//
// A workgroup of 4 waves owns 16 tokens x 32 output multivectors; the waves split the
// contraction, and gridDim.z splits it further into fp32 partial planes that the combine
// adds.  Bound by the weight stream, so every wave runs its own: chunks of 32 columns x
// 8 inputs (128 bytes a column, whole lines, eight columns per instruction) go straight
// to LDS into a ring of four that no other wave touches -- no barrier in the loop, three
// chunks (12 KiB) a wave in flight, 96 KiB a CU.  Loading the operands into registers
// instead takes 16 bytes from each of 32 columns per instruction and reached 2.8-3.5 TB/s
// of weights, this 4.5 TB/s over a whole layer call (64 tokens, 64 experts, d = 256,
// F = 1024: 537 MB in 119 us, 153 with the 64 x 64 tiles; 16 tokens 67, 113 with them).  The activations of a wave's range (at most 8 chunks at a
// time) are read into registers first; several row tiles of an expert read its weights
// through the XCD's L2 (a column tile's row tiles run on one XCD when the column tiles are
// a multiple of 8).

#include <algorithm>

#include "pauli_common.h"
#include "ygg_common.h"

namespace ygg {
namespace {

constexpr int kSmWaves = 4, kSmTok = 16, kSmCols = 32;
constexpr int kSmRing = 4;                 // chunks in a wave's ring
constexpr int kSmChunk = kSmCols * 128;    // bytes: 8 inputs of 32 columns
constexpr int kSmPhase = 8;                // chunks whose activations are held in registers
enum SmallOut : int { kSmPauliRows = 0, kSmPlanes = 1 };

// The tile-th tile of TOK rows over the experts' ranges: one lane per expert counts its
// tiles, a scan finds the one that holds it.
template <int TOK>
__device__ __forceinline__ bool small_find_tile(const int32_t* __restrict__ offsets, int E, int tile, int lane, int& e,
                                                int& row0, int& row_end) {
  const int beg = lane < E ? offsets[lane] : 0, end = lane < E ? offsets[lane + 1] : 0;
  const int nt = (end - beg + TOK - 1) / TOK;
  int incl = nt;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int v = __shfl_up(incl, o);
    if (lane >= o) incl += v;
  }
  const uint64_t after = __ballot(incl > tile);
  if (after == 0) return false;
  e = (int)__builtin_ctzll(after);  // the first expert whose tiles reach past `tile`
  const int b = __builtin_amdgcn_readlane(beg, e);
  row0 = b + (tile - (__builtin_amdgcn_readlane(incl, e) - __builtin_amdgcn_readlane(nt, e))) * TOK;
  row_end = __builtin_amdgcn_readlane(end, e);
  return true;
}

typedef __attribute__((address_space(3))) void sm_lds_t;
// 16 bytes per lane from buffer `r` at byte `off` + `soff` to lds + 16 lane
__device__ __forceinline__ void small_dma(__amdgpu_buffer_rsrc_t r, unsigned char* lds, uint32_t off, uint32_t soff) {
  const uint32_t m0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(sm_lds_t*)lds);
  const uint32_t so = __builtin_amdgcn_readfirstlane(soff);
  asm volatile("s_mov_b32 m0, %1\n\tbuffer_load_dwordx4 %0, %2, %3 offen lds" ::"v"(off), "s"(m0), "s"(r), "s"(so)
               : "m0", "memory");
}
// at most N of this wave's loads outstanding, and every LDS read returned
template <int N>
__device__ __forceinline__ void small_wait() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"i"(N) : "memory");
}
__device__ __forceinline__ int small_swz(int c) { return (c ^ (c >> 3)) & 7; }

template <int ACT, int OUT>
__global__ __launch_bounds__(64 * kSmWaves, 2) void pauli_small_kernel(
    const uint16_t* __restrict__ X, uint32_t x_bytes, const int32_t* __restrict__ gather, const uint16_t* __restrict__ Wp,
    const float* __restrict__ bias, const int32_t* __restrict__ offsets, int E, int d_in, int d_out, int P_max,
    void* __restrict__ Y) {
  constexpr int TOK = kSmTok;
  constexpr int RING = kSmRing * kSmChunk;
  __shared__ __attribute__((aligned(1024))) unsigned char smem[kSmWaves * RING];
  typedef float4 part_t[2 * TOK][kSmCols + 1];  // (a0 re, a0 im, a1 re, a1 im) of two waves, over the rings
  part_t* const part = reinterpret_cast<part_t*>(smem);
  static_assert(2 * sizeof(part_t) <= sizeof(smem), "partial sums over the rings");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, g = lane >> 5;
  const int n_ct = (d_out + kSmCols - 1) / kSmCols;
  const int ct = blockIdx.x % n_ct, rt = blockIdx.x / n_ct;
  int e, row0, row_end;
  if (!small_find_tile<TOK>(offsets, E, rt, lane, e, row0, row_end)) return;
  const int col0 = ct * kSmCols;
  const int IP = d_in >> 1, chunks = (IP + 3) >> 2;

  const __amdgpu_buffer_rsrc_t x_rsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(X), (short)0, x_bytes, kBufferFlags);
  const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(Wp) + (size_t)e * d_out * IP * 16, (short)0, (uint32_t)d_out * IP * 32, kBufferFlags);
  // GEMM row l32 = (token, b): its half-row; rows past the expert's range repeat the last
  const int m = min(row0 + (l32 >> 1), row_end - 1);
  const int src = gather ? gather[m] : m;
  const uint32_t a_row = (uint32_t)(2 * src + (l32 & 1)) * d_in * 8;

  // this (split, wave)'s chunks [c0, c0 + n)
  const int per_split = (chunks + gridDim.z - 1) / gridDim.z;
  const int c_beg = blockIdx.z * per_split, c_end = min(chunks, c_beg + per_split);
  const int per_wave = (max(c_end - c_beg, 0) + kSmWaves - 1) / kSmWaves;
  const int c0 = c_beg + wave * per_wave;
  const int n = __builtin_amdgcn_readfirstlane(max(0, min(c_end, c0 + per_wave) - c0));

  // W pieces of this lane: columns 8 u + lane / 8, piece (pair, a) lane % 8 through the
  // swizzle that keeps the operand reads free of bank conflicts.  A column past d_out lies
  // past the expert's range and reads zero.
  unsigned char* const ring = smem + wave * RING;
  uint32_t w_off[4];
  int w_lim[4];  // the piece is inside the contraction while its chunk's first pair is below this
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int c = 8 * u + (lane >> 3), piece = (lane & 7) ^ small_swz(c);
    w_off[u] = (uint32_t)(col0 + c) * IP * 32 + piece * 16;
    w_lim[u] = IP - (piece >> 1);
  }
  auto issue = [&](int i) __attribute__((always_inline)) {  // the i-th chunk of the range
    const int p0 = (c0 + i) * 4;
    unsigned char* st = ring + (i & (kSmRing - 1)) * kSmChunk;
#pragma unroll
    for (int u = 0; u < 4; ++u)
      small_dma(w_rsrc, st + u * 1024, p0 < w_lim[u] ? w_off[u] : kBufferOff, (uint32_t)p0 * 32);
  };
  // operand reads: column l32, pair 2 s + g, a
  uint32_t w_rd[2][2];
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int a = 0; a < 2; ++a) w_rd[s][a] = l32 * 128 + ((2 * (2 * s + g) + a) ^ small_swz(l32)) * 16;

  pf32x16_t acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[a][q][v] = 0.f;

  for (int ph = 0; ph < n; ph += kSmPhase) {
    uint4 x[kSmPhase][2];
#pragma unroll
    for (int i = 0; i < kSmPhase; ++i)
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const int p = (c0 + ph + i) * 4 + 2 * s + g;
        x[i][s] = __builtin_bit_cast(
            uint4, __builtin_amdgcn_raw_buffer_load_b128(x_rsrc, ph + i < n && p < IP ? a_row + (uint32_t)p * 16 : kBufferOff,
                                                         0, 0));
      }
    if (ph == 0) {
      if (n > 0) issue(0);
      if (n > 1) issue(1);
      if (n > 2) issue(2);
    }
#pragma unroll
    for (int i = 0; i < kSmPhase; ++i) {
      const int c = ph + i;
      if (c < n) {
        // chunk c has landed (later ones stay in flight); the slot of chunk c - 1 has been
        // read by this wave and takes chunk c + 3
        if (n - 1 - c >= 2) small_wait<8>();
        else if (n - 1 - c == 1) small_wait<4>();
        else small_wait<0>();
        if (c + 3 < n) issue(c + 3);
        const unsigned char* st = ring + (c & (kSmRing - 1)) * kSmChunk;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const uint4 v = x[i][s];
          const uint4 vr = make_uint4(rot_conj(v.x), rot_conj(v.y), rot_conj(v.z), rot_conj(v.w));
          const pbf16x8_t A0 = __builtin_bit_cast(pbf16x8_t, v), A1 = __builtin_bit_cast(pbf16x8_t, vr);
#pragma unroll
          for (int a = 0; a < 2; ++a) {
            const pbf16x8_t B = __builtin_bit_cast(pbf16x8_t, *reinterpret_cast<const uint4*>(st + w_rd[s][a]));
            acc[a][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A0, B, acc[a][0], 0, 0, 0);
            acc[a][1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A1, B, acc[a][1], 0, 0, 0);
          }
        }
      }
    }
  }
  __syncthreads();  // every wave is through with its ring

  // the waves' sums: 2 and 3 into 0 and 1, then both from LDS
  auto row_of = [&](int v) { return 8 * (v >> 2) + 4 * g + (v & 3); };
  if (wave >= 2) {
#pragma unroll
    for (int v = 0; v < 16; ++v)
      part[wave - 2][row_of(v)][l32] = make_float4(acc[0][0][v], acc[0][1][v], acc[1][0][v], acc[1][1][v]);
  }
  __syncthreads();
  if (wave < 2) {
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      float4* q = &part[wave][row_of(v)][l32];
      const float4 o = *q;
      *q = make_float4(acc[0][0][v] + o.x, acc[0][1][v] + o.y, acc[1][0][v] + o.z, acc[1][1][v] + o.w);
    }
  }
  __syncthreads();
#pragma unroll
  for (int h = 0; h < TOK * kSmCols / (64 * kSmWaves); ++h) {
    const int o = tid + h * 64 * kSmWaves, t = o / kSmCols, jj = o % kSmCols;
    const int row = row0 + t, j = col0 + jj;
    if (row >= row_end || j >= d_out) continue;
    float4 u0 = part[0][2 * t][jj], u1 = part[0][2 * t + 1][jj];
    const float4 w0 = part[1][2 * t][jj], w1 = part[1][2 * t + 1][jj];
    u0.x += w0.x; u0.y += w0.y; u0.z += w0.z; u0.w += w0.w;
    u1.x += w1.x; u1.y += w1.y; u1.z += w1.z; u1.w += w1.w;
    float y[8];
    pauli_to_blade(u0.x, u0.y, u1.x, u1.y, u0.z, u0.w, u1.z, u1.w, y);
    if (bias != nullptr && (OUT != kSmPlanes || blockIdx.z == 0)) {
#pragma unroll
      for (int c = 0; c < 8; ++c) y[c] += bias[((size_t)e * d_out + j) * 8 + blade_to_mask(c)];
    }
    if constexpr (OUT == kSmPauliRows) {
      activate_blade<ACT>(y);
      float c0[4], c1[4];
      blade_to_pauli(y, c0, c1);
      uint16_t* q = static_cast<uint16_t*>(Y) + ((size_t)row * 2 * d_out + j) * 4;
      *reinterpret_cast<uint2*>(q) = make_uint2(pack2_bf16(c0[0], c0[1]), pack2_bf16(c0[2], c0[3]));
      *reinterpret_cast<uint2*>(q + (size_t)d_out * 4) = make_uint2(pack2_bf16(c1[0], c1[1]), pack2_bf16(c1[2], c1[3]));
    } else {
      float4* q = reinterpret_cast<float4*>(static_cast<float*>(Y) +
                                            (((size_t)blockIdx.z * P_max + row) * d_out + j) * 8);
      q[0] = make_float4(y[0], y[1], y[2], y[3]);
      q[1] = make_float4(y[4], y[5], y[6], y[7]);
    }
  }
}

long long small_row_tiles(int P, int E) { return std::min<long long>(P, (P + kSmTok - 1) / kSmTok + E); }  // at most

template <int ACT, int OUT>
int launch_small(const void* x, int x_rows, const int32_t* gather, int P, const void* w, const float* bias,
                 const int32_t* offsets, int E, int d_in, int d_out, int splits, void* y, hipStream_t st) {
  const dim3 grid((unsigned)(small_row_tiles(P, E) * ((d_out + kSmCols - 1) / kSmCols)), 1, splits);
  const uint16_t* X = static_cast<const uint16_t*>(x);
  const uint16_t* W = static_cast<const uint16_t*>(w);
  const uint32_t xb = (uint32_t)((size_t)x_rows * d_in * 16);
  pauli_small_kernel<ACT, OUT><<<grid, 64 * kSmWaves, 0, st>>>(X, xb, gather, W, bias, offsets, E, d_in, d_out, P, y);
  return check_launch("pauli_small");
}

}  // namespace

// splits of the down product's contraction: as many as leave a wave eight chunks (64
// inputs), planes of at most 16 MiB
int pauli_small_splits(int P, int E, int d_in, int d_out) {
  (void)E;
  long long s = (d_in + 8 * kSmPhase * kSmWaves - 1) / (8 * kSmPhase * kSmWaves);
  s = std::min<long long>(s, ((long long)16 << 20) / std::max<long long>(1, (long long)P * d_out * 32));
  return (int)std::max<long long>(1, std::min<long long>(s, 8));
}

bool pauli_small_pays(int N, int P, int E, int d, int F) {
  const uint64_t lim = (uint64_t)1 << 31;
  return P >= 1 && P <= kPauliSmallRows && (uint64_t)(std::max(d, F) + 64) * std::min(d, F) * 16 < lim &&
         (uint64_t)P * std::max(d, F) * 16 < lim && (uint64_t)N * d * 16 < lim;
}

int pauli_small_up(const void* x, int x_rows, const int32_t* gather, int P, const void* w, const float* bias,
                   const int32_t* offsets, int E, int d_in, int d_out, int act, void* h, hipStream_t stream) {
#define YGG_PS(A) \
  return launch_small<A, kSmPauliRows>(x, x_rows, gather, P, w, bias, offsets, E, d_in, d_out, 1, h, stream)
  switch (act) {
    case kActNone: YGG_PS(kActNone);
    case kActGelu: YGG_PS(kActGelu);
    case kActRelu: YGG_PS(kActRelu);
    default: YGG_PS(kActSigmoid);
  }
#undef YGG_PS
}

int pauli_small_down(const void* h, int P, const void* w, const float* bias, const int32_t* offsets, int E, int d_in,
                     int d_out, int splits, float* planes, hipStream_t stream) {
  return launch_small<kActNone, kSmPlanes>(h, P, nullptr, P, w, bias, offsets, E, d_in, d_out, splits, planes, stream);
}

}  // namespace ygg
