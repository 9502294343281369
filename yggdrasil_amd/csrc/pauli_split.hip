// pauli_split.hip -- fp32 Pauli products of enough rows on the bf16 MFMA units (the sums:
// pauli_split.h), from the operands of pauli_f32.hip: Pauli rows and weights in format 4.
//
// A workgroup of four waves owns 64 tokens x 64 output multivectors, a wave 32 x 32; a step is
// eight inputs: 16 KiB of rows and 16 KiB of weights, direct to LDS, double buffered; the values
// are cut into parts on their way from LDS to the MFMA.  Bound by the MFMAs, at the rate that a
// large library product reaches on the card: 32768 rows, 128 -> 512, 32 experts 749 us, 1.10
// PFLOP/s issued.  geom_matmul 512 x 128 x 8192: 412 us on the fp32 units, 205-225 here, error
// against float64 2.1e-7 and 1.0e-7.

#include <algorithm>
#include <type_traits>

#include "pauli_f32.h"
#include "pauli_split.h"
#include "ygg_common.h"

namespace ygg {
namespace {

constexpr int kSpT = 64, kSpN = 64, kSpK = 8;              // tokens, columns, inputs of a step
constexpr int kSpA = kSpT * kSpK * 32, kSpW = kSpK * kSpN * 32;  // bytes of a stage: rows, weights
constexpr int kSpMaxExperts = 64;

template <int ACT, int OUT>
__global__ __launch_bounds__(256, 2) void pauli_split_kernel(
    const float* __restrict__ X, uint64_t x_bytes, const int32_t* __restrict__ gather, const float* __restrict__ Wp,
    const float* __restrict__ bias, const int32_t* __restrict__ offsets, int E, int d_in, int d_out, int P_max, int n_xcd,
    float* __restrict__ Y, float* __restrict__ Ypre) {
  __shared__ __attribute__((aligned(1024))) unsigned char smem[2 * (kSpA + kSpW)];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // The tiles (row tile of an expert) x (column tile), column tiles first, in one contiguous
  // range per XCD; one lane per expert counts its row tiles, a scan finds the one that holds
  // this workgroup's.
  const int beg = lane < E ? offsets[lane] : 0, end = lane < E ? offsets[lane + 1] : 0;
  const int nt = (end - beg + kSpT - 1) / kSpT;
  int incl = nt;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int v = __shfl_up(incl, o);
    if (lane >= o) incl += v;
  }
  const int CT = (d_out + kSpN - 1) / kSpN;
  const int n_tiles = __builtin_amdgcn_readlane(incl, 63) * CT, per = (n_tiles + n_xcd - 1) / n_xcd;
  const int slot = blockIdx.x / n_xcd, tile = (blockIdx.x - slot * n_xcd) * per + slot;
  if (slot >= per || tile >= n_tiles) return;
  const int rt = tile / CT, col0 = (tile - rt * CT) * kSpN;
  const int e = (int)__builtin_ctzll(__ballot(incl > rt));  // the first expert whose tiles reach past rt
  const int row_end = __builtin_amdgcn_readlane(end, e);
  const int row0 = __builtin_amdgcn_readlane(beg, e) +
                   (rt - (__builtin_amdgcn_readlane(incl, e) - __builtin_amdgcn_readlane(nt, e))) * kSpT;

  // rows: gathered ones index the whole of x (below 2 GiB), rows in place start at the tile's first
  const uint64_t x_first = gather ? 0 : (uint64_t)row0 * d_in * 32, x_left = x_bytes > x_first ? x_bytes - x_first : 0;
  const __amdgpu_buffer_rsrc_t x_rsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(reinterpret_cast<const char*>(X)) + x_first, (short)0,
                                        (uint32_t)(x_left < 0x7fffffffull ? x_left : 0x7fffffffull), kBufferFlags);
  const __amdgpu_buffer_rsrc_t w_rsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(Wp) + (size_t)e * d_in * 2 * d_out * 8, (short)0,
                                        (uint32_t)d_in * 2 * d_out * 32, kBufferFlags);
  // This lane's pieces (16 bytes).  Rows: load u covers tokens 16 wave + 4 u .. + 3, 256 bytes
  // each; LDS slot s of token t holds piece s ^ 2 (t % 8), piece 2 i + b being input i, half b.
  // Weights: load u covers input 2 wave + u / 2 and 32 columns (u % 2); slot 2 j + s of an input's
  // run holds (column j, c = s ^ (j / 8 % 2)).  Both orders keep the operand reads free of conflicts.
  uint32_t a_off[4], w_off[2];
  int a_lim[2];  // (by u % 2) the piece is inside the contraction while the step's first input is below this
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int t = 16 * wave + 4 * u + (lane >> 4), piece = (lane & 15) ^ ((t & 7) << 1);
    const int r = min(row0 + t, row_end - 1);  // rows past the range: computed, not stored
    const int src = gather ? gather[r] : r - row0;
    a_off[u] = (uint32_t)src * d_in * 32 + piece * 16;
    a_lim[u & 1] = d_in - (piece >> 1);
  }
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int j = u * 32 + (lane >> 1), c = (lane & 1) ^ ((j >> 3) & 1);
    w_off[u] = col0 + j < d_out ? (uint32_t)(col0 + j) * 32 + c * 16 : kBufferOff;
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(sp_lds_t*)smem;
  auto issue = [&](int f) __attribute__((always_inline)) {  // step f's operands to stage f % 2
    const uint32_t st = lds0 + (f & 1) * (kSpA + kSpW);
#pragma unroll
    for (int u = 0; u < 4; ++u)
      split_dma(x_rsrc, st + (4 * wave + u) * 1024, f * kSpK < a_lim[u & 1] ? a_off[u] : kBufferOff, (uint32_t)f * 256);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int i = f * kSpK + 2 * wave + (u >> 1);  // uniform; past the contraction: zeros
      split_dma(w_rsrc, st + kSpA + (4 * wave + u) * 1024, i < d_in ? w_off[u & 1] : kBufferOff,
                i < d_in ? (uint32_t)i * 64 * d_out : 0u);
    }
  };

  // Operands of v_mfma_f32_16x16x32_bf16: lane row / column lane % 16, inputs 2 g and 2 g + 1 of
  // the step, g = lane / 16.  A wave's row block rb is tokens 16 rb + 8 wt .. + 7, both halves.
  const int wt = wave & 1, wj = wave >> 1, l16 = lane & 15, g = lane >> 4;
  uint32_t a_rd[2];  // inputs 2 g, 2 g + 1 of token 8 wt + l16 / 2 (+ 4096 per row block)
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int t = 8 * wt + (l16 >> 1);
    a_rd[h] = t * 256 + (((2 * (2 * g + h) + (l16 & 1)) ^ ((t & 7) << 1)) * 16);
  }
  const int jl = wj * 32 + l16;  // (+ 16 per column block: j / 8 % 2 stays)
  const uint32_t w_rd = kSpA + 2 * g * 2048 + jl * 32 + ((jl >> 3) & 1) * 16;  // (c = 0; c = 1 at ^ 16; input 2 g + 1 at + 2048)

  pf32x4_t acc[4][4][2];  // [row block][column block, a][re, im]
#pragma unroll
  for (int rb = 0; rb < 4; ++rb)
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int q = 0; q < 2; ++q) acc[rb][c][q] = pf32x4_t{0.f, 0.f, 0.f, 0.f};

  // A step of NP pairs of row blocks.  (The barriers keep the scheduler from holding more parts
  // than the registers do: the other wave of the SIMD fills the gaps.)
  auto compute = [&](int f, auto pairs_tag) __attribute__((always_inline)) {
    constexpr int NP = decltype(pairs_tag)::value;
    const unsigned char* st = smem + (f & 1) * (kSpA + kSpW);
    const uint32_t neg = (f & 1) << 31;
    uint4 A[2 * NP][3];  // (re c0, re c1), (im c0, im c1) of two inputs
#pragma unroll
    for (int r = 0; r < 2 * NP; ++r)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const float4 x = *reinterpret_cast<const float4*>(st + a_rd[h] + r * 4096);
        split_operand(A[r], h, x.x, x.y, x.z, x.w);
      }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      __builtin_amdgcn_sched_barrier(0);
      uint4 B[2][3];  // (u, -v) for the real part, (v, u) for the imaginary one, of c0 and c1
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const uint32_t off = h * 2048 + (c >> 1) * 512 + (c & 1) * 8;
        const float2 w0 = *reinterpret_cast<const float2*>(st + w_rd + off);         // (u, v), c0
        const float2 w1 = *reinterpret_cast<const float2*>(st + (w_rd ^ 16) + off);  // c1
        split_operands<0x80008000u, 0u>(B, h, split_flip(w0.x, neg), split_flip(w1.x, neg), split_flip(w0.y, neg),
                                        split_flip(w1.y, neg));
      }
      split_accumulate(acc, c, A, B, f & 1 ? -1.f : 1.f);
    }
  };

  const int n = (d_in + kSpK - 1) / kSpK;
  issue(0);
  auto steps = [&](auto pairs_tag) __attribute__((always_inline)) {
    for (int f = 0; f < n; ++f) {
      split_wait();  // step f may be read and the other stage, read by step f - 1, overwritten
      if (f + 1 < n) issue(f + 1);
      compute(f, pairs_tag);
    }
  };
  if (row_end - row0 > 32) steps(std::integral_constant<int, 2>{});
  else steps(std::integral_constant<int, 1>{});  // the tile's upper half holds no rows

#pragma unroll
  for (int cb = 0; cb < 2; ++cb) {
    const int j = col0 + wj * 32 + cb * 16 + l16;
    if (j >= d_out) continue;
#pragma unroll
    for (int rb = 0; rb < 4; ++rb)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int row = row0 + rb * 16 + wt * 8 + 2 * g + h;  // its halves b = 0, 1 are sums 2 h, 2 h + 1
        if (row >= row_end) continue;
        const auto &s0 = acc[rb][2 * cb], &s1 = acc[rb][2 * cb + 1];  // a = 0, 1
        f32_store_mv<ACT, OUT>(s0[0][2 * h], s0[1][2 * h], s0[0][2 * h + 1], s0[1][2 * h + 1], s1[0][2 * h], s1[1][2 * h],
                               s1[0][2 * h + 1], s1[1][2 * h + 1], bias, e, row, j, d_out, 0, P_max, Y, Ypre, nullptr);
      }
  }
}

template <int ACT, int OUT>
int launch_split(const float* x, int x_rows, const int32_t* gather, int P_max, const float* w, const float* bias,
                 const int32_t* offsets, int E, int d_in, int d_out, float* y, float* y_pre, hipStream_t st) {
  const int n_xcd = 8;  // workgroups go to the XCDs round robin (8 on MI355X)
  const long long tiles = ((long long)(P_max + kSpT - 1) / kSpT + E) * ((d_out + kSpN - 1) / kSpN);  // at most
  pauli_split_kernel<ACT, OUT><<<(unsigned)((tiles + n_xcd - 1) / n_xcd * n_xcd), 256, 0, st>>>(
      x, (uint64_t)x_rows * d_in * 32, gather, w, bias, offsets, E, d_in, d_out, P_max, n_xcd, y, y_pre);
  return check_launch("pauli_split");
}

}  // namespace

// One product: from 32 inputs and about 100 tiles of 64 x 64 on.  A tile's steps are a chain of
// some 2.9 us per eight inputs whether one or two share a CU, and fewer tiles leave CUs idle that
// the fp32 MFMA kernel's 16 x 32 tiles use (geom_matmul, us, split / fp32 MFMA: 64 tiles, K = 32 26 / 21, 64
// 37 / 30, 128 61 / 49, 512 196 / 151; 128 tiles 28 / 29, 41 / 46, 67 / 76, 202 / 291; 512 tiles 51 / 72, 76 / 112, 118 / 218,
// 378 / 1060; K = 16: 128 tiles 22 / 19, 512 41 / 47).
bool pauli_split_pays(long long P, int d_in, int d_out) { return d_in >= 32 && P * d_out >= 100LL * 64 * 64; }

// A layer's two products together, whose smaller one may fill less (layer calls, us, split / fp32 MFMA: d =
// 128, F = 512, E = 32: 1024 rows 250 / 191, 2048 277 / 327, 8192 525 / 940; d = F = 128, E = 64: 1024 83 / 81,
// 2048 118 / 132; d = 256, F = 1024, E = 64: 1024 453 / 701).  Layers narrower than 128 keep the fp32 units and
// with them their outputs bit for bit, though 8192 rows of d = 64, F = 256, E = 8 take 274 us there and 187 here:
// through the sigmoid's gate c / |c|, whose derivative has no bound, any other order of the
// sums moves their gradients by up to 1.2e-5.
bool pauli_split_layer_pays(long long P, int E, int d, int F) {
  const int m = std::min(d, F);
  return m >= 128 && P * m >= 60LL * 64 * 64 && P >= 16LL * E;
}

bool pauli_split_fits(int E, long long x_rows, bool gathered, int d_in, int d_out) {
  const uint64_t lim = (uint64_t)1 << 31;
  return E >= 1 && E <= kSpMaxExperts && (uint64_t)(d_in + kSpK) * d_out * 64 < lim &&
         (gathered ? (uint64_t)x_rows * d_in * 32 < lim : (uint64_t)kSpT * d_in * 32 < lim);
}

int pauli_split_linear(const float* x, int x_rows, const int32_t* gather, int P_max, const float* w, const float* bias,
                       const int32_t* offsets, int E, int d_in, int d_out, int act, float* y, int y_layout, float* y_pre,
                       hipStream_t stream) {
  if (y_layout == kF32OutBlade)
    return launch_split<kActNone, kF32OutBlade>(x, x_rows, gather, P_max, w, bias, offsets, E, d_in, d_out, y, nullptr, stream);
  if (y_layout == kF32OutBladeT)
    return launch_split<kActNone, kF32OutBladeT>(x, x_rows, gather, P_max, w, bias, offsets, E, d_in, d_out, y, nullptr, stream);
#define YGG_SU(A) \
  return launch_split<A, kF32OutPauliRows>(x, x_rows, gather, P_max, w, bias, offsets, E, d_in, d_out, y, y_pre, stream)
  switch (act) {
    case kActNone: YGG_SU(kActNone);
    case kActGelu: YGG_SU(kActGelu);
    case kActRelu: YGG_SU(kActRelu);
    default: YGG_SU(kActSigmoid);
  }
#undef YGG_SU
}

}  // namespace ygg
