// pauli_small.hip -- bf16 Pauli expert products of few rows (decode and short prompts).
//
// The products of pauli_gemm.hip (layouts there), cut for the case where the weights are
// read once or a few times and set the time: the 64 x 64 tiles walk the whole contraction
// in one workgroup of two per CU, so a few tiles leave most of the chip idle.
//
// A wave owns 8 RB tokens x 16 CB output multivectors and is a workgroup of its own: nothing
// is shared, so there is no barrier, and every wave runs its own stream of chunks of 8
// inputs (weights 128 bytes a column, activations 64 bytes a half-row) straight to LDS into a
// ring of RING; the operands of chunk c + 1 are read from LDS while chunk c is multiplied.
// Bound by the chain of a wave's steps at the smallest sizes and by the weight stream above.
// Several row tiles of an expert read its weights through the XCD's L2 (a column tile's row
// tiles run on one XCD when the column tiles are a multiple of 8).
//
// An output element is the 64 x 64 tiles' chain of sums: the contraction is not cut, the
// bias enters where theirs does, and a 16 x 16 x 32 MFMA gives the bits of their two chained
// 32 x 32 x 16 ones (2^25 sums of random inputs over up to 60 binades compared, all the same).
// So a row's outputs do not depend on which of the two kernels its batch takes.

#include <algorithm>
#include <type_traits>

#include "pauli_tile.h"
#include "ygg_common.h"

namespace ygg {
namespace {

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
__device__ __forceinline__ uint32_t small_lds(const unsigned char* p) { return (uint32_t)(uintptr_t)(const sm_lds_t*)p; }
// 16 (or 4) bytes per lane from buffer `r` at byte `off` + `soff` to LDS address `lds` + 16 (4) lane
template <int BYTES>
__device__ __forceinline__ void small_dma(__amdgpu_buffer_rsrc_t r, uint32_t lds, uint32_t off, uint32_t soff) {
  const uint32_t m0 = __builtin_amdgcn_readfirstlane(lds), so = __builtin_amdgcn_readfirstlane(soff);
  if constexpr (BYTES == 4)
    asm volatile("s_mov_b32 m0, %1\n\tbuffer_load_dword %0, %2, %3 offen lds" ::"v"(off), "s"(m0), "s"(r), "s"(so)
                 : "m0", "memory");
  else
    asm volatile("s_mov_b32 m0, %1\n\tbuffer_load_dwordx4 %0, %2, %3 offen lds" ::"v"(off), "s"(m0), "s"(r), "s"(so)
                 : "m0", "memory");
}
// at most N of this wave's loads outstanding, and every LDS read returned
template <int N>
__device__ __forceinline__ void small_wait() {
  static_assert(N >= 0 && N < 64, "vmcnt field");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"i"(N) : "memory");
}
__device__ __forceinline__ int small_swz(int c) { return (c ^ (c >> 3)) & 7; }

template <int ACT, int OUT, bool BIAS_FIRST, int RB, int CB, int RING>
__global__ __launch_bounds__(64) void pauli_small_kernel(
    const uint16_t* __restrict__ X, uint32_t x_bytes, const int32_t* __restrict__ gather, const uint16_t* __restrict__ Wp,
    const float* __restrict__ bias, const int32_t* __restrict__ offsets, int E, int d_in, int d_out, int P_max,
    void* __restrict__ Y) {
  constexpr int TOK = 8 * RB, COLS = 16 * CB;
  constexpr int W_BYTES = COLS * 128, CHUNK = W_BYTES + TOK * 128;  // 8 inputs of the columns, then of the half-rows
  constexpr int WL = W_BYTES / 1024, LOADS = CHUNK / 1024;          // direct loads of 64 x 16 bytes
  __shared__ __attribute__((aligned(1024))) unsigned char smem[RING * CHUNK + 1024 + 256];
  unsigned char* const s_bias = smem + RING * CHUNK;  // 32 bytes a column
  unsigned char* const s_gather = s_bias + 1024;      // a row index per lane
  const int lane = threadIdx.x, l16 = lane & 15, g = lane >> 4;
  const int n_ct = (d_out + COLS - 1) / COLS;
  const int ct = blockIdx.x % n_ct, rt = blockIdx.x / n_ct;
  int e, row0, row_end;
  if (!small_find_tile<TOK>(offsets, E, rt, lane, e, row0, row_end)) return;
  const int col0 = ct * COLS;
  const int IP = d_in >> 1;
  const int n = 2 * ((IP + 7) >> 3);  // chunks of four pairs: an even number, as the 64 x 64 tiles' steps

  const __amdgpu_buffer_rsrc_t x_rsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(X), (short)0, x_bytes, kBufferFlags);
  const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(Wp) + (size_t)e * d_out * IP * 16, (short)0, (uint32_t)d_out * IP * 32, kBufferFlags);
  const __amdgpu_buffer_rsrc_t b_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(bias), (short)0, bias ? (uint32_t)E * d_out * 32 : 0u, kBufferFlags);
  const __amdgpu_buffer_rsrc_t g_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<int32_t*>(gather), (short)0, gather ? (uint32_t)P_max * 4 : 0u, kBufferFlags);

  // Weights: piece u of this lane is column 8 u + lane / 8, (pair, a) lane % 8 through the
  // swizzle that keeps the operand reads free of bank conflicts.  A column past d_out lies
  // past the expert's range and reads zero; so does a pair past the contraction.
  const uint32_t lds0 = small_lds(smem);
  uint32_t w_off[WL], a_off[RB];
  int w_lim[WL], a_lim[RB];  // the piece is inside the contraction while its chunk's first pair is below this
#pragma unroll
  for (int u = 0; u < WL; ++u) {
    const int c = 8 * u + (lane >> 3), piece = (lane & 7) ^ small_swz(c);
    w_off[u] = (uint32_t)(col0 + c) * IP * 32 + piece * 16;
    w_lim[u] = IP - (piece >> 1);
  }
  auto issue_w = [&](int c, int slot, int u) __attribute__((always_inline)) {  // piece u of chunk c to ring slot `slot`
    small_dma<16>(w_rsrc, lds0 + slot * CHUNK + u * 1024, c * 4 < w_lim[u] ? w_off[u] : kBufferOff, (uint32_t)c * 128);
  };
  // Activations: piece u is half-row 16 u + lane / 4 (token, b), pair lane % 4 through a swizzle
  auto issue_a = [&](int c, int slot) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < RB; ++u)
      small_dma<16>(x_rsrc, lds0 + slot * CHUNK + W_BYTES + u * 1024, c * 4 < a_lim[u] ? a_off[u] : kBufferOff, (uint32_t)c * 64);
  };

  // The prologue asks for the row indices and the bias, then the weights of the first chunks,
  // and, when the indices are here, those chunks' activations.
  const int my_row = min(row0 + (lane & (TOK - 1)), row_end - 1);  // past the range: the last row again
  small_dma<4>(g_rsrc, small_lds(s_gather), (uint32_t)my_row * 4, 0);
  small_dma<16>(b_rsrc, small_lds(s_bias),
                lane < 2 * COLS && col0 + (lane >> 1) < d_out ? (uint32_t)(e * d_out + col0) * 32 + lane * 16 : kBufferOff, 0);
#pragma unroll
  for (int c = 0; c < RING - 1; ++c)
#pragma unroll
    for (int u = 0; u < WL; ++u) issue_w(c, c, u);
  small_wait<WL * (RING - 1) + 1>();
#pragma unroll
  for (int u = 0; u < RB; ++u) {
    const int r = 16 * u + (lane >> 2), piece = (lane & 3) ^ ((r >> 2) & 3), tok = r >> 1;
    const int src = gather ? reinterpret_cast<const int*>(s_gather)[tok] : min(row0 + tok, row_end - 1);
    a_off[u] = (uint32_t)(2 * src + (r & 1)) * d_in * 8 + piece * 16;
    a_lim[u] = IP - piece;
  }
#pragma unroll
  for (int c = 0; c < RING - 1; ++c) issue_a(c, c);

  // operands of v_mfma_f32_16x16x32_bf16: lane column / half-row lane % 16, pair lane / 16
  uint32_t w_rd[CB][2], a_rd[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) a_rd[rb] = W_BYTES + (rb * 16 + l16) * 64 + (g ^ (l16 >> 2)) * 16;
#pragma unroll
  for (int cb = 0; cb < CB; ++cb)
#pragma unroll
    for (int a = 0; a < 2; ++a) w_rd[cb][a] = (cb * 16 + l16) * 128 + ((2 * g + a) ^ small_swz(cb * 16 + l16)) * 16;
  struct Ops {
    uint4 x[RB], w[CB][2];
  };
  auto read_x = [&](const unsigned char* st, Ops& o) __attribute__((always_inline)) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) o.x[rb] = *reinterpret_cast<const uint4*>(st + a_rd[rb]);
  };
  auto read_w = [&](const unsigned char* st, Ops& o, int cb) __attribute__((always_inline)) {
#pragma unroll
    for (int a = 0; a < 2; ++a) o.w[cb][a] = *reinterpret_cast<const uint4*>(st + w_rd[cb][a]);
  };
  pf32x4_t acc[RB][CB][2][2];
  auto mma = [&](const Ops& o, int cb, int q) __attribute__((always_inline)) {  // q: real or imaginary part
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      const uint4 v = o.x[rb];
      const uint4 vr = q == 0 ? v : make_uint4(rot_conj(v.x), rot_conj(v.y), rot_conj(v.z), rot_conj(v.w));
      const pbf16x8_t A = __builtin_bit_cast(pbf16x8_t, vr);
#pragma unroll
      for (int a = 0; a < 2; ++a)
        acc[rb][cb][a][q] =
            __builtin_amdgcn_mfma_f32_16x16x32_bf16(A, __builtin_bit_cast(pbf16x8_t, o.w[cb][a]), acc[rb][cb][a][q], 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  // The loads that may be outstanding when chunk k is needed, before chunk k + RING - 2 is
  // asked for: those of the chunks after it -- of the prologue's chunks their activations
  // only, since all its weights come first.
  constexpr int kSteady = LOADS * (RING - 3);
  static_assert(LOADS * (RING - 1) < 64, "the counter of outstanding loads");
  // step c, in ring slot SLOT: chunk c + 1 has landed (and chunk c's operands are in registers),
  // so the slot of chunk c - 1 is free and takes chunk c + RING - 1 (past the end: zeros,
  // read by nobody).  A wave issues in order and an MFMA keeps its unit for 16 cycles: the other
  // work goes between them.
  auto step = [&](int c, auto slot_tag, const Ops& now, Ops& next) __attribute__((always_inline)) {
    constexpr int slot = decltype(slot_tag)::value;
    constexpr int to = (slot + RING - 1) % RING;
    const unsigned char* st = smem + (slot + 1) % RING * CHUNK;
    if (slot + 1 < RING - 2 && c < RING) small_wait<RB * (slot + 1 < RING - 2 ? RING - 3 - slot : 0) + LOADS * (slot < RING - 3 ? slot : 0)>();
    else small_wait<kSteady>();
    read_x(st, next);
    mma(now, 0, 0);
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) read_w(st, next, cb);
    mma(now, 0, 1);
#pragma unroll
    for (int u = 0; u < 2; ++u) issue_w(c + RING - 1, to, u);
    if constexpr (CB == 2) {
      mma(now, 1, 0);
#pragma unroll
      for (int u = 2; u < 4; ++u) issue_w(c + RING - 1, to, u);
      mma(now, 1, 1);
    }
    issue_a(c + RING - 1, to);
  };
  small_wait<RB * (RING - 2)>();  // chunk 0, and with it the bias
  Ops o0, o1;
  read_x(smem, o0);
  float bvs[CB][8];
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) {
    read_w(smem, o0, cb);
    const unsigned char* bp = s_bias + (cb * 16 + l16) * 32;
    const uint4 lo = *reinterpret_cast<const uint4*>(bp), hi = *reinterpret_cast<const uint4*>(bp + 16);
    const uint32_t mk[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};  // mask order
#pragma unroll
    for (int c = 0; c < 8; ++c) bvs[cb][c] = __builtin_bit_cast(float, mk[blade_to_mask(c)]);
    float b[2][2][2] = {};
    if constexpr (BIAS_FIRST) pauli_bias_entries(bvs[cb], b);
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int q = 0; q < 2; ++q) acc[rb][cb][a][q] = pf32x4_t{b[a][q][0], b[a][q][1], b[a][q][0], b[a][q][1]};
  }
#pragma unroll 1
  for (int c = 0;; c += RING) {  // (n is even)
    static_assert(RING == 6 || RING == 8, "the steps of one round of the ring");
#define YGG_TWO(S)                                        \
  step(c + S, std::integral_constant<int, S>{}, o0, o1);         \
  step(c + S + 1, std::integral_constant<int, S + 1>{}, o1, o0); \
  if (c + S + 2 >= n) break
    YGG_TWO(0);
    YGG_TWO(2);
    YGG_TWO(4);
    if constexpr (RING == 8) {
      YGG_TWO(6);
    }
#undef YGG_TWO
  }
  small_wait<0>();  // nothing may land in LDS after the wave has ended

  const uint64_t y_bytes = (uint64_t)P_max * d_out * 16, first = (uint64_t)row0 * d_out * 16;
  const __amdgpu_buffer_rsrc_t y_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      static_cast<char*>(Y) + first, (short)0, (uint32_t)(y_bytes - first), kBufferFlags);
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) {
    const int j = col0 + cb * 16 + l16;
    if (j >= d_out) continue;
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int rl = rb * 8 + 2 * g + h;  // row of the tile; its halves b = 0, 1 are sums 2 h, 2 h + 1
        if (row0 + rl >= row_end) continue;
        const auto& s = acc[rb][cb];
        const uint32_t off = OUT == kOutPauliRows ? ((uint32_t)rl * 2 * d_out + j) * 8 : ((uint32_t)rl * d_out + j) * 16;
        pauli_store_mv<ACT, OUT, kBF16, BIAS_FIRST>(s[0][0][2 * h], s[0][1][2 * h], s[0][0][2 * h + 1], s[0][1][2 * h + 1],
                                                    s[1][0][2 * h], s[1][1][2 * h], s[1][0][2 * h + 1], s[1][1][2 * h + 1],
                                                    bvs[cb], y_rsrc, off, 0, d_out);
      }
  }
}

// at most this many tiles of `tok` rows
long long small_row_tiles(int P, int E, int tok) { return std::min<long long>(P, (P + tok - 1) / tok + E); }

template <int ACT, int OUT>
int launch_small(const void* x, int x_rows, const int32_t* gather, int P, const void* w, const float* bias,
                 const int32_t* offsets, int E, int d_in, int d_out, void* y, hipStream_t st) {
  const uint16_t* X = static_cast<const uint16_t*>(x);
  const uint16_t* W = static_cast<const uint16_t*>(w);
  const uint32_t xb = (uint32_t)((size_t)x_rows * d_in * 16);
  const bool bias_first = pauli_uses_dma(kInPauliRows, d_in);  // (the register-staged 64 x 64 tiles add it at the end)
#define YGG_PSL(RB, CB, RING)                                                                                          \
  do {                                                                                                                  \
    const unsigned grid = (unsigned)(small_row_tiles(P, E, 8 * RB) * ((d_out + 16 * CB - 1) / (16 * CB)));              \
    if (bias_first)                                                                                                     \
      pauli_small_kernel<ACT, OUT, true, RB, CB, RING><<<grid, 64, 0, st>>>(X, xb, gather, W, bias, offsets, E, d_in,  \
                                                                            d_out, P, y);                               \
    else                                                                                                                \
      pauli_small_kernel<ACT, OUT, false, RB, CB, RING><<<grid, 64, 0, st>>>(X, xb, gather, W, bias, offsets, E, d_in, \
                                                                             d_out, P, y);                              \
  } while (0)
  // 8 tokens x 16 columns a wave, six waves a CU, while the products are small: a wave's step is
  // four MFMAs.  Above, every row tile reads its expert's weights once more, and 16 x 32 a wave
  // are faster (layer calls, 8 x 16 / 16 x 32, us: d = 128, F = 512, E = 32: 2 rows 21 / 34, 512 39 / 46, 1024
  // 51 / 53, 2048 75 / 65; d = 256, F = 1024, E = 64: 32 52 / 69, 512 142 / 149, 1024 185 / 173; d = 200,
  // F = 800, E = 4: 128 34 / 51, 512 60 / 61, 1024 91 / 76; d = 64, F = 512, E = 64: 1024 48 / 50, 2048 64 / 59)
  if (P <= 1024 && (double)P * d_in * d_out <= 8e7) YGG_PSL(1, 1, 8);
  else YGG_PSL(2, 2, 6);
#undef YGG_PSL
  return check_launch("pauli_small");
}

}  // namespace

// From these sizes on the 64 x 64 tiles are faster (layer calls, few rows / tiles, us: d = 128,
// F = 512, E = 32: 2 rows 21 / 53, 512 39 / 64, 2048 65 / 74, 3072 80 / 81, 4096 105 / 89; d = 128, F = 1024,
// E = 16: 1 27 / 78, 1536 87 / 99; d = 256, F = 1024, E = 64: 2 31 / 92, 128 109 / 147, 512 142 / 169, 1024
// 173 / 178, 2048 249 / 202; d = 256, F = 512, E = 8: 1536 70 / 76, 2048 101 / 85; d = 200, F = 800, E = 4: 1024
// 76 / 86, 1536 92 / 92; d = 100, F = 302, E = 12: 1536 41 / 54, 3072 57 / 56; d = 64, F = 512, E = 64: 2048
// 59 / 73, 4096 82 / 81).
bool pauli_small_pays(long long N, long long P, int E, int d, int F) {
  if (P < 1 || P > 2048 || (double)P * d * F > 2e8) return false;
  const uint64_t lim = (uint64_t)1 << 31;  // the kernel's 32-bit offsets
  return (uint64_t)(std::max(d, F) + 64) * std::min(d, F) * 16 < lim && (uint64_t)P * std::max(d, F) * 16 < lim &&
         (uint64_t)N * d * 16 < lim && (uint64_t)E * std::max(d, F) * 32 < lim;
}

int pauli_small_up(const void* x, int x_rows, const int32_t* gather, int P, const void* w, const float* bias,
                   const int32_t* offsets, int E, int d_in, int d_out, int act, void* h, hipStream_t stream) {
#define YGG_PS(A) return launch_small<A, kOutPauliRows>(x, x_rows, gather, P, w, bias, offsets, E, d_in, d_out, h, stream)
  switch (act) {
    case kActNone: YGG_PS(kActNone);
    case kActGelu: YGG_PS(kActGelu);
    case kActRelu: YGG_PS(kActRelu);
    default: YGG_PS(kActSigmoid);
  }
#undef YGG_PS
}

int pauli_small_down(const void* h, int P, const void* w, const float* bias, const int32_t* offsets, int E, int d_in,
                     int d_out, void* y, hipStream_t stream) {
  return launch_small<kActNone, kOutBlade>(h, P, nullptr, P, w, bias, offsets, E, d_in, d_out, y, stream);
}

}  // namespace ygg
