// dsa_indexer_device.h -- device helpers shared by the indexer's kernels
// (dsa_indexer.hip, dsa_select.hip): e4m3fn codes, their 7-bit pieces, the
// lane-group sum and the candidate count.
#pragma once

#include "dsa_internal.h"

namespace dsa {
namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

constexpr int kIdxDim = 128;
constexpr int kKTokenBytes = kIdxDim + 4;  // paged K cache: codes + fp32 scale per token
constexpr int kChunk = 1024;              // one MFMA operand: 64 lanes x 16 bytes
constexpr int kBlockBytes = 3 * 2 * kChunk;  // k block: planes p0 and p1 (2 k-steps each), codes
constexpr int kCodeBlockBytes = 2 * kChunk;  // a block of codes alone
static_assert(kBlockBytes == kKPlaneBlockBytes && kKPlaneCodeOffset == 4 * kChunk, "k block layout");
constexpr int kTwoPieceLimit = 1 << 14;
constexpr int kBufferFlags = 0x00020000;  // raw buffer descriptor: 32-bit data format

// e4m3fn code -> x = value * 2^9 (integer), NaN codes -> 0.
__device__ __forceinline__ int e4m3_x(uint32_t c) {
  const int e = (c >> 3) & 15, m = c & 7;
  int x = (e == 0) ? m : ((8 + m) << (e - 1));
  if (e == 15 && m == 7) x = 0;
  return (c & 0x80) ? -x : x;
}

// Signed 7-bit piece `pc` of x (sign-magnitude split), as a byte.  The
// pieces of one value share its sign, so for |x| < 2^14 the difference
// p0 - p1 of its two pieces lies in [-127, 127] as well.
__device__ __forceinline__ uint32_t piece_byte(int x, int pc) {
  const int mag = x < 0 ? -x : x;
  const int v = (mag >> (7 * pc)) & 127;
  return (uint32_t)(x < 0 ? -v : v) & 0xffu;
}

__device__ __forceinline__ i32x4 load_chunk(const int8_t *p) { return *(const i32x4 *)p; }

__device__ __forceinline__ i32x4 mfma(i32x4 a, i32x4 b, i32x4 c) {
  return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
}

// ---- operand preparation -------------------------------------------------

// The top bit of each byte: set iff the byte is a NaN code (0x7f, 0xff; the low
// seven bits are all ones iff adding one carries).  The other bits are junk.
__device__ __forceinline__ uint32_t nan_bits(uint32_t w) { return (w & 0x7f7f7f7fu) + 0x01010101u; }

// Four codes with the NaN codes replaced by 0.
__device__ __forceinline__ uint32_t drop_nan(uint32_t w) {
  return w & ~(((nan_bits(w) & 0x80808080u) >> 7) * 255u);
}

// Sum of the squares of the eight e4m3fn values in w0, w1 (no NaN codes).
__device__ __forceinline__ float sum_squares8(uint32_t w0, uint32_t w1) {
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const uint32_t w = i == 0 ? w0 : w1;
    const auto a = __builtin_amdgcn_cvt_pk_f32_fp8((int)w, false);
    const auto b = __builtin_amdgcn_cvt_pk_f32_fp8((int)w, true);
    s = __builtin_fmaf(a[0], a[0], s);
    s = __builtin_fmaf(a[1], a[1], s);
    s = __builtin_fmaf(b[0], b[0], s);
    s = __builtin_fmaf(b[1], b[1], s);
  }
  return s;
}

// k_max words: the block's largest |x| in the low 18 bits, and in the upper 14
// the largest |c_s| * |k_s| (2-norm) of its positions as the top bits of a
// positive fp32, rounded up (0x3fff: NaN).
constexpr int kMaxXBits = 18;
__device__ __forceinline__ int block_max_x(int word) { return word & ((1 << kMaxXBits) - 1); }
__device__ __forceinline__ uint32_t norm_bits_up(uint32_t bits) {  // of a non-negative fp32
  return min((bits + 0x1ffffu) >> 17, 0x3fffu);
}
// |c_s| |k_s| of a position whose codes' squares sum to n2 (the factor covers
// the sum's and the root's rounding; 0 only if either is).
__device__ __forceinline__ uint32_t position_norm_bits(float cs, float n2) {
  const uint32_t tiny = cs != 0.f && n2 > 0.f ? 1u : 0u;
  return norm_bits_up(max(__float_as_uint(fabsf(cs) * sqrtf(n2) * 1.001f), tiny));
}
__device__ __forceinline__ float norm_from_bits(uint32_t b14) { return __uint_as_float(b14 << 17); }

// e4m3fn code -> its signed 7-bit pieces as bytes: p0 | p1 << 8 | p2 << 16 |
// (p0 - p1) << 24 (the kernels keep this table in LDS).
__device__ __forceinline__ uint32_t piece_word(uint32_t code) {
  const int x = e4m3_x(code);
  const uint32_t b0 = piece_byte(x, 0), b1 = piece_byte(x, 1);
  const uint32_t d = (uint32_t)((int)(int8_t)b0 - (int)(int8_t)b1) & 0xffu;
  return b0 | (b1 << 8) | (piece_byte(x, 2) << 16) | (d << 24);
}

// Largest |x| (x = value * 2^9) of a set of codes from its largest code &
// 0x7f (e4m3 magnitudes order like their codes; the NaN code 0x7f ranks above
// 448, which only makes a bound conservative).
__device__ __forceinline__ int magnitude_bound(uint32_t top) {
  return top == 0x7f ? (15 << 14) : e4m3_x(top);
}

// Lane 63 gets the wave's largest value.
__device__ __forceinline__ uint32_t wave_max_last(uint32_t v) {
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false));
  return max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false));
}

// Wave-wide largest code & 0x7f of the 32 codes a lane holds in w[8]: two bytes of
// a dword at a time.
__device__ __forceinline__ uint32_t wave_top_code(const uint32_t (&w)[8]) {
  typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
  u16x2 m = {0, 0};
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    m = __builtin_elementwise_max(m, __builtin_bit_cast(u16x2, w[i] & 0x007f007fu));
    m = __builtin_elementwise_max(m, __builtin_bit_cast(u16x2, (w[i] >> 8) & 0x007f007fu));
  }
  return __builtin_amdgcn_readlane(wave_max_last(max((uint32_t)m[0], (uint32_t)m[1])), 63);
}

// Plane `byte` of the LUT words v[32] of a lane's 2 x 16 codes (negated: the
// plane's bytes negated), as the two k-steps' 16-byte operand pieces.
__device__ __forceinline__ void pack_plane(const uint32_t (&v)[32], int byte, bool negate,
                                           i32x4 (&out)[2]) {
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      uint32_t packed = 0;
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        uint32_t x = (v[16 * ks + 4 * d + b] >> (8 * byte)) & 0xffu;
        if (negate) x = (0u - x) & 0xffu;
        packed |= x << (8 * b);
      }
      out[ks][d] = (int)packed;
    }
  }
}

// fl32(max(D, 0)) of D = lo + 2^14 hi (exact in fp64): rounding keeps the sign.
__device__ __forceinline__ float relu_dot(int lo, int hi) {
  const float r = (float)__builtin_fma(16384.0, (double)hi, (double)lo);
  return r > 0.f ? r : 0.f;
}

// The third pieces of the lane's 2 x 16 codes at src (dims +0 and +64), as the
// two k-steps' operands.
__device__ __forceinline__ void third_pieces(const uint32_t *lut, const uint8_t *src, i32x4 (&out)[2]) {
  const uint4 r0 = *(const uint4 *)src, r1 = *(const uint4 *)(src + 64);
  const uint32_t w[8] = {r0.x, r0.y, r0.z, r0.w, r1.x, r1.y, r1.z, r1.w};
  uint32_t v[32];
#pragma unroll
  for (int i = 0; i < 32; ++i) v[i] = lut[(w[i >> 2] >> (8 * (i & 3))) & 0xffu];
  pack_plane(v, 2, false, out);
}

// (G0 + G1) + (G2 + G3) over the four 16-lane rows; every lane gets the sum.
// permlane16_swap exchanges rows 0<->1 and 2<->3, permlane32_swap the two
// halves; fp32 addition is commutative, so both lanes of a pair agree.
__device__ __forceinline__ float sum_lane_groups(float v) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  const float s = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(s), __float_as_uint(s), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// Number of candidate positions of row t: s is one iff s <= causal_limit[t]
// and s < S.  Compared before adding one, so a limit of INT32_MAX (no limit)
// does not wrap to a negative count.
__device__ __forceinline__ int candidates(const IndexerParams &p, int t) {
  const int lim = p.limit[t];
  return lim >= p.S - 1 ? p.S : max(0, lim + 1);
}

}  // namespace
}  // namespace dsa
