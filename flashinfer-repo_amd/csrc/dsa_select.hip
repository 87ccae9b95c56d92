// dsa_select.hip -- the indexer's selection: score estimates, exact scores of
// the positions they leave open, and the per-row top-k, for gfx950.
//
// Kernels:
//   dsa_idx_estimate_kernel     every score within a bound, by bf16 MFMAs
//   dsa_idx_topk_kernel         from exact scores, up to 32768 positions: one
//                               workgroup per row, the row in registers
//                               (loaded coalesced, 1024-strided, through one
//                               buffer descriptor): two radix passes (8 bits
//                               each, histograms replicated 32 ways so equal
//                               digits do not collide in one LDS bank) find
//                               the 16-bit bin of the k-th largest order key;
//                               keys above it are taken and the few in (or,
//                               with estimates, near) it are ranked by exact
//                               score, then lower position (reference intent:
//                               indexer_kernel.py:289-343, strict '>' keeps
//                               the earlier index); many equal keys take two
//                               more passes.  The selection is a position
//                               bitmap built from ballots; one scan turns it
//                               into ranks in ascending position order.
//   dsa_idx_topk_estimates_kernel  the same from estimates
//   dsa_idx_topk_chunk_kernel,
//   dsa_idx_topk_merge_kernel   rows longer than 32768 positions, from
//                               estimates: a list per chunk, then the lists
//   dsa_idx_topk_stream_kernel  a four-pass selection re-reading the row from
//                               memory: longer rows from exact scores
#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "../../include/dsa_abi.h"
#include "dsa_indexer_device.h"

namespace dsa {
namespace {

constexpr int kTopkThreads = 1024;
constexpr int kMaxRegEpt = 32;            // register top-k up to 1024 * 32 positions
constexpr int kHistCopies = 32;
constexpr int kHistPitch = 257;           // copy c of bin j at c*257 + j: bank (c + j) % 64

// ---- score estimates ------------------------------------------------------
//
// A selection needs the exact score only of positions near the k-th largest
// one.  The estimate of every score is the same sum with the dots taken by
// bf16 MFMAs (e4m3 values and their products are exact in bf16 / fp32) and
// summed in fp32: s~ = fl(sum_h w_h max(d~_h, 0)) * k_scale.  Its distance from
// the exact score is at most
//   E = kEstimateError * (sum_h |w_h| |q_h|) * max_s |k_scale_s| |k_s|   (2-norms):
// The MFMA's fp32 sums are not documented; measured with directed codes (one
// large product beside 127 whose sum of eight falls just short of its last
// bit), it truncates each group of eight products and the sum so far to 24
// bits: 16 groups a dot, so 16 x 2^-23 = 2^-19 of |q_h| |k_s| (2^-19.27 was
// reached; random codes stay below 2^-22).  The bound does not lean on the
// groups: it lets every one of the 128 products lose 2^-24 by itself, 2^-17.
// The head sum's 19 roundings, and the 20 of the exact definition, add
// 39 x 2^-24 of sum_h |w_h| max(d_h, 0), the roundings of the selection's
// limits 2 x 2^-24: 169 x 2^-24 = 1.32 x 2^-17 together.  (The fp8 MFMAs, twice as fast,
// drop product bits below 2^-13 of a group's largest: 2^-13.5 was seen.)
constexpr float kEstimateError = 0x1.54p-17f;

constexpr int kEstWaves = 4;
constexpr int kEstWavesPerCU = 8;  // two per SIMD
constexpr int kEstFusedTokens = 8; // up to so many tokens an estimate prepares K itself

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// Eight e4m3fn codes (no NaN codes) as bf16, exactly.
__device__ __forceinline__ bf16x8 to_bf16x8(uint32_t w0, uint32_t w1) {
  const bf16x2 a = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w0, 1.0f, false);
  const bf16x2 b = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w0, 1.0f, true);
  const bf16x2 c = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w1, 1.0f, false);
  const bf16x2 d = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w1, 1.0f, true);
  return bf16x8{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}

// Where the estimate kernel takes K from.
enum KSource {
  kPrepared,  // codes, c_s and k_max are there (dsa_idx_prep_kernel)
  kFlat,      // the caller's flat codes and scales: c_s and k_max are written here
  kPaged,     // the caller's paged cache: codes, c_s and k_max are written here
};

// Estimates of two tokens' scores.  A wave holds both tokens' q as bf16 MFMA A
// operands (heads as M, the row order of q_operands) and walks pairs of
// 16-position blocks: a block's codes are one 16-byte load per lane and half
// (row by row: the wave reads the block's 2 KB), converted once for both
// tokens.  Bound: the 16 MFMAs (Hi = 64) of a block and token, 256 cycles of
// the SIMD's matrix pipe at the ~1.9 GHz the chip holds under them; beside them
// run 44 VALU instructions (the head sum of one (block, token) beside the
// MFMAs of the next).  64 rows of 32768 positions take 30 us (the three-product
// int8 kernel of the exact scores 47), 1024 rows of 16384 with codes up to 448
// take 200 us (the nine-product one 990).  Two tokens per wave halve the conversions and loads;
// four would need more than the 256 registers that two waves per SIMD leave
// each.  After two blocks the four lane groups' sums of the four (block,
// token) pairs are added by two permlane16 and one permlane32 swap, so lane
// group g holds, and stores, token g & 1 of block g >> 1.
//
// Of the two waves on a SIMD one is served first and would finish long before
// the other, which then waits for memory alone (1024 rows of 16384 positions:
// 107 and 201 us): a wave lowers its priority as it gets on, so the one behind
// catches up (145 and 192).
template <int NHB, int SRC>
__global__ __launch_bounds__(kEstWaves * 64, SRC == kPrepared ? 2 : 1) void dsa_idx_estimate_kernel(IndexerParams p) {
  __shared__ __attribute__((aligned(16))) float wsm[kEstWaves][2][64];
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // est_pairs (1, 2 or 4) waves of the workgroup take different token pairs
  // over the same positions, the others other positions
  const int tw = wave & (p.est_pairs - 1), rw = wave / p.est_pairs;
  const int t0 = (blockIdx.y * p.est_pairs + tw) * 2;
  if (t0 >= p.T) return;
  const int t1 = min(t0 + 1, p.T - 1);
  // rows with at most topk candidates take them all: nothing to estimate
  int n0 = candidates(p, t0), n1 = t0 + 1 < p.T ? candidates(p, t1) : 0;
  if (n0 <= p.topk) n0 = 0;
  if (n1 <= p.topk) n1 = 0;
  const int nkb = (max(n0, n1) + 15) >> 4;
  const int b0 = (blockIdx.x * (kEstWaves / p.est_pairs) + rw) * p.est_blocks;  // (even)
  const int b1 = min(nkb, b0 + p.est_blocks);
  if (b0 >= b1) return;

  uint4 qr[2][NHB][2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int t = u == 0 ? t0 : t1;
#pragma unroll
    for (int hb = 0; hb < NHB; ++hb) {
      const int head = (c >> 2) * (NHB * 4) + 4 * hb + (c & 3);
      const uint8_t *row = p.q + ((int64_t)t * (NHB * 16) + head) * kIdxDim + g * 16;
#pragma unroll
      for (int j = 0; j < 2; ++j) qr[u][hb][j] = *(const uint4 *)(row + 64 * j);
    }
    // this wave's own copy of the token's weights (read back by this wave only)
    wsm[wave][u][lane] = lane < NHB * 16 ? p.w[(int64_t)t * (NHB * 16) + lane] : 0.f;
  }
  const float *wl = &wsm[wave][0][g * (NHB * 4)];  // + u*64 + 4*hb: the lane's heads

  const int s_blocks = (p.S + 15) >> 4;
  const auto krs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t *>(SRC == kFlat ? p.k : p.k_codes), 0,
      SRC == kFlat ? p.S * kIdxDim : s_blocks * p.k_code_stride, kBufferFlags);
  const auto srs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float *>(SRC == kFlat ? p.k_scale : p.k_cs), 0, p.S * 4, kBufferFlags);
  const auto ors = __builtin_amdgcn_make_buffer_rsrc(p.scores + (int64_t)t0 * p.S, 0,
                                                     (t1 - t0 + 1) * p.S * 4, kBufferFlags);
  constexpr uint32_t kDropped = 0x80000000u;
  const int kvo = c * kIdxDim + g * 16;
  struct Raw {
    u32x4 h[2];
    float cs;  // kPaged: the position's scale
  };
  // kPaged: the page of the lane's position of block blk, loaded a step before
  // its codes (a position past S, or an unmapped page, reads as zeros)
  auto page_of = [&](int blk) {
    const int s = min(blk, b1 - 1) * 16 + c;
    return SRC == kPaged && s < p.S ? p.k_pages[s / p.k_page_size] : -1;
  };
  auto fetch = [&](int blk, int pg, Raw &r) {
    blk = min(blk, b1 - 1);
    if constexpr (SRC == kPaged) {
      r.h[0] = r.h[1] = u32x4{0u, 0u, 0u, 0u};
      r.cs = 0.f;
      if ((uint32_t)pg < (uint32_t)p.k_num_pages) {
        const int off = (blk * 16 + c) % p.k_page_size;
        const uint8_t *page = p.k_cache + (int64_t)pg * p.k_page_size * kKTokenBytes;
        r.h[0] = *(const u32x4 *)(page + off * kIdxDim + g * 16);
        r.h[1] = *(const u32x4 *)(page + off * kIdxDim + 64 + g * 16);
        r.cs = *(const float *)(page + p.k_page_size * kIdxDim + off * 4) * 0x1p-18f;
      }
    } else {
      const int stride = SRC == kFlat ? kCodeBlockBytes : p.k_code_stride;
#pragma unroll
      for (int j = 0; j < 2; ++j)
        r.h[j] = __builtin_bit_cast(
            u32x4, __builtin_amdgcn_raw_buffer_load_b128(krs, kvo + 64 * j, blk * stride, 0));
    }
  };
  // 2^18 c_s of the lane's position of the pair starting at blk: block g >> 1
  auto fetch_cs = [&](int blk) {
    const float v = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(srs, ((g >> 1) * 16 + c) * 4, blk * 64, 0));
    // (c_s, which the exact score and the bound take, is rounded where it is subnormal)
    return (SRC == kFlat ? v * 0x1p-18f : v) * 0x1p18f;
  };
  // What dsa_idx_prep_kernel writes, of block blk (of the caller's K)
  auto prepare = [&](int blk, Raw &r) {
    if constexpr (SRC != kPrepared) {
      if (blk >= b1) return;
      uint32_t nan = 0;
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int d = 0; d < 4; ++d) nan |= nan_bits(r.h[j][d]);
      if (__ballot(nan & 0x80808080u) != 0) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int d = 0; d < 4; ++d) r.h[j][d] = drop_nan(r.h[j][d]);
      }
      float n2 = 0.f;
#pragma unroll
      for (int j = 0; j < 2; ++j)
        n2 += sum_squares8(r.h[j][0], r.h[j][1]) + sum_squares8(r.h[j][2], r.h[j][3]);
      n2 = sum_lane_groups(n2);
      const int s = blk * 16 + c;
      float cs = r.cs;
      if constexpr (SRC == kFlat) cs = s < p.S ? p.k_scale[s] * 0x1p-18f : 0.f;
      const uint32_t nb = wave_max_last(position_norm_bits(cs, n2));
      if (lane == 63) p.k_max[blk] = (int32_t)(nb << kMaxXBits);
      if (g == 0 && s < p.S) p.k_cs[s] = cs;
      if constexpr (SRC == kPaged) {
        uint8_t *dst = p.k_codes + (int64_t)blk * kCodeBlockBytes + kvo;
#pragma unroll
        for (int j = 0; j < 2; ++j) *(u32x4 *)(dst + 64 * j) = r.h[j];
      }
    }
  };
  auto convert = [&](const Raw &r, bf16x8 (&k)[4]) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      k[2 * j] = to_bf16x8(r.h[j][0], r.h[j][1]);
      k[2 * j + 1] = to_bf16x8(r.h[j][2], r.h[j][3]);
    }
  };

  Raw r0, r1;
  int pg0 = page_of(b0), pg1 = page_of(b0 + 1);
  fetch(b0, pg0, r0);
  fetch(b0 + 1, pg1, r1);
  pg0 = page_of(b0 + 2);
  pg1 = page_of(b0 + 3);

  // NaN codes count as zeros; looked for first (2.5 instructions per dword
  // against 6 to drop them)
  uint32_t nan = 0;
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int hb = 0; hb < NHB; ++hb)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const uint4 r = qr[u][hb][j];
        nan |= nan_bits(r.x) | nan_bits(r.y);
        nan |= nan_bits(r.z) | nan_bits(r.w);
      }
  if (__ballot(nan & 0x80808080u) != 0) {
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int hb = 0; hb < NHB; ++hb)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          uint4 &r = qr[u][hb][j];
          r = make_uint4(drop_nan(r.x), drop_nan(r.y), drop_nan(r.z), drop_nan(r.w));
        }
  }
  bf16x8 q[2][NHB][4];
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int hb = 0; hb < NHB; ++hb)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const uint4 r = qr[u][hb][j];
        q[u][hb][2 * j] = to_bf16x8(r.x, r.y);
        q[u][hb][2 * j + 1] = to_bf16x8(r.z, r.w);
      }

  auto dots = [&](int u, const bf16x8 (&k)[4], f32x4 (&acc)[NHB]) {
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int hb = 0; hb < NHB; ++hb)
        acc[hb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            q[u][hb][s], k[s], s == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[hb], 0, 0, 0);
  };
  auto head_sum = [&](int u, const f32x4 (&acc)[NHB]) {
    float G = 0.f;
#pragma unroll
    for (int hb = 0; hb < NHB; ++hb) {
      const f32x4 w = *(const f32x4 *)(wl + u * 64 + 4 * hb);
#pragma unroll
      for (int i = 0; i < 4; ++i)  // (the integer max of the bits is max(., 0) in one instruction)
        G = __builtin_fmaf(w[i], __int_as_float(max(__float_as_int(acc[hb][i]), 0)), G);
    }
    return G;
  };
  const int n_lane = (g & 1) ? n1 : n0;
  const uint32_t row_off = (uint32_t)((g & 1) * p.S) * 4;
  float G[4];  // lane-group sums of (block, token): b t0, b t1, b+1 t0, b+1 t1
  auto store_pair = [&](int blk0, float cs) {
    const auto x = __builtin_amdgcn_permlane16_swap(__float_as_uint(G[0]), __float_as_uint(G[1]), false, false);
    const float a0 = __uint_as_float(x[0]) + __uint_as_float(x[1]);
    const auto y = __builtin_amdgcn_permlane16_swap(__float_as_uint(G[2]), __float_as_uint(G[3]), false, false);
    const float a1 = __uint_as_float(y[0]) + __uint_as_float(y[1]);
    const auto z = __builtin_amdgcn_permlane32_swap(__float_as_uint(a0), __float_as_uint(a1), false, false);
    const float v = (__uint_as_float(z[0]) + __uint_as_float(z[1])) * cs;
    const int blk = blk0 + (g >> 1), s = blk * 16 + c;
    const uint32_t off = s < n_lane && blk >= b0 && blk < b1 ? row_off + (uint32_t)s * 4 : kDropped;
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), ors, off, 0, 0);
  };

  bf16x8 k0[4], k1[4];
  f32x4 A[NHB], B[NHB];
#pragma unroll
  for (int hb = 0; hb < NHB; ++hb) B[hb] = f32x4{0.f, 0.f, 0.f, 0.f};
  G[0] = G[1] = G[2] = 0.f;
  // the pair's scale of the lane's position; kPaged: it came with the codes
  float cs = SRC == kPaged ? 0.f : fetch_cs(b0), cs_prev = 0.f, c0 = r0.cs;
  prepare(b0, r0);
  convert(r0, k0);
  fetch(b0 + 2, pg0, r0);
  pg0 = page_of(b0 + 4);
  // the order of a step: weights from LDS, then the MFMAs with NV VALU
  // instructions behind each
  auto spread = [&](auto nv) {
    if constexpr (SRC == kPrepared) {
      __builtin_amdgcn_sched_group_barrier(0x100, NHB, 0);
#pragma unroll
      for (int i = 0; i < 4 * NHB; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, decltype(nv)::value, 0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  using N2 = std::integral_constant<int, 2>;
  using N3 = std::integral_constant<int, 3>;
  const int len = b1 - b0;
  for (int b = b0; b < b1; b += 2) {
    // the (block, token) sums lag the MFMAs by one; the pair's fourth sum and
    // store come in the next iteration (or after the loop).  A block's codes
    // are converted one step before its first MFMAs, and the registers take
    // the block two ahead at once.
    const int left = b1 - b;
    if (2 * left > len) __builtin_amdgcn_s_setprio(3);
    else if (4 * left > len) __builtin_amdgcn_s_setprio(2);
    else if (8 * left > len) __builtin_amdgcn_s_setprio(1);
    else __builtin_amdgcn_s_setprio(0);
    dots(0, k0, A);
    G[3] = head_sum(1, B);
    store_pair(b - 2, cs_prev);
    spread(N3{});
    dots(1, k0, B);
    G[0] = head_sum(0, A);
    const float c1 = r1.cs;
    prepare(b + 1, r1);
    convert(r1, k1);
    spread(N3{});
    if constexpr (SRC == kPaged) {
      cs_prev = ((g >> 1) ? c1 : c0) * 0x1p18f;
    } else {
      cs_prev = cs;
      cs = fetch_cs(b + 2);
    }
    fetch(b + 3, pg1, r1);
    pg1 = page_of(b + 5);
    dots(0, k1, A);
    G[1] = head_sum(1, B);
    spread(N2{});
    dots(1, k1, B);
    G[2] = head_sum(0, A);
    c0 = r0.cs;
    prepare(b + 2, r0);
    convert(r0, k0);
    spread(N3{});
    fetch(b + 4, pg0, r0);
    pg0 = page_of(b + 6);
  }
  G[3] = head_sum(1, B);
  store_pair(b0 + ((b1 - 1 - b0) & ~1), cs_prev);
}

// ---- top-k ---------------------------------------------------------------

__device__ __forceinline__ uint32_t order_key(float f) {
  uint32_t u = __builtin_bit_cast(uint32_t, f == 0.f ? 0.f : f);  // -0 -> +0
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

__device__ __forceinline__ float key_value(uint32_t key) {
  return __uint_as_float((key & 0x80000000u) ? key ^ 0x80000000u : ~key);
}

__device__ __forceinline__ void emit_pos(const IndexerParams &p, int t, int32_t *out, int pos,
                                         int rank) {
  int v = pos;
  if (p.block_table != nullptr) {
    const int32_t page = p.block_table[(int64_t)t * p.bt_stride + pos / p.page_size];
    v = page * p.page_size + pos % p.page_size;
  }
  out[rank] = v;
}

// Inclusive prefix sum over the 64 lanes of a wave: row shifts within rows
// of 16 lanes, then the row totals carried with the row broadcasts (gfx9
// wave64 DPP; lanes without a source add 0).
__device__ __forceinline__ int wave_inclusive_sum(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);  // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);  // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);  // row_shr:8
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15 -> rows 1, 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31 -> rows 2, 3
  return v;
}

// Lane 15 of each row of 16 gets the row's sum.
__device__ __forceinline__ float row_sum_last(float v) {
  auto add = [](float x, int y) { return x + __int_as_float(y); };
  v = add(v, __builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x111, 0xf, 0xf, false));  // row_shr:1
  v = add(v, __builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x112, 0xf, 0xf, false));  // row_shr:2
  v = add(v, __builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x114, 0xf, 0xf, false));  // row_shr:4
  return add(v, __builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x118, 0xf, 0xf, false));  // row_shr:8
}

// Lane 63 gets the sum of lanes 15, 31, 47 and 63.
__device__ __forceinline__ float rows_sum_last(float v) {
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x142, 0xa, 0xf, false));
  return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x143, 0xc, 0xf, false));
}

// Exclusive prefix sums of (a, b) over the 1024 threads of the block; the
// totals go to *ta, *tb.  Wave sums, then wave 0 scans the 16 wave totals.
__device__ int2 block_exclusive_scan2(int a, int b, int2 *scratch, int *ta, int *tb) {
  constexpr int kWaves = kTopkThreads / 64;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int x = wave_inclusive_sum(a), y = wave_inclusive_sum(b);
  if (lane == 63) scratch[wave] = make_int2(x, y);
  __syncthreads();
  if (wave == 0) {
    const int2 w = lane < kWaves ? scratch[lane] : make_int2(0, 0);
    const int ix = wave_inclusive_sum(w.x), iy = wave_inclusive_sum(w.y);
    if (lane < kWaves) scratch[lane] = make_int2(ix - w.x, iy - w.y);
    if (lane == kWaves - 1) scratch[kWaves] = make_int2(ix, iy);
  }
  __syncthreads();
  const int2 base = scratch[wave];
  *ta = scratch[kWaves].x;
  *tb = scratch[kWaves].y;
  __syncthreads();
  return make_int2(base.x + x - a, base.y + y - b);
}

// After one pass's histogram is in tot[]: the digit that holds the
// `need`-th largest key among those matching the prefix.  Run by wave 0.
__device__ __forceinline__ void pick_digit(const uint32_t *tot, uint32_t prefix, uint32_t mask,
                                           int shift, int need, uint32_t *s_prefix,
                                           uint32_t *s_mask, int *s_need) {
  // Lane l owns bins b0 .. b0+3 with b0 = 4*(63 - l), so the bins above
  // its own belong to lanes 0..l-1: their count is an exclusive prefix sum.
  const int l = threadIdx.x;
  const int b0 = 4 * (63 - l);
  const uint32_t c0 = tot[b0], c1 = tot[b0 + 1], c2 = tot[b0 + 2], c3 = tot[b0 + 3];
  const uint32_t local = c0 + c1 + c2 + c3;
  uint32_t cum = (uint32_t)wave_inclusive_sum((int)local) - local;  // keys in the bins above
  const uint32_t cs[4] = {c0, c1, c2, c3};
#pragma unroll
  for (int b = 3; b >= 0; --b) {
    if ((int)cum < need && (int)(cum + cs[b]) >= need) {
      *s_prefix = prefix | ((uint32_t)(b0 + b) << shift);
      *s_mask = mask | (255u << shift);
      *s_need = need - (int)cum;
    }
    cum += cs[b];
  }
}

// v_writelane_b32 (the LLVM intrinsic; the compiler inserts the wait states
// it needs after the VALU write of its SGPR source).
extern "C" __device__ int amdgcn_writelane(int value, int lane, int old) __asm("llvm.amdgcn.writelane.i32");

// Keys whose place the register top-k decides by ranking them: at most this
// many; more are selected from by radix passes over their exact keys.
constexpr int kMaxSurvivors = 256;
constexpr int kMaxOpen = 512;
// From estimates: the open positions are first those of the k-th estimate's
// 16-bit bin (2^-7 of its value: about 100 of an ordinary row of 32768, hundreds
// to thousands where the weights have one sign or q and K share a component).
// With more than kMaxBinOpen they are narrowed to those within twice the bound of
// the k-th estimate itself, a handful: by ranking the list up to kMaxNarrowed
// (narrow_open; rows past 8192 positions only: the shorter ones' kernel takes
// 0.2 us longer with it whatever the row), past that by two more radix passes,
// which cost 4 us.  (64 rows of 32768 positions with a shared component four times
// the noise took 1393 us when a crowded bin was scored whole, 61 now; ordinary
// rows take 56.)
constexpr int kMaxBinOpen = 128;
constexpr int kMaxNarrowed = 256;

// Shared state of one top-k workgroup (KEYS = positions it holds).  One
// space serves the radix histograms, then the row's q pieces, then the
// selected positions by rank.  The bitmaps hold one bit per position: 64-bit
// word e*16 + w covers positions e*1024 + 64w .. +63, i.e. the keys e of wave
// w's 64 lanes.
template <int KEYS>
struct TopkShared {
  union {
    uint32_t hist[2][kHistCopies * kHistPitch];  // one per radix pass of the register top-k
    struct {
      int8_t qp[4 * 3 * 2 * kChunk];  // [head block][piece][k-step] MFMA A operands
      int8_t kp[4 * 3 * 2 * kChunk];  // [group of 16 positions][piece][k-step] B operands
      float4 r[kTopkThreads];         // relu'd dots, 1 KB per wave
    };
    struct {
      int8_t qp_[4 * 3 * 2 * kChunk];  // (qp)
      uint16_t open[KEYS];             // open places, ascending
    };
    int32_t pos[KEYS];
  };
  uint64_t bits[KEYS / 64 > 0 ? KEYS / 64 : 1];    // selected
  uint64_t eqbits[KEYS / 64 > 0 ? KEYS / 64 : 1];  // ties of the k-th key
  uint2 cand[kMaxOpen];                            // (key, position), any order
  uint32_t tot[256];
  uint32_t lut[256];              // e4m3 code -> its pieces
  float w[64];                    // the row's head weights
  float q_part[kTopkThreads / 64];     // per wave: sum of |w_h| |q_h| over its heads
  uint32_t k_part[kTopkThreads / 64];  // per wave: largest |c_s| |k_s| (norm_bits)
  float band;                     // 2 E, or NaN where E is not a safe bound
  int2 scan[kTopkThreads / 64 + 1];
  uint32_t prefix, mask;
  int need, n_cand, n_above;  // n_above: open keys above the k-th largest key's bin
  uint32_t kth;               // narrow_open: the k-th key, and how many listed keys
  int n_sure, n_left;         // are taken for sure and how many stay open
};

// Rows with at most topk candidates: every candidate, then -1.
__device__ __forceinline__ bool take_all(const IndexerParams &p, int t, int32_t *out, int n) {
  if (n > p.topk) return false;
  for (int i = threadIdx.x; i < p.topk; i += kTopkThreads) {
    if (i < n) emit_pos(p, t, out, i, i);
    else out[i] = -1;
  }
  return true;
}

// One radix pass: histogram of the digit at `shift` over the keys matching
// the prefix (everything else is counted in the spare bin 256 of each copy,
// so the atomics need no branch), then the digit of the need-th largest.
// for_keys(f) calls f(key, is_candidate) for each of this thread's keys.
// `phantom` keys of value 0 that are not candidates were counted too (they
// sit in bin 0 while the prefix is 0) and are taken out of that bin.
template <typename Shared, typename ForKeys>
__device__ __forceinline__ void radix_pass(Shared &sh, int shift, ForKeys for_keys,
                                           uint32_t &prefix, uint32_t &mask, int &need,
                                           int phantom = 0) {
  for (int i = threadIdx.x; i < kHistCopies * kHistPitch; i += kTopkThreads) sh.hist[0][i] = 0;
  __syncthreads();
  uint32_t *myhist = sh.hist[0] + (threadIdx.x & (kHistCopies - 1)) * kHistPitch;
  const uint32_t pf = prefix, mk = mask;
  for_keys([&](uint32_t key, bool cand) {
    const uint32_t bin = (cand && (key & mk) == pf) ? ((key >> shift) & 255u) : 256u;
    atomicAdd(&myhist[bin], 1u);
  });
  __syncthreads();
  if (threadIdx.x < 256) {
    uint32_t c = 0;
#pragma unroll 8
    for (int j = 0; j < kHistCopies; ++j) c += sh.hist[0][j * kHistPitch + threadIdx.x];
    if (threadIdx.x == 0 && prefix == 0) c -= (uint32_t)phantom;
    sh.tot[threadIdx.x] = c;
  }
  __syncthreads();
  if (threadIdx.x < 64) pick_digit(sh.tot, prefix, mask, shift, need, &sh.prefix, &sh.mask, &sh.need);
  __syncthreads();
  prefix = sh.prefix;
  mask = sh.mask;
  need = sh.need;
}

// Key of the positions past a row's candidates in the register top-k.
constexpr uint32_t kPhantomKey = 0;

// One radix pass over the register-resident keys of a row, into histogram
// `hist`: with `zeroed` the caller zeroed it and passed a barrier since,
// otherwise the pass zeroes it first.  Under prefix pf (the digits above
// `shift` fixed so far) a key's digit is (k - pf) >> shift when it matches the
// prefix (then below 256) and at least 256 otherwise.  The first pass (no
// prefix, shift 24) counts every key; later passes issue atomics only for the
// keys under the prefix.  The copies are added by
// all threads, four per bin (eight copies each, then a quad sum).  The
// `phantom` copies of kPhantomKey are taken out of their bin.
template <int EPT, typename Shared>
__device__ __forceinline__ void radix_pass_regs(Shared &sh, uint32_t *hist, bool zeroed, int shift,
                                                const uint32_t (&key)[EPT], uint32_t &prefix,
                                                uint32_t &mask, int &need, int phantom) {
  static_assert(kTopkThreads == 4 * 256, "four threads per bin in the copy sum");
  if (!zeroed) {
    for (int i = threadIdx.x; i < kHistCopies * kHistPitch; i += kTopkThreads) hist[i] = 0;
    __syncthreads();
  }
  uint32_t *myhist = hist + (threadIdx.x & (kHistCopies - 1)) * kHistPitch;
  const uint32_t pf = prefix;
  if (mask == 0) {  // first pass: every key counts
#pragma unroll
    for (int e = 0; e < EPT; ++e) atomicAdd(&myhist[key[e] >> 24], 1u);
  } else {  // later passes: only the keys under the prefix (few) issue an atomic
#pragma unroll
    for (int e = 0; e < EPT; ++e) {
      const uint32_t d = (key[e] - pf) >> shift;
      if (d < 256u) atomicAdd(&myhist[d], 1u);
    }
  }
  __syncthreads();
  {
    const int bin = threadIdx.x >> 2, q = threadIdx.x & 3;
    constexpr int kPer = kHistCopies / 4;
    uint32_t c = 0;
#pragma unroll
    for (int j = 0; j < kPer; ++j) c += hist[(q * kPer + j) * kHistPitch + bin];
    c += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)c, 0xb1, 0xf, 0xf, false);  // quad_perm [1,0,3,2]
    c += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)c, 0x4e, 0xf, 0xf, false);  // quad_perm [2,3,0,1]
    if (bin == (int)min((kPhantomKey - pf) >> shift, 256u)) c -= (uint32_t)phantom;
    if (q == 0) sh.tot[bin] = c;
  }
  __syncthreads();
  if (threadIdx.x < 64) pick_digit(sh.tot, prefix, mask, shift, need, &sh.prefix, &sh.mask, &sh.need);
  __syncthreads();
  prefix = sh.prefix;
  mask = sh.mask;
  need = sh.need;
}

// The pieces p0, p1, p2 of four codes, from their table words, one dword each.
__device__ __forceinline__ void pack_pieces4(uint32_t v0, uint32_t v1, uint32_t v2, uint32_t v3,
                                             uint32_t (&out)[3]) {
  const uint32_t a = __builtin_amdgcn_perm(v1, v0, 0x05010400);  // v0.0 v1.0 v0.1 v1.1
  const uint32_t b = __builtin_amdgcn_perm(v3, v2, 0x05010400);
  const uint32_t c = __builtin_amdgcn_perm(v1, v0, 0x0c0c0602);  // v0.2 v1.2
  const uint32_t d = __builtin_amdgcn_perm(v3, v2, 0x0c0c0602);
  out[0] = __builtin_amdgcn_perm(b, a, 0x05040100);
  out[1] = __builtin_amdgcn_perm(b, a, 0x07060302);
  out[2] = __builtin_amdgcn_perm(d, c, 0x05040100);
}

// Eight codes (dims d .. d+7 of row or position `rc` of a group) as pieces in
// the group's six operand chunks ([piece][k-step], lane order).
__device__ __forceinline__ void store_pieces8(const uint32_t *lut, int8_t *group, int rc, int d, uint2 w) {
  uint32_t lo[3], hi[3];
  pack_pieces4(lut[w.x & 0xffu], lut[(w.x >> 8) & 0xffu], lut[(w.x >> 16) & 0xffu], lut[w.x >> 24], lo);
  pack_pieces4(lut[w.y & 0xffu], lut[(w.y >> 8) & 0xffu], lut[(w.y >> 16) & 0xffu], lut[w.y >> 24], hi);
  int8_t *dst = group + (d >> 6) * kChunk + (16 * ((d >> 4) & 3) + rc) * 16 + (d & 15);
#pragma unroll
  for (int pc = 0; pc < 3; ++pc) *(uint2 *)(dst + pc * 2 * kChunk) = make_uint2(lo[pc], hi[pc]);
}

// Exact scores of n_blocks groups of 16 positions by the whole workgroup, in
// the definition's rounding order: pos_of(b, c) is position c of group b,
// put(b, c, score) takes its score (lanes 0..15 of one wave).  Four groups a
// round: every thread makes the pieces of eight codes, a wave computes one head
// block's dots of one group (nine piece products), and one wave per group runs
// the weighted sums -- so the few groups a row leaves open take one short
// latency chain (a wave per group: 2.7 us for cfg5 rows; a wave per group and
// head block, each making the group's pieces: 3.2, bound by the table reads).
template <typename Shared, typename PosOf, typename Put>
__device__ __forceinline__ void exact_scores(const IndexerParams &p, Shared &sh, int n_blocks, PosOf pos_of,
                                             Put put) {
#pragma clang fp contract(off)
  static_assert(kTopkThreads == 4 * 16 * (kIdxDim / 8), "eight codes per thread and round");
  const int nhb = p.Hi >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ub = wave & 3, hb = wave >> 2;
#pragma unroll 1
  for (int b0 = 0; b0 < n_blocks; b0 += 4) {
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));  // the addresses below stay inside the loop
    const int lane = tid & 63, c = lane & 15, g = lane >> 4;
    const bool sums = hb == 0 && b0 + ub < n_blocks;
    float cs = 0.f;
    if (sums) cs = p.k_cs[pos_of(b0 + ub, c)];
    if (b0 + (tid >> 8) < n_blocks) {  // whole waves
      const int rc = (tid >> 4) & 15, d = (tid & 15) * 8;
      const int pos = pos_of(b0 + (tid >> 8), rc);
      const uint2 w = *(const uint2 *)(p.k_codes + (int64_t)(pos >> 4) * p.k_code_stride +
                                       (pos & 15) * kIdxDim + d);
      store_pieces8(sh.lut, sh.kp + (tid >> 8) * (6 * kChunk), rc, d, w);
    }
    __syncthreads();
    if (hb < nhb && b0 + ub < n_blocks) {
      i32x4 k[3][2];
#pragma unroll
      for (int i = 0; i < 6; ++i) k[i >> 1][i & 1] = *(const i32x4 *)(sh.kp + (ub * 6 + i) * kChunk + lane * 16);
      i32x4 C[5];
#pragma unroll
      for (int d = 0; d < 5; ++d) C[d] = i32x4{0, 0, 0, 0};
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          const i32x4 q = *(const i32x4 *)(sh.qp + ((hb * 3 + a) * 2 + ks) * kChunk + lane * 16);
#pragma unroll
          for (int b = 0; b < 3; ++b) C[a + b] = mfma(q, k[b][ks], C[a + b]);
        }
      float r[4];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        r[i] = relu_dot(C[0][i] + (C[1][i] << 7), C[2][i] + (C[3][i] << 7) + (C[4][i] << 14));
      sh.r[wave * 64 + lane] = make_float4(r[0], r[1], r[2], r[3]);
    }
    __syncthreads();
    if (sums) {
      float G = 0.f;
      for (int h = 0; h < nhb; ++h) {
        const float4 r = sh.r[(h * 4 + ub) * 64 + lane];
        const float *wl = sh.w + g * (p.Hi >> 2) + 4 * h;
        G = __builtin_fmaf(wl[0], r.x, G);
        G = __builtin_fmaf(wl[1], r.y, G);
        G = __builtin_fmaf(wl[2], r.z, G);
        G = __builtin_fmaf(wl[3], r.w, G);
      }
      const float score = sum_lane_groups(G) * cs;
      if (lane < 16) put(b0 + ub, c, score);
    }
    __syncthreads();
  }
}

// The pieces of the lane's 2 x 16 codes at src (dims +0 and +64) as its operands.
__device__ __forceinline__ void lane_pieces(const uint32_t *lut, const uint8_t *src, i32x4 (&k)[3][2]) {
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    const uint4 r = *(const uint4 *)(src + 64 * ks);
    const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      uint32_t o[3];
      pack_pieces4(lut[w[d] & 0xffu], lut[(w[d] >> 8) & 0xffu], lut[(w[d] >> 16) & 0xffu], lut[w[d] >> 24], o);
#pragma unroll
      for (int pc = 0; pc < 3; ++pc) k[pc][ks][d] = (int)o[pc];
    }
  }
}

// The same scores where there are more than a few groups: every wave takes a
// group at a time on its own, so no barrier stands between rounds and the SIMD's
// four waves hide each other's loads.  pos_of(i) is position i of the n, put(i,
// score) takes its score.  NPC = 2: no third pieces in q and the group (every
// magnitude below 32).  Bound by VALU work (table reads to pieces, the fp64 rounding
// of the dots): 32768 positions 440 us (in the rounds above 1340).
template <int NPC, typename Shared>
__device__ __forceinline__ float group_score(const IndexerParams &p, const Shared &sh, const i32x4 (&k)[3][2],
                                             float cs) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x & 63, g = lane >> 4;
  const int nhb = p.Hi >> 4;
  float G = 0.f;
#pragma unroll 1
  for (int h = 0; h < nhb; ++h) {
    i32x4 C[2 * NPC - 1];
#pragma unroll
    for (int d = 0; d < 2 * NPC - 1; ++d) C[d] = i32x4{0, 0, 0, 0};
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int a = 0; a < NPC; ++a) {
        const i32x4 q = *(const i32x4 *)(sh.qp + ((h * 3 + a) * 2 + ks) * kChunk + lane * 16);
#pragma unroll
        for (int b = 0; b < NPC; ++b) C[a + b] = mfma(q, k[b][ks], C[a + b]);
      }
    const float *wl = sh.w + g * (p.Hi >> 2) + 4 * h;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      int hi = C[2][i];
      if constexpr (NPC == 3) hi += (C[3][i] << 7) + (C[4][i] << 14);
      G = __builtin_fmaf(wl[i], relu_dot(C[0][i] + (C[1][i] << 7), hi), G);
    }
  }
  return sum_lane_groups(G) * cs;
}

template <typename Shared, typename PosOf, typename Put>
__device__ __forceinline__ void exact_scores_many(const IndexerParams &p, Shared &sh, int n, PosOf pos_of, Put put) {
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int q_third = 0;
#pragma unroll 1
  for (int i = 0; i < (p.Hi >> 4) * 2; ++i) {
    const i32x4 q = *(const i32x4 *)(sh.qp + (((i >> 1) * 3 + 2) * 2 + (i & 1)) * kChunk + lane * 16);
    q_third |= q[0] | q[1] | q[2] | q[3];
  }
#pragma unroll 1
  for (int i0 = wave * 16; i0 < n; i0 += kTopkThreads / 4) {
    const int pos = pos_of(min(i0 + c, n - 1));
    const float cs = p.k_cs[pos];
    i32x4 k[3][2];
    lane_pieces(sh.lut, p.k_codes + (int64_t)(pos >> 4) * p.k_code_stride + (pos & 15) * kIdxDim + g * 16, k);
    int third = q_third;
#pragma unroll
    for (int j = 0; j < 8; ++j) third |= k[2][j >> 2][j & 3];
    const float score = __ballot(third != 0) == 0 ? group_score<2>(p, sh, k, cs) : group_score<3>(p, sh, k, cs);
    if (lane < 16 && i0 + c < n) put(i0 + c, score);
  }
  __syncthreads();
}

// ---- the register top-k, one row per workgroup -----------------------------

// Key e of thread tid is position e*1024 + tid (coalesced), so the 64 lanes of
// a wave hold 64 consecutive positions of every e.  A buffer load over the
// `len` scores needs one 32-bit offset register for all loads (kept in flight
// together).
template <int EPT>
__device__ __forceinline__ void load_keys(const float *scores, int len, uint32_t (&key)[EPT]) {
  const auto rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(scores), 0, len * 4, kBufferFlags);
#pragma unroll
  for (int e = 0; e < EPT; ++e)
    key[e] = __builtin_amdgcn_raw_buffer_load_b32(rs, threadIdx.x * 4, e * kTopkThreads * 4, 0);
}

// Both passes' histograms (while the key loads are in flight) and the list's
// counters, ordered before their use by the caller's barrier.
template <typename Shared>
__device__ __forceinline__ void clear_counts(Shared &sh) {
  static_assert(2 * kHistCopies * kHistPitch % 4 == 0, "zeroed 16 bytes at a time");
  for (int i = threadIdx.x; i < 2 * kHistCopies * kHistPitch / 4; i += kTopkThreads)
    ((u32x4 *)&sh.hist[0][0])[i] = u32x4{0u, 0u, 0u, 0u};
  if (threadIdx.x == 0) {
    sh.n_cand = sh.n_above = sh.n_sure = sh.n_left = 0;
    sh.kth = 0;
  }
}

// Scores to order keys.  Adding +0.0 turns -0.0 into +0.0; the key orders the
// scores as unsigned integers.  The keys past the n candidates become 0, the
// lowest, and are taken out of the histograms.
template <int EPT>
__device__ __forceinline__ void to_keys(int n, uint32_t (&key)[EPT]) {
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int full = max(0, n - wave * 64) / kTopkThreads;  // keys e below it are all candidates
#pragma unroll
  for (int e = 0; e < EPT; ++e) {
    const uint32_t u = __builtin_bit_cast(uint32_t, __builtin_bit_cast(float, key[e]) + 0.0f);
    key[e] = u ^ ((uint32_t)((int32_t)u >> 31) | 0x80000000u);
    if (e >= full && e * kTopkThreads + tid >= n) key[e] = kPhantomKey;  // the first test is uniform
  }
}

// Two radix passes: the k-th largest key lies in the 16-bit bin `prefix`, and
// `need` of the bin's keys are among the k largest.
template <int EPT, typename Shared>
__device__ __forceinline__ void find_bin(const IndexerParams &p, Shared &sh, const uint32_t (&key)[EPT],
                                         int phantom, uint32_t &prefix, uint32_t &mask, int &need) {
  prefix = 0;
  mask = 0;
  need = p.topk;
#pragma unroll 1
  for (int shift = 24; shift >= 16; shift -= 8)
    radix_pass_regs(sh, sh.hist[shift == 24 ? 0 : 1], true, shift, key, prefix, mask, need, phantom);
}

// Keys above hi are taken, keys in [lo, hi] are open; `top` is the bin's last key.
template <int EPT, typename Shared>
__device__ __forceinline__ void mark_taken(Shared &sh, int n, const uint32_t (&key)[EPT], uint32_t lo,
                                           uint32_t hi, uint32_t top) {
  constexpr int kWaves = kTopkThreads / 64;
  int tid = threadIdx.x;
  // many keys' positions are made here, not kept from to_keys on (32 registers:
  // 64 rows of 32768 49.6 -> 47.2 us)
  if constexpr (EPT > 8) asm volatile("" : "+v"(tid));
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // known uniform: scalar masks
  uint32_t *bits32 = (uint32_t *)sh.bits;  // word w: positions 32w .. 32w+31
  // The selection as a position bitmap, built from ballots of the registers
  // (64-bit word e*16 + wave holds key e of the wave's lanes: lane 2e + h
  // collects half h and one store per lane writes them).  Waves holding open
  // keys list them (key, position).
  uint32_t bw = 0;
#pragma unroll
  for (int e = 0; e < EPT; ++e) {
    const uint64_t ab = __ballot(key[e] > hi);
    const uint64_t sb = __ballot(key[e] >= lo) & ~ab;
    bw = (uint32_t)amdgcn_writelane((int)(uint32_t)ab, 2 * e, (int)bw);
    bw = (uint32_t)amdgcn_writelane((int)(uint32_t)(ab >> 32), 2 * e + 1, (int)bw);
    if (sb != 0) {  // uniform
      const int pos = e * kTopkThreads + tid;
      const bool open = ((sb >> lane) & 1) && pos < n;  // (lo may be a phantom's key)
      const uint64_t ob = __ballot(open), tb = __ballot(open && key[e] > top);
      int o = 0;
      if (lane == 0) {
        o = atomicAdd(&sh.n_cand, __popcll(ob));
        if (tb != 0) atomicAdd(&sh.n_above, __popcll(tb));
      }
      o = __builtin_amdgcn_readfirstlane(o) +
          __builtin_amdgcn_mbcnt_hi((uint32_t)(ob >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)ob, 0));
      if (open && o < kMaxOpen) sh.cand[o] = make_uint2(key[e], (uint32_t)pos);
    }
  }
  if (lane < 2 * EPT) bits32[((lane >> 1) * kWaves + wave) * 2 + (lane & 1)] = bw;
}

// Marks the `need` largest of the listed keys: key descending, position
// ascending.  Four lanes per key each count the keys ahead of it in a quarter
// of the list, and two DPP quad swaps add the counts.
template <typename Shared>
__device__ __forceinline__ void rank_open(Shared &sh, int n_open, int need) {
  const int tid = threadIdx.x;
  uint32_t *bits32 = (uint32_t *)sh.bits;
  for (int i0 = 0; i0 < n_open; i0 += kTopkThreads / 4) {
    const int i = i0 + (tid >> 2), q = tid & 3;
    if (i < ((n_open + 15) & ~15)) {  // whole waves
      const uint2 me = sh.cand[min(i, n_open - 1)];
      int r = 0;
      // four reads in flight per step (entries past the list count nothing)
      for (int j0 = q; j0 < n_open; j0 += 16) {
        uint2 c[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) c[u] = sh.cand[min(j0 + 4 * u, kMaxOpen - 1)];
#pragma unroll
        for (int u = 0; u < 4; ++u)
          r += j0 + 4 * u < n_open && (c[u].x > me.x || (c[u].x == me.x && c[u].y < me.y));
      }
      r += __builtin_amdgcn_update_dpp(0, r, 0xb1, 0xf, 0xf, false);  // quad_perm [1,0,3,2]
      r += __builtin_amdgcn_update_dpp(0, r, 0x4e, 0xf, 0xf, false);  // quad_perm [2,3,0,1]
      if (q == 0 && i < n_open && r < need) atomicOr(&bits32[me.y >> 5], 1u << (me.y & 31));
    }
  }
  __syncthreads();
}

// The marked places (of the first n), as positions at(place) or their slots, in
// ascending order.
template <int KEYS, typename Shared, typename At>
__device__ __forceinline__ void write_marked(const IndexerParams &p, Shared &sh, int t, int n, int32_t *out,
                                             At at) {
  const int tid = threadIdx.x;
  const uint32_t *bits32 = (const uint32_t *)sh.bits;
  int unused;
  // Output ranks in position order: thread tid owns bitmap word tid; the
  // selected positions go to LDS by rank (the scan's barriers order this
  // after every bitmap read), then each thread maps up to four of them
  // through the block table with the loads issued together and stores them
  // coalesced.
  const int nw = n - tid * 32;  // this word's positions below n
  uint32_t sel = tid < KEYS / 32 ? bits32[tid] : 0u;
  sel &= nw >= 32 ? ~0u : (nw <= 0 ? 0u : (1u << nw) - 1u);
  int n_sel;
  const int2 rx = block_exclusive_scan2(__builtin_popcount(sel), 0, sh.scan, &n_sel, &unused);
  int o = rx.x;
  while (sel != 0) {
    const int e = __builtin_ctz(sel);
    sel &= sel - 1;
    sh.pos[o++] = tid * 32 + e;
  }
  __syncthreads();
  for (int r0 = tid; r0 < p.topk; r0 += 4 * kTopkThreads) {
    int v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = at(sh.pos[min(r0 + u * kTopkThreads, p.topk - 1)]);
    if (p.block_table != nullptr) {
      const int32_t *bt = p.block_table + (int64_t)t * p.bt_stride;
      int page[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) page[u] = bt[v[u] / p.page_size];
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = page[u] * p.page_size + v[u] % p.page_size;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (r0 + u * kTopkThreads < p.topk) out[r0 + u * kTopkThreads] = v[u];
  }
}

// Marks the k largest of exact keys: the keys above the bin are taken, those in
// it ranked, or, where many share it, two more passes pin the k-th key.  The
// `phantom` keys past the first n are 0 (the lowest) and may be marked.
template <int EPT, typename Shared>
__device__ __forceinline__ void mark_exact(const IndexerParams &p, Shared &sh, int n,
                                           const uint32_t (&key)[EPT], int phantom) {
  constexpr int KEYS = EPT * kTopkThreads;
  constexpr int kWaves = kTopkThreads / 64;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  uint32_t *bits32 = (uint32_t *)sh.bits;
  uint32_t prefix, mask;
  int need, unused;
  clear_counts(sh);
  __syncthreads();
  find_bin(p, sh, key, phantom, prefix, mask, need);
  mark_taken(sh, n, key, prefix, prefix | 0xffffu, prefix | 0xffffu);
  __syncthreads();
  const int n_open = sh.n_cand;
  if (n_open <= kMaxSurvivors) {  // uniform
    rank_open(sh, n_open, need);
  } else {
    // Many keys share the bin: two more passes pin the k-th key itself;
    // keys above it are taken, and `need` of its ties, lowest positions first.
    need = sh.need;
#pragma unroll 1
    for (int shift = 8; shift >= 0; shift -= 8)
      radix_pass_regs(sh, sh.hist[0], false, shift, key, prefix, mask, need, phantom);
    // (Ties past n sit after every real position and `need` counts real
    // ones only, so they are never taken; the masking below clears the rest.)
#pragma unroll
    for (int e = 0; e < EPT; ++e) {
      const uint64_t gb = __ballot(key[e] > prefix);
      const uint64_t qb = __ballot(key[e] == prefix);
      if (lane == 0) {
        sh.bits[e * kWaves + wave] = gb;
        sh.eqbits[e * kWaves + wave] = qb;
      }
    }
    __syncthreads();
    uint32_t eq = tid < KEYS / 32 ? ((const uint32_t *)sh.eqbits)[tid] : 0u;
    int tot_eq;
    const int2 ex = block_exclusive_scan2(__builtin_popcount(eq), 0, sh.scan, &tot_eq, &unused);
    uint32_t take = 0;
    for (int left = need - ex.x; left > 0 && eq != 0; --left) {
      take |= eq & (~eq + 1);
      eq &= eq - 1;
    }
    if (take != 0) bits32[tid] |= take;  // this thread's own word
    __syncthreads();
  }
}

// ---- the estimates' bound ---------------------------------------------------

// Eight q codes of a row per thread, for the bound and the exact scores: 16
// threads per head, heads in the order of the MFMA rows (q_operands).
struct RowCodes {
  int row, hb, head;  // MFMA row, head block and head
  uint2 codes;
  float w;  // the head's weight
};
__device__ __forceinline__ RowCodes load_row_codes(const IndexerParams &p, int t) {
  const int tid = threadIdx.x;
  RowCodes r;
  r.row = (tid >> 4) & 15;
  r.hb = tid >> 8;
  r.head = (r.row >> 2) * (p.Hi >> 2) + 4 * r.hb + (r.row & 3);
  r.codes = make_uint2(0, 0);
  r.w = 0.f;
  if (tid < p.Hi * 16) {
    r.codes = *(const uint2 *)(p.q + ((int64_t)t * p.Hi + r.head) * kIdxDim + (tid & 15) * 8);
    r.w = p.w[(int64_t)t * p.Hi + r.head];
  }
  return r;
}

// Whether any of the 16 threads' codes (a head's) is not zero.
__device__ __forceinline__ bool row_any_code(uint2 codes) {
  const bool any = ((drop_nan(codes.x) | drop_nan(codes.y)) & 0x7f7f7f7fu) != 0;
  return ((__ballot(any) >> (threadIdx.x & 48)) & 0xffffu) != 0;
}

// Each wave's share of sum_h |w_h| |q_h| (four heads) and of max_s |c_s| |k_s|
// over k_max blocks [blk0, blk1); the weights and the code table.  bound()
// follows, behind a barrier.
template <typename Shared>
__device__ __forceinline__ void bound_shares(const IndexerParams &p, Shared &sh, const RowCodes &r, int blk0,
                                             int blk1) {
  constexpr int kWaves = kTopkThreads / 64;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  uint32_t kn = 0;
  for (int b = blk0 + tid; b < blk1; b += kTopkThreads) kn = max(kn, (uint32_t)p.k_max[b] >> kMaxXBits);
  float x = row_sum_last(sum_squares8(drop_nan(r.codes.x), drop_nan(r.codes.y)));
  // (a product that is not zero counts as at least the smallest normal, so the
  // sum is 0 only where every score is 0)
  x = (lane & 15) == 15 ? __builtin_amdgcn_sqrtf(x) * fabsf(r.w) : 0.f;
  const bool any = row_any_code(r.codes);
  if ((lane & 15) == 15 && x == 0.f && r.w != 0.f && any) x = 0x1p-126f;
  x = rows_sum_last(x);
  const uint32_t m = wave_max_last(kn);
  if (lane == 63) {
    sh.q_part[wave] = x;
    sh.k_part[wave] = m;
  }
  if (tid < p.Hi * 16 && (tid & 15) == 0) sh.w[r.head] = r.w;
  if (wave >= kWaves - 4) sh.lut[tid & 255] = piece_word(tid & 255);
}

// 2 E into sh.band, or NaN where E is not a safe bound (by the last wave; read
// behind a later barrier).  0: every exact score is 0, and so is its estimate.
template <typename Shared>
__device__ __forceinline__ void bound(Shared &sh) {
  constexpr int kWaves = kTopkThreads / 64;
  const int lane = threadIdx.x & 63;
  if (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) != kWaves - 1) return;
  const int i = min(lane, kWaves - 1);
  const float x = row_sum_last(lane < kWaves ? sh.q_part[i] : 0.f);
  const uint32_t m = wave_max_last(lane < kWaves ? sh.k_part[i] : 0u);
  const float W = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(x), 15));
  const float A = norm_from_bits(__builtin_amdgcn_readlane(m, 63)) * 0x1p18f, WA = W * A;
  // no overflow on either side's way (the exact sum carries 2^18), no
  // underflow that matters, no NaN
  const bool safe = W > 0x1p-60f && W < 0x1p95f && A > 0x1p-60f && A < 0x1p60f && WA < 0x1p100f;
  const bool zero = (W == 0.f && A < INFINITY) || (A == 0.f && W < INFINITY);
  if (lane == 0)
    sh.band = safe ? 2.f * kEstimateError * WA : zero ? 0.f : __uint_as_float(0x7fc00000u);
}

// The row's q pieces, in the histograms' place.
template <typename Shared>
__device__ __forceinline__ void store_row_pieces(const IndexerParams &p, Shared &sh, const RowCodes &r) {
  if ((int)threadIdx.x < p.Hi * 16)
    store_pieces8(sh.lut, sh.qp + r.hb * (6 * kChunk), r.row, (threadIdx.x & 15) * 8, r.codes);
}

// Narrows the list (at most kMaxNarrowed) to the keys within band of the k-th
// key, which is the need-th largest listed one; the keys above are marked, and
// `need` falls by as many.  Returns how many are left.  Four lanes per key, as in
// rank_open.  Once per workgroup.
template <typename Shared>
__device__ __forceinline__ int narrow_open(Shared &sh, int n_open, float band, int &need) {
  static_assert(kMaxNarrowed <= kTopkThreads / 4, "one key per four lanes");
  const int i = threadIdx.x >> 2, q = threadIdx.x & 3, lane = threadIdx.x & 63;
  const bool mine = q == 0 && i < n_open;
  const uint2 me = sh.cand[min(i, n_open - 1)];
  int reach = 0;  // listed keys of at least mine
  if (i < ((n_open + 15) & ~15)) {  // whole waves
    for (int j0 = q; j0 < n_open; j0 += 16) {
      uint32_t c[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) c[u] = sh.cand[min(j0 + 4 * u, kMaxOpen - 1)].x;
#pragma unroll
      for (int u = 0; u < 4; ++u) reach += j0 + 4 * u < n_open && c[u] >= me.x;
    }
    reach += __builtin_amdgcn_update_dpp(0, reach, 0xb1, 0xf, 0xf, false);  // quad_perm [1,0,3,2]
    reach += __builtin_amdgcn_update_dpp(0, reach, 0x4e, 0xf, 0xf, false);  // quad_perm [2,3,0,1]
  }
  if (mine && reach >= need) atomicMax(&sh.kth, me.x);
  __syncthreads();  // (and every wave has read the list)
  const float kth = key_value(sh.kth);
  const uint32_t lo = max(order_key(kth - band), 1u), hi = order_key(kth + band);
  const bool sure = mine && me.x > hi, open = mine && me.x >= lo && me.x <= hi;
  if (sure) atomicOr((uint32_t *)sh.bits + (me.y >> 5), 1u << (me.y & 31));
  const uint64_t sb = __ballot(sure), ob = __ballot(open);
  int o = 0;
  if (lane == 0) {
    if (sb != 0) atomicAdd(&sh.n_sure, __popcll(sb));
    if (ob != 0) o = atomicAdd(&sh.n_left, __popcll(ob));
  }
  o = __builtin_amdgcn_readfirstlane(o) +
      __builtin_amdgcn_mbcnt_hi((uint32_t)(ob >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)ob, 0));
  if (open) sh.cand[o] = me;
  __syncthreads();
  need -= sh.n_sure;
  return sh.n_left;
}

// Marks the keys that are taken for sure and lists the open ones: those within
// band of the k-th key's bin [prefix, top], or, where they are many (see
// kMaxBinOpen) and the band is a safe bound, within band of the k-th key
// itself (prefix == top where two more passes gave it).  Returns how many are
// open, of which `need` are among the k largest.  With the row's q pieces in
// the histograms' place.
template <int EPT, typename Shared>
__device__ __forceinline__ int mark_open(const IndexerParams &p, Shared &sh, const RowCodes &rc, int n,
                                         const uint32_t (&key)[EPT], int phantom, float band, uint32_t &prefix,
                                         uint32_t &top, uint32_t mask, int &need) {
  top = prefix | 0xffffu;
#pragma unroll 1
  for (;;) {
    mark_taken(sh, n, key, max(order_key(key_value(prefix) - band), 1u), order_key(key_value(top) + band), top);
    store_row_pieces(p, sh, rc);
    __syncthreads();
    const int n_open = sh.n_cand;
    const int above = sh.n_above;
    constexpr int kNoPasses = EPT > 8 ? kMaxNarrowed : kMaxBinOpen;
    if (!(band > 0.f) || n_open <= kNoPasses || top == prefix) {  // uniform
      need += above;  // (the keys above the bin, or the k-th, that are open are not taken for sure)
      if constexpr (EPT > 8)
        if (band > 0.f && n_open > kMaxBinOpen && top != prefix) return narrow_open(sh, n_open, band, need);
      return n_open;
    }
    __syncthreads();  // every wave has read the counts
    if (threadIdx.x == 0) sh.n_cand = sh.n_above = 0;
#pragma unroll 1
    for (int shift = 8; shift >= 0; shift -= 8)
      radix_pass_regs(sh, sh.hist[0], false, shift, key, prefix, mask, need, phantom);
    top = prefix;
  }
}

// Exact scores of the listed open positions (at most kMaxOpen) in place of their
// estimates: place_of(place) is a position.
template <typename Shared, typename PosOf>
__device__ __forceinline__ void score_listed(const IndexerParams &p, Shared &sh, int n_open, PosOf pos_of) {
  if (n_open <= 64) {
    exact_scores(p, sh, (n_open + 15) >> 4,
                 [&](int b, int c) { return pos_of((int)sh.cand[min(b * 16 + c, n_open - 1)].y); },
                 [&](int b, int c, float v) {
                   if (b * 16 + c < n_open) sh.cand[b * 16 + c].x = max(order_key(v), 1u);
                 });
  } else {
    exact_scores_many(p, sh, n_open, [&](int i) { return pos_of((int)sh.cand[i].y); },
                      [&](int i, float v) { sh.cand[i].x = max(order_key(v), 1u); });
  }
}

// More open keys than are listed (positions apart by less than the bound, or no
// safe bound: all): the places of the keys in [lo, hi] among the first n go to
// sh.open, as marks to sh.eqbits, and the keys above hi as marks to sh.bits.
// Returns how many are open; `taken` how many are above.
template <int EPT, typename Shared>
__device__ __forceinline__ int list_open(Shared &sh, int n, const uint32_t (&key)[EPT], uint32_t lo, uint32_t hi,
                                         int &taken) {
  constexpr int kWords = EPT * kTopkThreads / 32, kWaves = kTopkThreads / 64;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
#pragma unroll
  for (int e = 0; e < EPT; ++e) {
    const uint64_t gb = __ballot(key[e] > hi);
    const uint64_t ob = __ballot(key[e] >= lo) & ~gb;
    if (lane == 0) {
      sh.bits[e * kWaves + wave] = gb;
      sh.eqbits[e * kWaves + wave] = ob;
    }
  }
  __syncthreads();
  const int nw = n - tid * 32;  // this word's places below n
  uint32_t open = tid < kWords ? ((const uint32_t *)sh.eqbits)[tid] : 0u;
  open &= nw >= 32 ? ~0u : (nw <= 0 ? 0u : (1u << nw) - 1u);
  const int above = tid < kWords ? __builtin_popcount(((const uint32_t *)sh.bits)[tid]) : 0;
  if (tid < kWords) ((uint32_t *)sh.eqbits)[tid] = open;
  int total;
  int o = block_exclusive_scan2(__builtin_popcount(open), above, sh.scan, &total, &taken).x;
  while (open != 0) {
    sh.open[o++] = (uint16_t)(tid * 32 + __builtin_ctz(open));
    open &= open - 1;
  }
  __syncthreads();
  return total;
}

// The keys for a selection from exact scores: open ones keep theirs, the taken
// rank above all, the others below (as phantoms).
template <int EPT, typename Shared>
__device__ __forceinline__ void keep_open(const Shared &sh, uint32_t (&key)[EPT]) {
  constexpr int kWaves = kTopkThreads / 64;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // (lane 2e + h holds half h of the wave's words of keys e)
  const int word = ((min(lane, 2 * EPT - 1) >> 1) * kWaves + wave) * 2 + (lane & 1);
  const int gw = ((const int *)sh.bits)[word], ow = ((const int *)sh.eqbits)[word];
#pragma unroll
  for (int e = 0; e < EPT; ++e) {
    const int g = (lane & 32) ? __builtin_amdgcn_readlane(gw, 2 * e + 1) : __builtin_amdgcn_readlane(gw, 2 * e);
    const int o = (lane & 32) ? __builtin_amdgcn_readlane(ow, 2 * e + 1) : __builtin_amdgcn_readlane(ow, 2 * e);
    key[e] = (g >> (lane & 31)) & 1 ? ~0u : (o >> (lane & 31)) & 1 ? key[e] : kPhantomKey;
  }
  __syncthreads();  // the marks are free
}

// Top-k of one row per workgroup from exact scores.
template <int EPT>
__global__ __launch_bounds__(kTopkThreads) void dsa_idx_topk_kernel(IndexerParams p) {
  static_assert(EPT <= 32, "one 32-bit bitmap word per thread at most");
  constexpr int KEYS = EPT * kTopkThreads;
  __shared__ __attribute__((aligned(16))) TopkShared<KEYS> sh;
  const int t = blockIdx.x;
  int32_t *out = p.out + (int64_t)t * p.topk;
  const int n = candidates(p, t);  // candidates 0..n-1
  if (take_all(p, t, out, n)) return;               // n > topk >= 1 below
  uint32_t key[EPT];
  load_keys(p.scores + (int64_t)t * p.S, p.S, key);
  to_keys(n, key);
  mark_exact(p, sh, n, key, KEYS - n);
  write_marked<KEYS>(p, sh, t, n, out, [](int i) { return i; });
}

// Top-k of one row per workgroup from estimates.  The exact k-th largest score
// lies within E of the estimates' bin, so keys more than 2 E above the bin are
// taken, those more than 2 E below it are not, and the exact scores of the ones
// between (a few dozen of 32768 ordinary scores) are computed here and ranked.
// A crowded bin is narrowed to the k-th estimate first (mark_open).  Where more
// than kMaxOpen scores are still closer than E tells apart, or E is not a safe
// bound (huge, tiny or non-finite weights or scales: all are open), the open
// positions' exact scores replace their estimates in memory and the row is
// selected from once more -- by this one workgroup: 64 rows of 32768
// positions all tied at 0 take 471 us, of which a third are one same row 222 (115
// and 83 with every score from the score kernel).
template <int EPT>
__global__ __launch_bounds__(kTopkThreads) void dsa_idx_topk_estimates_kernel(IndexerParams p) {
  constexpr int KEYS = EPT * kTopkThreads;
  __shared__ __attribute__((aligned(16))) TopkShared<KEYS> sh;
  const int t = blockIdx.x;
  float *row = p.scores + (int64_t)t * p.S;
  int32_t *out = p.out + (int64_t)t * p.topk;
  const RowCodes rc = load_row_codes(p, t);
  uint32_t key[EPT];
  load_keys(row, p.S, key);  // beside the load of the row's limit
  const int n = candidates(p, t);  // candidates 0..n-1
  if (take_all(p, t, out, n)) return;               // n > topk >= 1 below

  clear_counts(sh);
  bound_shares(p, sh, rc, 0, (n + 15) >> 4);
  __syncthreads();
  bound(sh);
  to_keys(n, key);
  uint32_t prefix, mask;
  int need;
  find_bin(p, sh, key, KEYS - n, prefix, mask, need);
  const float band = sh.band;
  int phantom = KEYS - n;
  uint32_t top;
  int n_open = mark_open(p, sh, rc, n, key, phantom, band, prefix, top, mask, need);
  if (band == band && n_open <= kMaxOpen) {  // uniform
    score_listed(p, sh, n_open, [](int i) { return i; });
    rank_open(sh, n_open, need);
    write_marked<KEYS>(p, sh, t, n, out, [](int i) { return i; });
    return;
  }
  __syncthreads();  // every wave has read n_cand: mark_exact clears it
  if (!(band == 0.f)) {  // (estimates of zeros are exact)
    int taken;
    const bool safe = band == band;  // else every position is open
    const uint32_t lo = safe ? max(order_key(key_value(prefix) - band), 1u) : 0u;
    const uint32_t hi = safe ? order_key(key_value(top) + band) : ~0u;
    n_open = list_open(sh, n, key, lo, hi, taken);
    exact_scores_many(p, sh, n_open, [&](int i) { return (int)sh.open[i]; },
                      [&](int i, float v) { row[sh.open[i]] = v; });
    load_keys(row, p.S, key);
    to_keys(n, key);
    keep_open(sh, key);
    phantom = KEYS - n_open - taken;
  }
  mark_exact(p, sh, n, key, phantom);
  write_marked<KEYS>(p, sh, t, n, out, [](int i) { return i; });
}

// ---- rows longer than the registers hold: chunks, then their lists ----------
//
// A row of p.n_chunks chunks: one workgroup per chunk lists the chunk's
// positions that can be among the row's k largest -- those whose estimate is
// within 2 E of the chunk's own k-th largest, or above -- and one workgroup per
// row selects from the lists as the kernel above does from a row.  A list
// takes the place of its chunk's estimates (all of a chunk's are in registers
// by then): p.list_len order keys, 0 past the list's end, then their
// positions, ascending.  A chunk whose bound is not safe, or too many of whose
// scores lie within the bound of the k-th, lists its k largest, by the exact
// scores of those.  2 rows of 131071 positions, top-k
// 2048: chunks 17 us, lists 17, against 235 for the four passes over exact
// scores (one workgroup re-reading the row, its last pass uncoalesced).

// The chunk's marked keys (of its first n places) as its list.
template <int EPT, typename Shared>
__device__ __forceinline__ void write_list(const IndexerParams &p, Shared &sh, int n, int c0,
                                           const uint32_t (&key)[EPT], int total, float *list) {
  constexpr int kWaves = kTopkThreads / 64;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int *rank = (const int *)sh.eqbits;  // first rank of each 32-place word
  uint32_t *keys = (uint32_t *)list;
  int32_t *places = (int32_t *)list + p.list_len;
#pragma unroll
  for (int e = 0; e < EPT; ++e) {
    const uint64_t m = sh.bits[e * kWaves + wave];
    if (m != 0 && ((m >> lane) & 1)) {
      const int o = rank[(e * kWaves + wave) * 2] +
                    __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
      keys[o] = max(key[e], 1u);
      places[o] = c0 + e * kTopkThreads + tid;
    }
  }
  for (int i = total + tid; i < p.list_len; i += kTopkThreads) keys[i] = 0;
}

// Masks the marks to the first n places and ranks their words; returns how
// many are marked.
template <int KEYS, typename Shared>
__device__ __forceinline__ int rank_marks(Shared &sh, int n) {
  const int tid = threadIdx.x;
  uint32_t *bits32 = (uint32_t *)sh.bits;
  const int nw = n - tid * 32;
  uint32_t sel = tid < KEYS / 32 ? bits32[tid] : 0u;
  sel &= nw >= 32 ? ~0u : (nw <= 0 ? 0u : (1u << nw) - 1u);
  int total, unused;
  const int2 r = block_exclusive_scan2(__builtin_popcount(sel), 0, sh.scan, &total, &unused);
  if (tid < KEYS / 32) {
    bits32[tid] = sel;
    ((int *)sh.eqbits)[tid] = r.x;
  }
  __syncthreads();
  return total;
}

template <int EPT>
__global__ __launch_bounds__(kTopkThreads) void dsa_idx_topk_chunk_kernel(IndexerParams p) {
  constexpr int KEYS = EPT * kTopkThreads;
  __shared__ __attribute__((aligned(16))) TopkShared<KEYS> sh;
  const int t = blockIdx.y, c0 = blockIdx.x * p.chunk;
  const int tid = threadIdx.x;
  float *chunk = p.scores + (int64_t)t * p.S + c0;
  const RowCodes rc = load_row_codes(p, t);
  uint32_t key[EPT];
  load_keys(chunk, min(p.chunk, p.S - c0), key);
  const int n_row = candidates(p, t), n = min(n_row - c0, p.chunk);
  if (n_row <= p.topk) return;  // the row takes all its candidates
  if (n <= p.topk) {            // few or none: all are listed
    to_keys(max(n, 0), key);
    __syncthreads();  // every wave's keys have arrived: the list may take their place
#pragma unroll
    for (int e = 0; e < EPT; ++e) {
      const int i = e * kTopkThreads + tid;
      if (i < p.list_len) {
        ((uint32_t *)chunk)[i] = i < n ? max(key[e], 1u) : 0u;
        ((int32_t *)chunk)[p.list_len + i] = c0 + i;
      }
    }
    return;
  }
  clear_counts(sh);
  bound_shares(p, sh, rc, c0 >> 4, (c0 + n + 15) >> 4);
  __syncthreads();
  bound(sh);
  to_keys(n, key);
  uint32_t prefix, mask;
  int need;
  find_bin(p, sh, key, KEYS - n, prefix, mask, need);
  const float band = sh.band;
  int phantom = KEYS - n, total;
  uint32_t lo;
  // every key from 2 E below the k-th key's bin on; where those do not fit, from
  // 2 E below the k-th key itself, which two more passes give
#pragma unroll 1
  for (bool pinned = false;; pinned = true) {
    lo = max(order_key(key_value(prefix) - band), 1u);
    mark_taken(sh, n, key, ~0u, lo - 1, ~0u);
    __syncthreads();
    total = rank_marks<KEYS>(sh, n);
    if (!(band > 0.f) || total <= p.list_len || pinned) break;  // uniform
#pragma unroll 1
    for (int shift = 8; shift >= 0; shift -= 8)
      radix_pass_regs(sh, sh.hist[0], false, shift, key, prefix, mask, need, phantom);
  }
  if (!(band == band && total <= p.list_len)) {  // uniform
    if (!(band == 0.f)) {
      int taken;
      const bool safe = band == band;
      store_row_pieces(p, sh, rc);
      const int n_open = list_open(sh, n, key, safe ? lo : 0u, safe ? order_key(key_value(prefix) + band) : ~0u, taken);
      exact_scores_many(p, sh, n_open, [&](int i) { return c0 + (int)sh.open[i]; },
                        [&](int i, float v) { chunk[sh.open[i]] = v; });
      load_keys(chunk, n, key);
      to_keys(n, key);
      keep_open(sh, key);
      phantom = KEYS - n_open - taken;
    }
    mark_exact(p, sh, n, key, phantom);
    total = rank_marks<KEYS>(sh, n);
    if (!(band == 0.f)) {  // the taken keep their estimates
      load_keys(chunk, n, key);
      to_keys(n, key);
      __syncthreads();  // every wave's keys have arrived: the list may take their place
    }
  }
  write_list(p, sh, n, c0, key, total, chunk);
}

// Selection of a row from its chunks' lists (EPT * 1024 places, list_len per list).
template <int EPT>
__global__ __launch_bounds__(kTopkThreads) void dsa_idx_topk_merge_kernel(IndexerParams p) {
  constexpr int KEYS = EPT * kTopkThreads;
  __shared__ __attribute__((aligned(16))) TopkShared<KEYS> sh;
  const int t = blockIdx.x;
  const int tid = threadIdx.x;
  float *row = p.scores + (int64_t)t * p.S;
  int32_t *out = p.out + (int64_t)t * p.topk;
  const RowCodes rc = load_row_codes(p, t);
  // place i: entry i % list_len (a power of two, at least 1024) of list i / list_len
  auto entry = [&](int i) { return (i >> p.list_shift) * p.chunk + (i & (p.list_len - 1)); };
  const int places = p.n_chunks << p.list_shift;
  uint32_t key[EPT];
  auto load_lists = [&]() {
    const auto rs = __builtin_amdgcn_make_buffer_rsrc(row, 0, p.S * 4, kBufferFlags);
#pragma unroll
    for (int e = 0; e < EPT; ++e)
      key[e] = e * kTopkThreads < places
                   ? __builtin_amdgcn_raw_buffer_load_b32(rs, tid * 4, entry(e * kTopkThreads) * 4, 0)
                   : 0u;
  };
  load_lists();
  const int n = candidates(p, t);
  if (take_all(p, t, out, n)) return;  // (nothing was listed)

  auto position = [&](int i) { return ((const int32_t *)row)[entry(i) + p.list_len]; };
  clear_counts(sh);
  bound_shares(p, sh, rc, 0, (n + 15) >> 4);
  __syncthreads();
  bound(sh);
  uint32_t prefix, mask;
  int need;
  find_bin(p, sh, key, 0, prefix, mask, need);  // (empty entries are the lowest keys)
  const float band = sh.band;
  uint32_t top;
  int n_open = mark_open(p, sh, rc, KEYS, key, 0, band, prefix, top, mask, need);
  if (band == band && n_open <= kMaxOpen) {  // uniform
    score_listed(p, sh, n_open, position);
    rank_open(sh, n_open, need);
    write_marked<KEYS>(p, sh, t, KEYS, out, position);
    return;
  }
  __syncthreads();  // every wave has read n_cand: mark_exact clears it
  int phantom = 0;
  if (!(band == 0.f)) {
    int taken;
    uint32_t *keys = (uint32_t *)row;
    const bool safe = band == band;  // else every listed position is open
    const uint32_t lo = safe ? max(order_key(key_value(prefix) - band), 1u) : 1u;
    const uint32_t hi = safe ? order_key(key_value(top) + band) : ~0u;
    n_open = list_open(sh, KEYS, key, lo, hi, taken);
    exact_scores_many(p, sh, n_open, [&](int i) { return position((int)sh.open[i]); },
                      [&](int i, float v) { keys[entry((int)sh.open[i])] = max(order_key(v), 1u); });
    load_lists();
    keep_open(sh, key);
    phantom = KEYS - n_open - taken;
  }
  mark_exact(p, sh, KEYS, key, phantom);
  write_marked<KEYS>(p, sh, t, KEYS, out, position);
}

// Rows longer than the register kernel holds: the same selection, reading
// the row from memory in every pass.
__global__ __launch_bounds__(kTopkThreads) void dsa_idx_topk_stream_kernel(IndexerParams p) {
  __shared__ TopkShared<0> sh;
  const int t = blockIdx.x;
  const float *row = p.scores + (int64_t)t * p.S;
  int32_t *out = p.out + (int64_t)t * p.topk;
  const int n = candidates(p, t);
  if (take_all(p, t, out, n)) return;

  uint32_t prefix = 0, mask = 0;
  int need = p.topk;
  for (int shift = 24; shift >= 0; shift -= 8)
    radix_pass(sh, shift,
               [&](auto f) {
                 for (int i = threadIdx.x; i < n; i += kTopkThreads) f(order_key(row[i]), true);
               },
               prefix, mask, need);
  // ordered compaction: thread i owns positions [i*chunk, (i+1)*chunk)
  const int chunk = (n + kTopkThreads - 1) / kTopkThreads;
  const int c0 = min(n, (int)threadIdx.x * chunk), c1 = min(n, c0 + chunk);
  int n_gt = 0, n_eq = 0;
  for (int i = c0; i < c1; ++i) {
    const uint32_t key = order_key(row[i]);
    n_gt += key > prefix;
    n_eq += key == prefix;
  }
  int tot_gt, tot_eq;
  const int2 ex = block_exclusive_scan2(n_gt, n_eq, sh.scan, &tot_gt, &tot_eq);
  int o = ex.x + min(ex.y, need);
  int eq_left = need - ex.y;
  for (int i = c0; i < c1; ++i) {
    const uint32_t key = order_key(row[i]);
    bool sel = key > prefix;
    if (key == prefix) {
      sel = eq_left > 0;
      --eq_left;
    }
    if (sel) emit_pos(p, t, out, i, o++);
  }
}

template <int EPT>
hipError_t launch_topk_regs(const IndexerParams &p, hipStream_t stream) {
  const dim3 grid(p.T), block(kTopkThreads);
  if (p.estimated) hipLaunchKernelGGL(dsa_idx_topk_estimates_kernel<EPT>, grid, block, 0, stream, p);
  else hipLaunchKernelGGL(dsa_idx_topk_kernel<EPT>, grid, block, 0, stream, p);
  return hipGetLastError();
}

template <int NHB>
hipError_t launch_estimate(const IndexerParams &p, dim3 grid, hipStream_t stream) {
  const dim3 block(kEstWaves * 64);
  if (!p.est_fused) hipLaunchKernelGGL((dsa_idx_estimate_kernel<NHB, kPrepared>), grid, block, 0, stream, p);
  else if (p.k_cache) hipLaunchKernelGGL((dsa_idx_estimate_kernel<NHB, kPaged>), grid, block, 0, stream, p);
  else hipLaunchKernelGGL((dsa_idx_estimate_kernel<NHB, kFlat>), grid, block, 0, stream, p);
  return hipGetLastError();
}

}  // namespace

// Rows longer than 32768 positions run in chunks of at most that: as few as
// possible (the lists of all must fit one workgroup's registers, and two
// list lengths a chunk).  A list holds twice the top-k or so: the chunk's k
// largest, and those whose estimates are too close to tell.
static bool chunk_plan(const IndexerParams &p, int *chunk, int *n_chunks, int *list_shift) {
  constexpr int kMax = kTopkThreads * kMaxRegEpt;
  const int c = (p.S + kMax - 1) / kMax;
  const int len = ((p.S + c - 1) / c + 15) / 16 * 16;
  int shift = 10;
  while ((1 << shift) < p.topk + 512) {
    if (++shift > 15) return false;
  }
  if ((int64_t)c << shift > kMax || p.S - (int64_t)(c - 1) * len < 2 << shift) return false;
  *chunk = len;
  *n_chunks = c;
  *list_shift = shift;
  return true;
}

bool estimates_apply(const IndexerParams &p) {
  int chunk, n, shift;
  return p.T <= 65535 && (p.S <= kTopkThreads * kMaxRegEpt || chunk_plan(p, &chunk, &n, &shift));
}

// Few tokens: the estimate kernel is bound by latency and prepares K on its way
// (a launch less: 3 tokens, 2500 positions, 32 heads 20.6 -> 16.1 us); from 9
// tokens on several workgroups would prepare the same blocks.  With more than
// one pair of tokens the waves of a workgroup already do, and a kernel that holds
// the operands of many heads beside its preparation runs one wave per SIMD: where
// that costs more than a launch, long rows are prepared first.  8 tokens of 64 heads over
// 32768 positions: paged 40.5 -> 32.4 us, flat 35.5 -> 32.4; over 131071: 95.9 ->
// 65.6, 79.7 -> 66.1; 4 tokens, paged, 32768: 35.1 -> 31.5.  Kept: flat, 2 tokens of
// 64 heads over 131071 52 us against 58, 8 of 48 heads over 32768 29.6 against
// 31.4; paged, 4 tokens of 32 heads over 65536 44.4 against 46.5.
bool estimates_prepare_k(const IndexerParams &p) {
  if (p.T > kEstFusedTokens) return false;
  const int pairs = (p.T + 1) / 2;
  const int64_t work = (int64_t)pairs * p.S;
  if (p.k_cache != nullptr) return p.Hi > 32 ? work <= 32768 : pairs <= 2 || work <= 65536;
  return p.Hi <= 48 || pairs <= 2 || work <= 65536;
}

hipError_t launch_estimates(const IndexerParams &pin, hipStream_t stream) {
  IndexerParams p = pin;
  const int nkb = (p.S + 15) / 16, pairs = (p.T + 1) / 2;
  p.est_pairs = pairs >= 3 ? 4 : pairs;
  const int gy = (pairs + p.est_pairs - 1) / p.est_pairs;
  // Workgroups per token group: as many as take the fewest block times over the
  // rounds of workgroups (two per CU; a wave's start costs about as much as 12
  // blocks of its own).
  const int ranges = kEstWaves / p.est_pairs;  // per workgroup
  int best = 1;
  int64_t best_cost = INT64_MAX;
  for (int gx = 1; gx <= std::min((nkb + 2 * ranges - 1) / (2 * ranges), 1024); ++gx) {
    const int64_t rounds = ((int64_t)gx * gy * kEstWaves + kNumCU * kEstWavesPerCU - 1) /
                           (kNumCU * kEstWavesPerCU);
    const int64_t cost = rounds * ((nkb + gx * ranges - 1) / (gx * ranges) + 12);
    if (cost < best_cost) {
      best_cost = cost;
      best = gx;
    }
  }
  p.est_blocks = ((nkb + best * ranges - 1) / (best * ranges) + 1) / 2 * 2;
  const dim3 grid((nkb + p.est_blocks * ranges - 1) / (p.est_blocks * ranges), gy);
  switch (p.Hi / 16) {
    case 1: return launch_estimate<1>(p, grid, stream);
    case 2: return launch_estimate<2>(p, grid, stream);
    case 3: return launch_estimate<3>(p, grid, stream);
    default: return launch_estimate<4>(p, grid, stream);
  }
}

static hipError_t launch_topk_chunks(const IndexerParams &pin, hipStream_t stream) {
  IndexerParams p = pin;
  if (!chunk_plan(p, &p.chunk, &p.n_chunks, &p.list_shift)) return hipErrorInvalidValue;
  p.list_len = 1 << p.list_shift;
  const dim3 block(kTopkThreads), grid(p.n_chunks, p.T);
  hipLaunchKernelGGL(dsa_idx_topk_chunk_kernel<kMaxRegEpt>, grid, block, 0, stream, p);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const int places = p.n_chunks << p.list_shift;
  if (places <= kTopkThreads * 8) hipLaunchKernelGGL(dsa_idx_topk_merge_kernel<8>, dim3(p.T), block, 0, stream, p);
  else if (places <= kTopkThreads * 16) hipLaunchKernelGGL(dsa_idx_topk_merge_kernel<16>, dim3(p.T), block, 0, stream, p);
  else hipLaunchKernelGGL(dsa_idx_topk_merge_kernel<kMaxRegEpt>, dim3(p.T), block, 0, stream, p);
  return hipGetLastError();
}

hipError_t launch_topk(const IndexerParams &p, hipStream_t stream) {
  if (p.S <= kTopkThreads * 8) return launch_topk_regs<8>(p, stream);
  if (p.S <= kTopkThreads * 16) return launch_topk_regs<16>(p, stream);
  if (p.S <= kTopkThreads * kMaxRegEpt) return launch_topk_regs<kMaxRegEpt>(p, stream);
  if (p.estimated) return launch_topk_chunks(p, stream);
  hipLaunchKernelGGL(dsa_idx_topk_stream_kernel, dim3(p.T), dim3(kTopkThreads), 0, stream, p);
  return hipGetLastError();
}

}  // namespace dsa
