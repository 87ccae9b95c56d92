// dsa_indexer.hip -- lightning-indexer scores and per-row top-k for gfx950.
//
// Score (the structure of the reference's indexer_kernel,
// solution/triton/indexer_kernel.py:185-275: dequantise -> dot -> ReLU ->
// head weight -> sum over heads; BASELINE config 5 form):
//
//   score[t,s] = sum_h w[t,h] * relu(q[t,h,:] . k[s,:] * k_scale[s])
//
// computed in the factored form k_scale[s] * sum_h w[t,h] * relu(d[t,s,h])
// (equal for a positive quantisation scale) with one exact rounding order, so
// the GPU reproduces the CPU oracle bit for bit:
//   D_h = d * 2^18, the exact integer dot of the values times 2^9;
//   r_h = fl32(max(D_h, 0));
//   the heads form 4 groups of Hi/4 consecutive heads; group g sums
//   G_g = fma(w_h, r_h, G_g) over its heads in ascending order from 0;
//   total = fl32(fl32(G_0 + G_1) + fl32(G_2 + G_3));
//   score = fl32(total * c_s), c_s = fl32(k_scale[s] * 2^-18).
// Positions beyond causal_limit[t] score -inf and are never selected.
//
// Exact dot on int8 MFMA.  Every finite e4m3fn value times 2^9 is an integer
// x with |x| <= 229376 (18 bits); x = p0 + 2^7 p1 + 2^14 p2 with signed 7-bit
// pieces (sign-magnitude split), so
//   D = sum_{a,b} 2^(7(a+b)) sum_j pq_a[j] pk_b[j]
// where each inner 128-term sum (|.| <= 128*127*127) is exact in the int32
// accumulator of v_mfma_i32_16x16x64_i8.  When every |x| < 2^14 (values below
// 32) the third piece is zero and D = P00 + 2^7 X + 2^14 P11 (X the two cross
// products) is combined in int32 when the operand maxima bound |D| below
// 2^31, else in fp64.  Where a whole range of positions allows the int32
// combine, three products suffice: the pieces lie in [0, 127] with the
// value's sign, so q1 - q0 and k0 - k1 fit int8 and C3 = P00 + (q1 - q0).(k0
// - k1) = X - P11 gives D = ((C3 + 129 P11) << 7) + P00.  Larger values take
// nine products and an fp64 combine (exact: every partial sum stays below
// 2^50).  e4m3fn NaN codes (0x7f, 0xff) count as zero.
//
// Kernels (the selection, and the score estimates most selections run from,
// are in dsa_select.hip):
//   dsa_idx_prep_kernel    k codes -> piece planes laid out as MFMA
//                          operands in lane order (one 1 KB chunk per 16
//                          positions, piece and 64-wide k-step) beside the
//                          codes themselves, the largest |x| and |c_s| |k_s|
//                          of every 16-position block, and c_s of every
//                          position (kept by the caller as prepared K
//                          planes, or in the call's workspace; without the
//                          planes for a selection from estimates).  With a
//                          paged K cache it reads each position's codes and
//                          scale through the page map.
//   dsa_idx_score_kernel   every exact score, for calls that return them: two
//                          waves per query token, up to 4 tokens per
//                          workgroup sharing a range of positions.  The
//                          token's q pieces are derived from its codes in
//                          registers (A operands, heads as M, through a code
//                          -> pieces table in LDS); each 16-position block's k pieces are
//                          one coalesced 1 KB load per operand (B, positions
//                          as N).  When every block of the range takes the
//                          three-product int32 path, the token's two waves
//                          claim chunks of six blocks from a counter in LDS
//                          and the loop is software-pipelined: a head block's
//                          MFMAs are issued beside the epilogue of the head
//                          block two before it.
//   dsa_k_append_kernel    quantise-on-append into the paged fp8 K cache:
//                          one wave per token (per-token fp32 scale from the
//                          row's largest magnitude, e4m3 round to nearest
//                          even).
#include <algorithm>

#include "../../include/dsa_abi.h"
#include "dsa_indexer_device.h"

namespace dsa {
namespace {

constexpr int kPrepThreads = 256;         // four waves, one destination block each
constexpr int kScoreWaves = 8;            // waves per score workgroup (two per token)
constexpr int kTargetScoreWaves = 2048;   // two waves per SIMD on 256 CUs
constexpr int kMinBlocksPerWave = 8;

// K blocks k_block0 .. k_block0 + k_blocks - 1 (16 positions each): c_s of
// every position, the k_max word of every block (largest |x| and, but for
// kPrepDiff, largest |c_s| * |k_s|) and, by WHAT, the codes row by row without
// NaN codes and the piece planes laid out as MFMA B operands in lane order (one
// 1 KB chunk per plane and 64-wide k-step): planes p0 and p1, then (kPrepDiff) a plane of p2 if
// the block holds a value of magnitude >= 32, else of p0 - p1.  One wave per
// block; lane l = 16*g + c holds position 16*block + c at dims 64*ks + 16*g for
// k-steps ks = 0, 1, so every plane store of the wave is one contiguous 1 KB
// chunk.  Positions at or past S read as zeros.
template <int WHAT>
__global__ __launch_bounds__(kPrepThreads) void dsa_idx_prep_kernel(IndexerParams p) {
  __shared__ uint32_t lut[256];
  if constexpr (WHAT != kPrepCodes) {
    lut[threadIdx.x] = piece_word(threadIdx.x);
    __syncthreads();
  }
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wblk = blockIdx.x * (kPrepThreads / 64) + wave;
  if (wblk >= p.k_blocks) return;
  const int blk = p.k_block0 + wblk;

  uint4 raw[2] = {make_uint4(0, 0, 0, 0), make_uint4(0, 0, 0, 0)};
  float cs = 0.f;
  const int s = blk * 16 + c;
  if (s < p.S) {
    if (p.k_cache != nullptr) {  // paged: codes and scale through the page map
      const int pg = p.k_pages[s / p.k_page_size], off = s % p.k_page_size;
      if ((uint32_t)pg < (uint32_t)p.k_num_pages) {  // else a zero row of scale 0
        const uint8_t *page = p.k_cache + (int64_t)pg * p.k_page_size * kKTokenBytes;
        raw[0] = *(const uint4 *)(page + off * kIdxDim + g * 16);
        raw[1] = *(const uint4 *)(page + off * kIdxDim + 64 + g * 16);
        cs = *(const float *)(page + p.k_page_size * kIdxDim + off * 4) * 0x1p-18f;
      }
    } else {
      const uint8_t *row = p.k + (int64_t)s * kIdxDim;
      raw[0] = *(const uint4 *)(row + g * 16);
      raw[1] = *(const uint4 *)(row + 64 + g * 16);
      cs = p.k_scale[s] * 0x1p-18f;
    }
    if (g == 0) p.k_cs[s] = cs;
  }
  const uint32_t w[8] = {raw[0].x, raw[0].y, raw[0].z, raw[0].w, raw[1].x, raw[1].y, raw[1].z, raw[1].w};
  const int bmax = magnitude_bound(wave_top_code(w));
  uint32_t v[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = drop_nan(w[i]);
  uint32_t nb = 0;
  if constexpr (WHAT != kPrepDiff) {  // (exact scores need no norms)
    float n2 = 0.f;
#pragma unroll
    for (int i = 0; i < 8; i += 2) n2 += sum_squares8(v[i], v[i + 1]);
    n2 = sum_lane_groups(n2);  // the position's four lanes
    nb = wave_max_last(position_norm_bits(cs, n2));
  }
  if (lane == 63) p.k_max[blk] = (int32_t)((uint32_t)bmax | (nb << kMaxXBits));

  // non-temporal stores: the planes are read by the next kernel, and stores
  // kept in L2 cost a write-back at the kernel's end (measured: 1.6 us of 10.8)
  if constexpr (WHAT != kPrepDiff) {
    // lanes c and c ^ 8 of a row of 16 exchange halves, so that a store covers
    // eight whole rows (1 KB) and not one half of sixteen: planes of 524288
    // positions 46.3 -> 42.7 us
    const bool low = c < 8;
    uint8_t *codes = p.k_codes + (int64_t)blk * p.k_code_stride + (c & 7) * kIdxDim + (low ? 0 : 64) + g * 16;
    u32x4 top, bottom;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const uint32_t other = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(low ? v[4 + d] : v[d]), 0x128,  // row_ror:8
                                                                     0xf, 0xf, false);
      top[d] = low ? v[d] : other;
      bottom[d] = low ? other : v[4 + d];
    }
    __builtin_nontemporal_store(top, (u32x4 *)codes);
    __builtin_nontemporal_store(bottom, (u32x4 *)(codes + 8 * kIdxDim));
  }
  if constexpr (WHAT != kPrepCodes) {
    uint32_t pw[32];
#pragma unroll
    for (int i = 0; i < 32; ++i) pw[i] = lut[(w[i >> 2] >> (8 * (i & 3))) & 0xffu];
    int8_t *dst = p.k_pieces + (int64_t)blk * kBlockBytes + lane * 16;
    const int bytes[3] = {0, 1, bmax < kTwoPieceLimit ? 3 : 2};
#pragma unroll
    for (int slot = 0; slot < (WHAT == kPrepDiff ? 3 : 2); ++slot) {
      i32x4 o[2];
      pack_plane(pw, bytes[slot], false, o);
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
        __builtin_nontemporal_store(__builtin_bit_cast(u32x4, o[ks]),
                                    (u32x4 *)(dst + (slot * 2 + ks) * kChunk));
    }
  }
}

// The A operands of token t's head block hb, derived in registers from the
// raw codes: lane l = 16*g + c holds MFMA row c, which stands for head
// (c / 4) * Hi/4 + 4*hb + c % 4 (so the four output rows a lane receives,
// rows 4g..4g+3, are consecutive heads of head group g), dims 64*ks + 16*g ..
// +15 for k-steps ks = 0, 1.  Planes NPL of them, by LUT byte (4: p1 - p0).
template <int NPL>
__device__ __forceinline__ void q_operands(const IndexerParams &p, const uint32_t *lut, int t, int hb,
                                           const int (&plane)[NPL], i32x4 (&out)[NPL][2]) {
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int head = (c >> 2) * (p.Hi >> 2) + 4 * hb + (c & 3);
  const uint8_t *row = p.q + ((int64_t)t * p.Hi + head) * kIdxDim;
  const uint4 r0 = *(const uint4 *)(row + g * 16), r1 = *(const uint4 *)(row + 64 + g * 16);
  const uint32_t w[8] = {r0.x, r0.y, r0.z, r0.w, r1.x, r1.y, r1.z, r1.w};
  uint32_t v[32];
#pragma unroll
  for (int i = 0; i < 32; ++i) v[i] = lut[(w[i >> 2] >> (8 * (i & 3))) & 0xffu];
#pragma unroll
  for (int k = 0; k < NPL; ++k) pack_plane(v, plane[k] == 4 ? 3 : plane[k], plane[k] == 4, out[k]);
}

// Largest |x| over every code of token t (all heads), the same in every lane.
__device__ __forceinline__ int q_magnitude_bound(const IndexerParams &p, int t) {
  const int lane = threadIdx.x & 63;
  const uint4 *src = (const uint4 *)(p.q + (int64_t)t * p.Hi * kIdxDim);
  const int n16 = p.Hi * kIdxDim / 16;  // 16-byte pieces of the token's codes
  uint32_t mc = 0;
  for (int i = lane; i < n16; i += 64) {
    const uint4 r = src[i];
    const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
    for (int j = 0; j < 16; ++j) mc = max(mc, (w[j >> 2] >> (8 * (j & 3))) & 0x7fu);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mc = max(mc, (uint32_t)__shfl_xor((int)mc, o));
  return magnitude_bound(__builtin_amdgcn_readfirstlane(mc));
}

// ---- scores --------------------------------------------------------------

// Scores of token t over the 16-position blocks [b0, b1).  NQP = pieces of
// q in play (3 when the token holds a value of magnitude >= 32).
template <int NHB, int NQP, bool DIFF>
__device__ __forceinline__ void score_range(const IndexerParams &p, const uint32_t *lut, int t, int b0,
                                            int b1, int qmax) {
  // The rounding order is part of the score's definition: no contraction of
  // the products and sums written below into fused multiply-adds (the one
  // fused step of the definition is the explicit fmaf).
#pragma clang fp contract(off)
  const int lane = threadIdx.x & 63;
  const int col = lane & 15, g = lane >> 4;
  const int lim = p.limit[t];
  float *srow = p.scores + (int64_t)t * p.S;
  uint32_t sh7;
  asm volatile("s_mov_b32 %0, 7" : "=s"(sh7));

  // A operands of this token: [head block][piece][k-step]
  i32x4 qa[NHB][NQP][2];
  {
    int planes[NQP];
#pragma unroll
    for (int pc = 0; pc < NQP; ++pc) planes[pc] = pc;
#pragma unroll
    for (int hb = 0; hb < NHB; ++hb) q_operands<NQP>(p, lut, t, hb, planes, qa[hb]);
  }
  // weights of the lane's rows: heads g*Hi/4 + 4*hb + i
  float wl[NHB][4];
  const float *wsrc = p.w + (int64_t)t * p.Hi + g * (p.Hi >> 2);
#pragma unroll
  for (int hb = 0; hb < NHB; ++hb)
#pragma unroll
    for (int i = 0; i < 4; ++i) wl[hb][i] = wsrc[4 * hb + i];

  // Blocks are fetched two ahead: pieces 0 and 1, the lane's scale, the
  // block's magnitude bound.  Indices past the range are clamped so every
  // step issues the same loads.
  struct KBlock {
    i32x4 k[2][2];
    float cs;
    int kmax;
  };
  auto fetch = [&](int b, KBlock &kb) {
    b = min(b, b1 - 1);
    const int8_t *src = p.k_pieces + (int64_t)b * kBlockBytes + lane * 16;
#pragma unroll
    for (int pc = 0; pc < 2; ++pc)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) kb.k[pc][ks] = load_chunk(src + (pc * 2 + ks) * kChunk);
    kb.cs = p.k_cs[min(b * 16 + col, p.S - 1)];
    kb.kmax = block_max_x(p.k_max[b]);
  };

  // the lane's group sum for its position -> the score, stored by lanes 0..15
  auto finish = [&](float G, float cs, int s) {
    const float total = sum_lane_groups(G);
    const float score = total * cs;
    if (g == 0 && s >= 0 && s < p.S) srow[s] = (s > lim) ? -INFINITY : score;
  };
  // int32 combine of one head block's products into the lane's group sum:
  // D = ((P11 * 2^7 + X) * 2^7) + P00, two v_lshl_add_u32.  The shift amount
  // is an opaque scalar so that the compiler keeps this nesting instead of
  // redistributing the shifts into two shifts and an add3.
  auto epilogue = [&](const i32x4 &P00, const i32x4 &X, const i32x4 &P11, int hb, float &G) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t hi = ((uint32_t)P11[i] << sh7) + (uint32_t)X[i];
      const int D = (int)((hi << sh7) + (uint32_t)P00[i]);
      G = __builtin_fmaf(wl[hb][i], (float)max(D, 0), G);
    }
  };
  auto two_piece = [&](const i32x4 (&kc)[2][2], int hb, i32x4 &P00, i32x4 &X, i32x4 &P11) {
    const i32x4 z = {0, 0, 0, 0};
    P00 = mfma(qa[hb][0][1], kc[0][1], mfma(qa[hb][0][0], kc[0][0], z));
    X = mfma(qa[hb][0][0], kc[1][0], z);
    X = mfma(qa[hb][0][1], kc[1][1], X);
    X = mfma(qa[hb][1][0], kc[0][0], X);
    X = mfma(qa[hb][1][1], kc[0][1], X);
    P11 = mfma(qa[hb][1][1], kc[1][1], mfma(qa[hb][1][0], kc[1][0], z));
  };

  // The general cases: the piece products of like powers of two are added in
  // int32 (every sum stays below 2^30), the two halves in fp64 (exact for
  // every |D| < 2^53).
  auto general = [&](const KBlock &kc, int b, int s, bool two) {
    float G = 0.f;
    if (NQP == 2 && two) {
#pragma unroll
      for (int hb = 0; hb < NHB; ++hb) {
        i32x4 P00, X, P11;
        two_piece(kc.k, hb, P00, X, P11);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          G = __builtin_fmaf(wl[hb][i], relu_dot(P00[i] + (X[i] << 7), P11[i]), G);
      }
    } else {
      // all piece products, grouped by the power 2^(7(a+c)) they carry; the
      // third pieces come from their plane or the block's codes
      i32x4 kb3[3][2];
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        kb3[0][ks] = kc.k[0][ks];
        kb3[1][ks] = kc.k[1][ks];
        kb3[2][ks] = i32x4{0, 0, 0, 0};
      }
      if (!two) {
        if constexpr (DIFF) {
          const int8_t *plane = p.k_pieces + (int64_t)b * kBlockBytes + 4 * kChunk + lane * 16;
#pragma unroll
          for (int ks = 0; ks < 2; ++ks) kb3[2][ks] = load_chunk(plane + ks * kChunk);
        } else {
          third_pieces(lut, p.k_codes + (int64_t)b * p.k_code_stride + col * kIdxDim + g * 16, kb3[2]);
        }
      }
#pragma unroll
      for (int hb = 0; hb < NHB; ++hb) {
        i32x4 C[5];
#pragma unroll
        for (int d = 0; d < 5; ++d) C[d] = i32x4{0, 0, 0, 0};
#pragma unroll
        for (int a = 0; a < NQP; ++a)
#pragma unroll
          for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) C[a + c] = mfma(qa[hb][a][ks], kb3[c][ks], C[a + c]);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          G = __builtin_fmaf(wl[hb][i], relu_dot(C[0][i] + (C[1][i] << 7),
                                                 C[2][i] + (C[3][i] << 7) + (C[4][i] << 14)), G);
      }
    }
    finish(G, kc.cs, s);
  };

  KBlock ka, kb, kc3;
  fetch(b0, ka);
  fetch(b0 + 1, kb);

  // One block: prefetch block b+2 into `ahead`, then score block b from `kc`.
  // Returns false once the rest of the range is causally masked.  The loop
  // below is unrolled by three so that the three buffers keep fixed roles
  // (a rotation by copies would wait for the loads just issued).
  auto step = [&](int b, const KBlock &kc, KBlock &ahead) -> bool {
    fetch(b + 2, ahead);  // unconditional: `ahead` then needs no merge of two versions
    if (b * 16 > lim) {   // every later position is masked as well
      for (int bb = b; bb < b1; ++bb) {
        const int s = bb * 16 + col;
        if (g == 0 && s < p.S) srow[s] = -INFINITY;
      }
      return false;
    }
    const int s = b * 16 + col;
    const bool two = kc.kmax < kTwoPieceLimit;
    const bool fits = (int64_t)qmax * kc.kmax * kIdxDim < (1LL << 31);
    if constexpr (NQP == 2) {
      if (two && fits) {
        i32x4 P00[NHB], X[NHB], P11[NHB];
        float G = 0.f;
#pragma unroll
        for (int hb = 0; hb < NHB; ++hb) two_piece(kc.k, hb, P00[hb], X[hb], P11[hb]);
#pragma unroll
        for (int hb = 0; hb < NHB; ++hb) epilogue(P00[hb], X[hb], P11[hb], hb, G);
        finish(G, kc.cs, s);
        return true;
      }
    }
    general(kc, b, s, two);
    return true;
  };
  for (int b = b0; b < b1; b += 3) {
    if (!step(b, ka, kc3) || b + 1 >= b1) break;
    if (!step(b + 1, kb, ka) || b + 2 >= b1) break;
    if (!step(b + 2, kc3, kb)) break;
  }
}

// a - b of four bytes at a time, two 16-bit halves at once: the low bytes from
// the plain differences, the high bytes from those with b's low bytes taken
// out, which borrow nothing (four instructions).
__device__ __forceinline__ uint32_t sub_bytes(uint32_t a, uint32_t b) {
  typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
  constexpr uint32_t kLow = 0x00ff00ffu;
  const u16x2 x = __builtin_bit_cast(u16x2, a);
  const uint32_t lo = __builtin_bit_cast(uint32_t, (u16x2)(x - __builtin_bit_cast(u16x2, b)));
  const uint32_t hi = __builtin_bit_cast(uint32_t, (u16x2)(x - __builtin_bit_cast(u16x2, b & ~kLow)));
  return (lo & kLow) | (hi & ~kLow);
}

// Instruction groups for the scheduler (__builtin_amdgcn_sched_group_barrier
// masks: 0x002 VALU, 0x008 MFMA, 0x020 vector memory read, 0x040 write): NM
// MFMAs, each followed by NV VALU instructions.
template <int NM, int NV>
__device__ __forceinline__ void mfma_valu_groups() {
#pragma unroll
  for (int i = 0; i < NM; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x002, NV, 0);
  }
}

// Scores of token t over the blocks [b0, b1) when every block of the range
// takes the two-piece int32 path, for NHB >= 2: the same exact D and the same
// rounding order as score_range, from three piece products instead of four.
//
// With the pieces of every value below 2^14 in [0, 127] and of one sign,
// (q1 - q0) and (k0 - k1) fit int8.  DIFF: the k difference is a plane of its
// own; prepared planes hold the codes in its place, and it is taken four bytes
// at a time from the loaded planes, a block ahead of its use: eight VALU
// instructions a head block beside 18 (64 rows of 32768 positions with the top-k
// 65.0 us, 61.9 if the planes held the difference; 66.0 with six-instruction
// differences).
// With P00 = q0.k0, P11 = q1.k1 and the cross term X = q0.k1 + q1.k0,
// (q1 - q0).(k0 - k1) = X - P00 - P11, so the chain
//   C3 = P00 + (q1 - q0).(k0 - k1) = X - P11
// gives D = P00 + 2^7 X + 2^14 P11 = ((C3 + 129 P11) << 7) + P00:
// six MFMAs per head block (C3's chain starts from P00's result) and two
// integer instructions per element (v_mad_i32_i24: |P11| < 2^23; the
// arithmetic is modulo 2^32 and D itself fits int32).  The int8 MFMA path
// is bound by the chip's power limit, not by issue: fewer MFMAs are faster.
//
// Two waves share the token's range (the two waves of one SIMD: one of
// them is issued first, and with fixed halves it would finish long before
// the other, which then runs alone): each claims chunks of six blocks from
// the pair's counter in LDS (`claim`, counting blocks from b0), one chunk
// ahead, until the range is used up.  Claims only grow, so every wave ends.
//
// Software-pipelined over the wave's sequence of head blocks j: the six
// MFMAs of head block j are issued between the epilogue instructions of head
// block j - 2, whose accumulators are complete by then; the pipeline runs
// on across chunk boundaries.  A chunk holds six blocks, so the three
// accumulator sets (j mod 3), the three operand buffers (fetched two blocks
// ahead), the group sums G[slot mod 2] and the pair scales, indexed by a
// block's slot in its chunk, all have static indices.  A pair of blocks
// shares one reduction over the four lane groups (a permlane16 swap of the
// two blocks' sums, a permlane32 swap, two adds: lane groups 0 and 1 end
// with blocks q and q + 1), one scale load and one store.
//
// Loads and stores go through buffer descriptors with scalar block offsets;
// scale loads and score stores carry the position in the per-lane offset,
// which the descriptor's bound checks (positions past S read 0 and are not
// stored; an offset of 2^31 is past every bound).  No per-block bound is
// loaded: a wave-uniform loaded value is moved to a scalar register right
// after its load, a wait that would tie each prefetch to its own step.
template <int NHB, bool DIFF>
__device__ __forceinline__ void score_range_fast(const IndexerParams &p, const uint32_t *lut, int t,
                                                 int b0, int b1, int *claim, bool lead) {
#pragma clang fp contract(off)
  static_assert(NHB >= 2, "the epilogue runs two head blocks behind");
  const int lane = threadIdx.x & 63;
  const int col = lane & 15, g = lane >> 4;
  const int lim = p.limit[t];
  const int nkb = (p.S + 15) >> 4;
  const auto krs = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t *>(p.k_pieces), 0,
                                                     nkb * kBlockBytes, kBufferFlags);
  const auto srs = __builtin_amdgcn_make_buffer_rsrc(p.k_cs, 0, p.S * 4, kBufferFlags);
  const auto ors = __builtin_amdgcn_make_buffer_rsrc(p.scores + (int64_t)t * p.S, 0, p.S * 4,
                                                     kBufferFlags);
  constexpr uint32_t kDropped = 0x80000000u;  // S * 4 < 2^31
  const uint32_t pair4 = (uint32_t)((g & 1) * 16 + col) * 4;  // lane's position in a pair, bytes
  uint32_t sh7;
  asm volatile("s_mov_b32 %0, 7" : "=s"(sh7));

  // blocks [b0, bend) hold a position at or below the causal limit; every
  // position of the blocks before bend - 1 is below it
  const int bend = min(b1, max(b0, (lim >> 4) + 1));
  if (lead)
    for (int b = bend; b < b1; ++b)
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(-INFINITY), ors,
                                            g == 0 ? col * 4 + b * 64 : kDropped, 0, 0);
  // first block of the next chunk of six the pair has not claimed yet
  auto claim_chunk = [&]() {
    int c = 0;
    if (lane == 0) c = atomicAdd(claim, 6);
    return b0 + __builtin_amdgcn_readfirstlane(c);
  };
  int B = claim_chunk();  // the current chunk
  if (B >= bend) return;
  int N = claim_chunk();  // the next one

  // A operands [hb][q0, q1, q1 - q0][k-step]
  i32x4 qa[NHB][3][2];
  {
    const int planes[3] = {0, 1, 4};
#pragma unroll
    for (int hb = 0; hb < NHB; ++hb) q_operands<3>(p, lut, t, hb, planes, qa[hb]);
  }
  float wl[NHB][4];
  const float *wsrc = p.w + (int64_t)t * p.Hi + g * (p.Hi >> 2);
#pragma unroll
  for (int hb = 0; hb < NHB; ++hb)
#pragma unroll
    for (int i = 0; i < 4; ++i) wl[hb][i] = wsrc[4 * hb + i];

  // B operands [k0, k1, k0 - k1][k-step] of a block
  i32x4 kbuf[3][3][2];
  auto fetch_k = [&](int b, i32x4 (&k)[3][2]) {
    b = min(b, bend - 1);
#pragma unroll
    for (int pl = 0; pl < (DIFF ? 3 : 2); ++pl)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
        k[pl][ks] = __builtin_bit_cast(
            i32x4, __builtin_amdgcn_raw_buffer_load_b128(krs, lane * 16,
                                                         b * kBlockBytes + (pl * 2 + ks) * kChunk, 0));
  };
  // k0 - k1 of dwords [d0, d1) of the block's eight
  auto derive_k = [&](i32x4 (&k)[3][2], int d0, int d1) {
    if constexpr (DIFF) return;
#pragma unroll
    for (int d = 0; d < 8; ++d)
      if (d >= d0 && d < d1)
        k[2][d >> 2][d & 3] = (int)sub_bytes((uint32_t)k[0][d >> 2][d & 3], (uint32_t)k[1][d >> 2][d & 3]);
  };
  // c_s of the pair starting at block q: lane groups g and g ^ 2 hold block q + (g & 1)
  auto fetch_cs = [&](int q) {
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(srs, pair4 + q * 64, 0, 0));
  };
  struct Acc {
    i32x4 P00, C3, P11;
  };
  Acc acc[3];
  auto mm = [&](const i32x4 (&k)[3][2], int hb, Acc &a) {
    const i32x4 z = {0, 0, 0, 0};
    a.P00 = mfma(qa[hb][0][1], k[0][1], mfma(qa[hb][0][0], k[0][0], z));
    a.P11 = mfma(qa[hb][1][1], k[1][1], mfma(qa[hb][1][0], k[1][0], z));
    a.C3 = mfma(qa[hb][2][1], k[2][1], mfma(qa[hb][2][0], k[2][0], a.P00));
  };
  // D = ((C3 + 129 P11) << 7) + P00, then the ReLU, the conversion and the
  // head's fused multiply-add into the group sum
  auto epi = [&](const Acc &a, int hb, float &G) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t hi = (uint32_t)__mul24(a.P11[i], 129) + (uint32_t)a.C3[i];
      const int D = (int)((hi << sh7) + (uint32_t)a.P00[i]);
      G = __builtin_fmaf(wl[hb][i], (float)max(D, 0), G);
    }
  };
  float G[2] = {0.f, 0.f};  // the lane's group sums of the current pair's blocks
  // the pair starting at block q: (G0 + G1) + (G2 + G3) of both blocks, times
  // c_s, stored by lane groups 0 and 1; `last` masks the positions past the
  // causal limit and a second block at or past bend
  auto store_pair = [&](int q, float cs, bool last) {
    auto x = __builtin_amdgcn_permlane16_swap(__float_as_uint(G[0]), __float_as_uint(G[1]), false, false);
    const float a = __uint_as_float(x[0]) + __uint_as_float(x[1]);  // rows: G0+G1 | G2+G3 of q, q+1
    auto y = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(a), false, false);
    const float total = __uint_as_float(y[0]) + __uint_as_float(y[1]);  // block q + (g & 1)
    float v = total * cs;
    const int blk = q + (g & 1);
    uint32_t off = g < 2 ? pair4 + q * 64 : kDropped;
    if (last) {
      if (blk * 16 + col > lim) v = -INFINITY;
      if (blk >= bend) off = kDropped;
    }
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), ors, off, 0, 0);
  };

  float cs_pair[3];  // scales of the pairs starting at slots 0, 2, 4
  fetch_k(B, kbuf[0]);
  fetch_k(B + 1, kbuf[1]);
  fetch_k(B + 2, kbuf[2]);
  cs_pair[0] = fetch_cs(B);
  derive_k(kbuf[0], 0, 8);
  derive_k(kbuf[1], 0, 8);
  {  // block B (slot 0; the stages fetch two blocks ahead)
    float Gc = 0.f;
#pragma unroll
    for (int hb = 0; hb < NHB; ++hb) {
      if (hb >= 2) epi(acc[(hb - 2) % 3], hb - 2, Gc);
      mm(kbuf[0], hb, acc[hb % 3]);
    }
    G[0] = Gc;
  }
  // block b in slot SLOT of its chunk: fetch the block two ahead (`ahead`:
  // past the chunk, in the next one), finish the previous block (and, for an
  // even SLOT, store the pair before it, which starts at `pair`), issue block
  // b's MFMAs
  auto stage = [&](int b, auto slot_c, int ahead, int pair) {
    constexpr int SLOT = decltype(slot_c)::value;
    constexpr bool kEven = (SLOT & 1) == 0;
    fetch_k(ahead, kbuf[(SLOT + 2) % 3]);
    if constexpr (kEven) {
      cs_pair[SLOT / 2] = fetch_cs(b);
      __builtin_amdgcn_sched_group_barrier(0x020, DIFF ? 7 : 5, 0);
    } else {
      __builtin_amdgcn_sched_group_barrier(0x020, DIFF ? 6 : 4, 0);
    }
    float Gc = 0.f;
#pragma unroll
    for (int hb = 0; hb < NHB; ++hb) {
      const int j = SLOT * NHB + hb;
      if (hb < 2) {
        epi(acc[(j + 1) % 3], hb + NHB - 2, G[(SLOT + 1) & 1]);
        if (kEven && hb == 1) store_pair(pair, cs_pair[(SLOT / 2 + 2) % 3], false);
      } else {
        epi(acc[(j + 1) % 3], hb - 2, Gc);
      }
      // the next block's difference plane (its loads were issued a stage ago)
      derive_k(kbuf[(SLOT + 1) % 3], 8 * hb / NHB, 8 * (hb + 1) / NHB);
      mm(kbuf[SLOT % 3], hb, acc[j % 3]);
      if (kEven && hb == 1) {
        mfma_valu_groups<6, DIFF ? 4 : 6>();
        __builtin_amdgcn_sched_group_barrier(0x040, 1, 0);
      } else {
        mfma_valu_groups<6, DIFF ? 3 : 5>();
      }
      // the pipeline above pairs each head block's MFMAs with finished
      // accumulators: nothing moves between head blocks (an MFMA moved
      // earlier would wait for operands loaded in the same iteration)
      __builtin_amdgcn_sched_barrier(0);
    }
    G[SLOT & 1] = Gc;
  };
  // after the wave's last block (slot SLOT of its chunk): its last two head
  // blocks, then its pair
  auto drain = [&](auto slot_c, int last) {
    constexpr int SLOT = decltype(slot_c)::value;
    constexpr int j = SLOT * NHB + NHB - 1;
    epi(acc[(j + 2) % 3], NHB - 2, G[SLOT & 1]);
    epi(acc[j % 3], NHB - 1, G[SLOT & 1]);
    store_pair(last - (SLOT & 1), cs_pair[SLOT / 2], true);
  };
  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, 1>;
  using S2 = std::integral_constant<int, 2>;
  using S3 = std::integral_constant<int, 3>;
  using S4 = std::integral_constant<int, 4>;
  using S5 = std::integral_constant<int, 5>;
  // blocks 1 .. 5 of a full chunk B, then block 0 of the next chunk N
  while (B + 6 <= bend && N < bend) {
    const int N2 = claim_chunk();
    stage(B + 1, S1{}, B + 3, 0);
    stage(B + 2, S2{}, B + 4, B);
    stage(B + 3, S3{}, B + 5, 0);
    stage(B + 4, S4{}, N, B + 2);
    stage(B + 5, S5{}, N + 1, 0);
    stage(N, S0{}, N + 2, B + 4);
    B = N;
    N = N2;
  }
  // the wave's last chunk: blocks 1 .. rest (the operand fetches past it are
  // clamped to bend - 1 and unused)
  const int rest = min(bend, B + 6) - 1 - B;
  if (rest > 0) stage(B + 1, S1{}, B + 3, 0);
  if (rest > 1) stage(B + 2, S2{}, B + 4, B);
  if (rest > 2) stage(B + 3, S3{}, B + 5, 0);
  if (rest > 3) stage(B + 4, S4{}, B + 6, B + 2);
  if (rest > 4) stage(B + 5, S5{}, B + 7, 0);
  switch (rest) {
    case 0: drain(S0{}, B); break;
    case 1: drain(S1{}, B + 1); break;
    case 2: drain(S2{}, B + 2); break;
    case 3: drain(S3{}, B + 3); break;
    case 4: drain(S4{}, B + 4); break;
    default: drain(S5{}, B + 5); break;
  }
}

template <int NHB, bool DIFF>
__global__ __launch_bounds__(kScoreWaves * 64) void dsa_idx_score_kernel(IndexerParams p) {
  // two waves per token: slot = the token's place in the workgroup, member
  // 0 or 1 (waves w and w + tpw, which the hardware places on one SIMD)
  __shared__ int claim[kScoreWaves / 2];
  __shared__ uint32_t lut[256];  // code -> its pieces (piece_word)
  const int tpw = blockDim.x >> 7;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int slot = wave % tpw, member = wave / tpw;
  if (threadIdx.x < kScoreWaves / 2) claim[threadIdx.x] = 0;
  for (int i = threadIdx.x; i < 256; i += blockDim.x) lut[i] = piece_word(i);
  __syncthreads();
  const int t = blockIdx.y * tpw + slot;
  const int nkb = (p.S + 15) >> 4;
  const int b0 = blockIdx.x * p.blocks_per_wg;
  const int b1 = min(nkb, b0 + p.blocks_per_wg);
  if (t >= p.T || b0 >= b1) return;
  // the general paths split the range in halves
  const int mid = b0 + (b1 - b0 + 1) / 2;
  const int h0 = member == 0 ? b0 : mid, h1 = member == 0 ? mid : b1;
  const int qmax = q_magnitude_bound(p, t);
  if (qmax >= kTwoPieceLimit) {
    if (h0 < h1) score_range<NHB, 3, DIFF>(p, lut, t, h0, h1, qmax);
    return;
  }
  // the range's largest block bound decides whether every block takes the
  // three-product path
  if constexpr (NHB >= 2) {
    const int lane = threadIdx.x & 63;
    int rmax = 0;
    for (int b = b0 + lane; b < b1; b += 64) rmax = max(rmax, block_max_x(p.k_max[b]));
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) rmax = max(rmax, __shfl_xor(rmax, o));
    rmax = __builtin_amdgcn_readfirstlane(rmax);
    const bool descriptors_fit = (int64_t)nkb * kBlockBytes < (1LL << 31);
    if (rmax < kTwoPieceLimit && (int64_t)qmax * rmax * kIdxDim < (1LL << 31) && descriptors_fit) {
      score_range_fast<NHB, DIFF>(p, lut, t, b0, b1, &claim[slot], member == 0);
      return;
    }
  }
  if (h0 < h1) score_range<NHB, 2, DIFF>(p, lut, t, h0, h1, qmax);
}

// ---- quantise-on-append into the paged K cache ---------------------------

// e4m3fn code of x (finite, |x| <= 448), rounded to nearest, ties to even.
__device__ __forceinline__ uint32_t e4m3_encode(float x) {
  const uint32_t sign = (__float_as_uint(x) >> 24) & 0x80u;
  const float a = fabsf(x);
  uint32_t code;
  if (a < 0x1p-6f) {  // zero and the subnormals: multiples of 2^-9 (8 = the smallest normal)
    code = (uint32_t)__builtin_rintf(a * 512.0f);
  } else {            // 3 mantissa bits, ties to even; exponent rebiased 127 -> 7
    const uint32_t m = __float_as_uint(a);
    const uint32_t r = m + 0x7ffffu + ((m >> 20) & 1u);
    code = (((r >> 23) - 120u) << 3) | ((r >> 20) & 7u);
  }
  return sign | code;
}

// One wave per token: lane l quantises elements 2l, 2l+1.
__global__ __launch_bounds__(256) void dsa_k_append_kernel(KAppendParams p) {
  const int lane = threadIdx.x & 63;
  const int i = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (i >= p.n) return;
  const int slot = p.slots[i];
  if (slot < 0 || slot >= p.num_slots) return;
  const uint32_t pair = *(const uint32_t *)(p.k + (int64_t)i * p.k_stride + 2 * lane);
  const float x0 = __uint_as_float(pair << 16), x1 = __uint_as_float(pair & 0xffff0000u);
  float amax = fmaxf(fabsf(x0), fabsf(x1));
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) amax = fmaxf(amax, __shfl_xor(amax, o));
  const float scale = fmaxf(amax, 1e-4f) / 448.0f;
  const float y0 = fminf(fmaxf(x0 / scale, -448.0f), 448.0f);
  const float y1 = fminf(fmaxf(x1 / scale, -448.0f), 448.0f);
  const int pg = slot / p.page_size, off = slot - pg * p.page_size;
  uint8_t *page = p.cache + (int64_t)pg * p.page_size * kKTokenBytes;
  *(uint16_t *)(page + off * kIdxDim + 2 * lane) =
      (uint16_t)(e4m3_encode(y0) | (e4m3_encode(y1) << 8));
  if (lane == 0) *(float *)(page + p.page_size * kIdxDim + off * 4) = scale;
}

template <int NHB>
hipError_t launch_score(const IndexerParams &p, dim3 grid, dim3 block, hipStream_t stream) {
  if (p.k_blocks > 0) hipLaunchKernelGGL((dsa_idx_score_kernel<NHB, true>), grid, block, 0, stream, p);
  else hipLaunchKernelGGL((dsa_idx_score_kernel<NHB, false>), grid, block, 0, stream, p);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_k_append(const KAppendParams &p, hipStream_t stream) {
  if (p.n == 0) return hipSuccess;
  hipLaunchKernelGGL(dsa_k_append_kernel, dim3((p.n + 3) / 4), dim3(256), 0, stream, p);
  return hipGetLastError();
}

hipError_t launch_indexer_prepare_k(const IndexerParams &p, KPrep what, hipStream_t stream) {
  if (p.k_blocks <= 0) return hipSuccess;
  const int prep_blocks = (p.k_blocks + kPrepThreads / 64 - 1) / (kPrepThreads / 64);
  const dim3 grid(prep_blocks), block(kPrepThreads);
  if (what == kPrepCodes) hipLaunchKernelGGL(dsa_idx_prep_kernel<kPrepCodes>, grid, block, 0, stream, p);
  else if (what == kPrepPlanes) hipLaunchKernelGGL(dsa_idx_prep_kernel<kPrepPlanes>, grid, block, 0, stream, p);
  else hipLaunchKernelGGL(dsa_idx_prep_kernel<kPrepDiff>, grid, block, 0, stream, p);
  return hipGetLastError();
}

namespace {

// Exact scores of every position into p.scores, from the piece planes.
hipError_t launch_scores(const IndexerParams &pin, hipStream_t stream) {
  IndexerParams p = pin;
  const int nkb = (p.S + 15) / 16;
  // tokens per workgroup (two waves each) and 16-position blocks per
  // workgroup range, aiming at two waves per SIMD with at least 8 blocks
  // per wave
  const int tpw = std::min(p.T, kScoreWaves / 2);
  const int tgroups = (p.T + tpw - 1) / tpw;
  int bx = (kTargetScoreWaves + 2 * tpw * tgroups - 1) / (2 * tpw * tgroups);
  bx = std::min(bx, (nkb + 2 * kMinBlocksPerWave - 1) / (2 * kMinBlocksPerWave));
  bx = std::max(bx, 1);
  p.blocks_per_wg = (nkb + bx - 1) / bx;
  bx = (nkb + p.blocks_per_wg - 1) / p.blocks_per_wg;
  const dim3 grid(bx, tgroups), block(128 * tpw);
  switch (p.Hi / 16) {
    case 1: return launch_score<1>(p, grid, block, stream);
    case 2: return launch_score<2>(p, grid, block, stream);
    case 3: return launch_score<3>(p, grid, block, stream);
    default: return launch_score<4>(p, grid, block, stream);
  }
}

}  // namespace

hipError_t launch_indexer(const IndexerParams &pin, hipStream_t stream) {
  if (pin.T == 0) return hipSuccess;
  IndexerParams p = pin;
  if (!p.want_scores) {
    // only the selection is wanted: nothing to score where every row takes
    // all its candidates, else estimates and the exact scores of the few
    // positions they leave open
    if (p.topk == 0) return hipSuccess;
    if (p.topk >= p.S) return launch_topk(p, stream);
    if (estimates_apply(p)) {
      p.estimated = 1;
      hipError_t e = hipSuccess;
      if (p.k_blocks == 0) {  // prepared planes
        p.k_codes = (uint8_t *)p.k_pieces + kKPlaneCodeOffset;
        p.k_code_stride = kBlockBytes;
      } else {  // the call's own workspace: codes alone, packed (flat codes lie so already)
        p.k_codes = (uint8_t *)p.k_pieces;
        p.k_code_stride = kCodeBlockBytes;
        p.est_fused = estimates_prepare_k(p);
        if (!p.est_fused) e = launch_indexer_prepare_k(p, kPrepCodes, stream);
        else if (!p.k_cache) p.k_codes = const_cast<uint8_t *>(p.k);
      }
      if (e == hipSuccess) e = launch_estimates(p, stream);
      return e == hipSuccess ? launch_topk(p, stream) : e;
    }
  }
  // piece blocks: planes p0 and p1, then the codes (prepared) or the third plane
  p.k_codes = (uint8_t *)p.k_pieces + kKPlaneCodeOffset;
  p.k_code_stride = kBlockBytes;
  hipError_t e = launch_indexer_prepare_k(p, kPrepDiff, stream);
  if (e == hipSuccess && p.S > 0) e = launch_scores(p, stream);
  if (e == hipSuccess && p.topk > 0) e = launch_topk(p, stream);
  return e;
}

}  // namespace dsa
